"""The shares of a tile's points that the workgroups of the box pass take
(csrc/owm_kernels.h): together the whole tile, up to the most points a call may have."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))

SOURCE = """
#include "%s/owm_kernels.h"
int main()
{
    const uint32_t ns[] = {0, 1, 2047, 2048, 2049, 4096, 70001, 4292870143u, 4292870144u, 4292870145u,
                           4294966272u, 4294966273u, 4294967293u, 4294967294u};
    for (uint32_t n : ns)
        for (uint32_t nb : {1u, 2u, 3u, 1000u, 1023u, 1024u, 4096u}) {
            uint32_t at = 0;
            for (uint32_t k = 0; k < nb; ++k) {
                uint32_t c0, c1;
                owm::box_share(n, nb, k, c0, c1);
                if (c0 != at || c1 < c0 || c1 > n)
                    return 1;
                // a round's indices stay below 2^32 (one workgroup: launches that large have more)
                if (nb > 1 && (uint64_t)(c1 - c0) + 2048 > 0xFFFFFFFFull)
                    return 2;
                at = c1;
            }
            if (at != n)
                return 3;
        }
    return 0;
}
"""


def test_shares_hold_every_point(tmp_path):
    src, exe = str(tmp_path / "shares.cpp"), str(tmp_path / "shares")
    with open(src, "w") as f:
        f.write(SOURCE % os.path.join(os.path.dirname(HERE), "fastowm_amd", "csrc"))
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIPCC__", "-I", os.path.join(HERE, "hipcpu"), "-o", exe, src],
                   check=True)
    assert subprocess.run([exe]).returncode == 0
