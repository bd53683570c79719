"""Device memory a context keeps for later, on the CPU (tests/hipcpu)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "fastowm_amd", "csrc")


def test_kept_tree_memory_is_given_back(tmp_path):
    """Every buffer grows through owm_ctx::grow (DevBuf's own is private to it)."""
    exe = str(tmp_path / "spare_cpu")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIPCC__", "-I", os.path.join(HERE, "hipcpu"),
                    "-Wl,--unresolved-symbols=ignore-all", "-o", exe, os.path.join(HERE, "hipcpu", "spare_cpu.cpp"),
                    os.path.join(CSRC, "owm_host.cpp")], check=True)
    assert subprocess.run([exe]).returncode == 0
