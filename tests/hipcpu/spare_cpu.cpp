// The memory a context keeps of the last freed tree (csrc/owm_host.cpp on the HIP of
// hip/hip_runtime.h): given back to whatever buffer of the context, or of its serving
// slots, the device has no room for.  Exits with the number of the first failing step.
#include "../../fastowm_amd/csrc/owm_host.h"

owm_ctx::~owm_ctx() {}

static void keep(owm_ctx &c, uint64_t bytes)
{
    owm::DevBuf tree;
    if (c.grow(tree, bytes, bytes) != hipSuccess)
        exit(99);
    c.spare.swap(tree);
}

int main()
{
    constexpr uint64_t KB = 1024;
    hipcpu::memory_left = 1000 * KB;
    owm_ctx ctx, slot;
    slot.owner = &ctx;
    keep(ctx, 600 * KB);
    if (ctx.held_bytes() != 600 * KB || ctx.grow(ctx.upload, 500 * KB, 500 * KB) != hipSuccess || ctx.spare.ptr)
        return 1;
    if (ctx.grow(ctx.qs_work, 600 * KB, 600 * KB) != hipErrorOutOfMemory || ctx.qs_work.ptr)
        return 2;
    ctx.upload.release();
    keep(ctx, 600 * KB);
    if (owm::ensure_s1_list(&ctx, 150 * KB) != OWM_OK || ctx.spare.ptr)
        return 3;
    ctx.s1_list.release();
    keep(ctx, 600 * KB);
    if (ctx.arena.ensure(&ctx, 700 * KB) != OWM_OK || ctx.spare.ptr)
        return 4;
    ctx.arena.buf.release();
    keep(ctx, 600 * KB);
    if (slot.grow(slot.upload, 500 * KB, 500 * KB) != hipSuccess || ctx.spare.ptr)
        return 5;
    slot.upload.release();
    keep(ctx, 600 * KB);
    owm::DevBuf small;
    if (ctx.grow(small, 300 * KB, 300 * KB) != hipSuccess || !ctx.spare.ptr)
        return 6;  // room for both: kept
    ctx.budget = 1000 * KB;
    if (ctx.exceeds(300 * KB) || !ctx.spare.ptr || ctx.exceeds(500 * KB) || ctx.spare.ptr)
        return 7;
    // a borrowed region never grows, whatever could be given back
    keep(ctx, 600 * KB);
    owm::DevBuf lent;
    lent.borrowed = true;
    if (ctx.grow(lent, 100 * KB) != hipErrorOutOfMemory || !ctx.spare.ptr)
        return 8;
    return 0;
}
