// grns_scale.hip -- launches of the scaling of long arrays (grns_scale.hpp).
#include <hip/hip_runtime.h>

#include "grns_internal.hpp"
#include "grns_scale.hpp"

using namespace grns;

grns_status matrix_scale(grns_ctx *c, const int *x, long long smod, long long snum, const unsigned *D, size_t count,
                         int *y, hipStream_t s) {
    long long blocks = (long long)((count + BLOCK / 2 - 1) / (BLOCK / 2));
    if (blocks >= 8) blocks = (blocks + 7) / 8 * 8;  // a multiple of the XCD count (see xcd_block)
    const dim3 grid((unsigned)blocks), blk(BLOCK);
    const long long cnt = (long long)count;
    if (c->n <= 8) hipLaunchKernelGGL((k_scale_mat<8>), grid, blk, 0, s, c->d, c->mat, x, smod, snum, D, cnt, y);
    else if (c->n <= 16) hipLaunchKernelGGL((k_scale_mat<16>), grid, blk, 0, s, c->d, c->mat, x, smod, snum, D, cnt, y);
    else if (c->n <= 32) hipLaunchKernelGGL((k_scale_mat<32>), grid, blk, 0, s, c->d, c->mat, x, smod, snum, D, cnt, y);
    else hipLaunchKernelGGL((k_scale_mat<64>), grid, blk, 0, s, c->d, c->mat, x, smod, snum, D, cnt, y);
    return hipGetLastError() == hipSuccess ? GRNS_OK : GRNS_ERR_HIP;
}
