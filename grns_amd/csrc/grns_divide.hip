// grns_divide.hip -- launches of the lane-per-pair division (grns_divide.hpp).
#include <hip/hip_runtime.h>

#include "grns_divide.hpp"
#include "grns_internal.hpp"

using namespace grns;

grns_status matrix_div(grns_ctx *c, const int *x, const int *d, long long smod, long long snum, size_t count, int *q,
                       int *r, const RareQ &rq, hipStream_t s) {
    long long blocks = (long long)((count + BLOCK - 1) / BLOCK);
    if (blocks >= 8) blocks = (blocks + 7) / 8 * 8;  // a multiple of the XCD count (see xcd_block)
    const dim3 grid((unsigned)blocks), blk(BLOCK);
    const long long cnt = (long long)count;
    if (c->n <= 8) hipLaunchKernelGGL((k_div_mat<8>), grid, blk, 0, s, c->d, c->mat, x, d, smod, snum, cnt, q, r, rq);
    else if (c->n <= 16) hipLaunchKernelGGL((k_div_mat<16>), grid, blk, 0, s, c->d, c->mat, x, d, smod, snum, cnt, q, r, rq);
    else if (c->n <= 32) hipLaunchKernelGGL((k_div_mat<32>), grid, blk, 0, s, c->d, c->mat, x, d, smod, snum, cnt, q, r, rq);
    else hipLaunchKernelGGL((k_div_mat<64>), grid, blk, 0, s, c->d, c->mat, x, d, smod, snum, cnt, q, r, rq);
    return hipGetLastError() == hipSuccess ? GRNS_OK : GRNS_ERR_HIP;
}
