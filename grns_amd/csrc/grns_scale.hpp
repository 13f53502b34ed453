// grns_scale.hpp -- rns_scale2pow (src/rnsscal.cuh:93-119) of long arrays: 32 numbers per wave.
//
// The steps are those of group_scale_digits, a wave group per number with a lane per modulus; what they
// need first, the number's bits, comes from the matrix cores for 32 numbers at a time, where group_words
// sums them number by number.  The words go to LDS, a group turns its number's into 30-bit digits,
// and the steps read these four at a time, the same address in every lane.  The residues are loaded a
// second time, now with the modulus as the lane, a register per number (16 bytes for four numbers
// where the array allows); the results take the place of the words in LDS and leave together, a row of
// numbers per modulus.  2^20 numbers of 64 moduli, exponents to 1900: 2.31 -> 0.94 ms, of which 0.31 ms
// are left at exponent 0; a step of 2^-30 of all of them takes 17 us, the rate at which its 47 vector
// instructions per four steps (16 of them 32-bit multiplications) issue.  Numbers of 32, 16, 8
// moduli: 0.93, 0.61, 0.26 -> 0.42, 0.17, 0.077 ms.
#pragma once

#include "grns_matrix.hpp"

namespace grns {

// A block's LDS.
template <int NP>
struct ScaleShared {
    __align__(16) int init[Mat<NP>::WT * 32];
    __align__(16) int mdig[8 * Mat<NP>::WT];
    ModRec rec[NP];
    unsigned words[BLOCK / 64][32 * (NP + 1)];
    __align__(16) unsigned digits[BLOCK / 64][(64 / NP) * (2 * NP + 4)];  // four are read past the last
};

// The wave's numbers j0 .. j0 + 31 (those below count; all waves of a block call it).
template <int NP>
GRNS_D void scale_wave(const DevCtx *__restrict__ c, const MatTab &tab, ScaleShared<NP> &sh, const int *x, long long smod,
                       long long snum, const unsigned *__restrict__ D, long long count, long long j0, int *y) {
    constexpr int WT = Mat<NP>::WT, KR = Mat<NP>::KR, S = NP + 1, GD = NP, K = NP / 2;  // K numbers per group
    int *init = sh.init, *mdig = sh.mdig;
    ModRec *rec = sh.rec;
    for (int i = threadIdx.x; i < WT * 32; i += BLOCK) init[i] = tab.crt8_init[i];
    for (int i = threadIdx.x; i < 8 * WT; i += BLOCK) mdig[i] = tab.m8[i];
    for (int i = threadIdx.x; i < NP; i += BLOCK) rec[i] = tab.rec[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int n = c->n;
    const Group g = make_group(GD, n);
    const bool quad = quads(x, smod, snum);
    const bool rows = snum == 1 && (smod & 3) == 0 && ((uintptr_t)x & 15) == 0;
    unsigned *st = sh.words[threadIdx.x >> 6], *dp = sh.digits[threadIdx.x >> 6] + (g.base / NP) * (2 * NP + 4);
    if (j0 >= count) return;
    const long long jl = j0 + (lane & 31), jc = jl < count ? jl : count - 1;
    const int Dl = (int)D[jc];
    unsigned bad;  // bit k: number j0 + k has a residue outside [0, m)
    {
        const int *p[1] = {x + jc * snum};
        unsigned *own = st + (lane & 31) * S;
        const DigitColumn col[1] = {{own, own, 1, NP}};
        v4i B[1][KR];
        int k[1];
        LaneAny nc[1];
        load_residues<NP, 1>(p, smod, quad, n, h, B);
        crt_operand<NP, 1>(rec, h, B, k, nc);
        crt_digits<NP, 8, WT, 1, 1>(tab.crt8, init, mdig, tab.m32, B, k, lane, col);
        bad = (unsigned)nc[0].m | (unsigned)(nc[0].m >> 32);
    }
    wave_lds_fence();
    const int first = GD == 64 ? 0 : (g.base / GD) * K;  // the group's numbers are j0 + first .. + K - 1
    const int *xg = x + (j0 + first) * snum + (long long)(g.gl < n ? g.gl : 0) * smod;
    const long long left = count - j0 - first;
    // the group's residues, one register per number
    typedef int Res __attribute__((ext_vector_type(K)));
    Res res;
    if (rows && left >= K) {
#pragma unroll
        for (int k = 0; k < K; k += 4) {
            const v4i v = *reinterpret_cast<const v4i *>(xg + k);
#pragma unroll
            for (int b = 0; b < 4; b++) res[k + b] = v[b];
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; k++) res[k] = left > k ? xg[k * snum] : 0;
    }
    const ScaleLane lc = scale_lane(c, g);
#pragma unroll 1
    for (int k = 0; k < K; k++) {
        const int num = first + k, xi = res[k];
        unsigned *row = st + num * S;
        unsigned dig2[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int b = 30 * (g.gl + i * GD), w0 = b >> 5;
            const unsigned lo = w0 < NP ? row[w0 < NP ? w0 : 0] : 0u, hi = w0 + 1 < NP ? row[w0 + 1 < NP ? w0 + 1 : 0] : 0u;
            dig2[i] = (unsigned)((((unsigned long long)hi << 32) | lo) >> (b & 31)) & 0x3fffffffu;
            dp[g.gl + i * GD] = dig2[i];
        }
        wave_lds_fence();
        const unsigned long long t0 = gballot<GD>(g, dig2[0] != 0), t1 = gballot<GD>(g, dig2[1] != 0);
        const int xbits = t1 ? 30 * (GD + 64 - __clzll((long long)t1)) : t0 ? 30 * (64 - __clzll((long long)t0)) : 0;
        unsigned Dn;
        if constexpr (GD == 64) Dn = (unsigned)__builtin_amdgcn_readlane(Dl, num);
        else Dn = (unsigned)__shfl(Dl, num, 64);
        if (left > k) {
            const int v = group_scale_digits<GD>(c, g, lc, xi, Dn, xbits, group_uniform<GD>(!(bad >> num & 1)),
                                                 [&](int s) { return s < 2 * GD ? dp[s] : 0u; },
                                                 [&](int s, unsigned(&r)[4]) {
                                                     const uint4 q = *reinterpret_cast<const uint4 *>(dp + s);
                                                     r[0] = q.x, r[1] = q.y, r[2] = q.z, r[3] = q.w;
                                                 });
            row[g.gl] = (unsigned)v;
        }
        wave_lds_fence();
    }
    if (smod == 1) {
#pragma unroll 1
        for (int k = 0; k < K; k++)
            if (left > k && g.gl < n) y[(j0 + first + k) * snum + g.gl] = (int)st[(first + k) * S + g.gl];
    } else if (jl < count) {
        for (int i = h; i < n; i += 2) y[jl * snum + (long long)i * smod] = (int)st[(lane & 31) * S + i];
    }
}

template <int NP>
__global__ __launch_bounds__(BLOCK, 4) void k_scale_mat(const DevCtx *__restrict__ c, MatTab tab, const int *x,
                                                        long long smod, long long snum,
                                                        const unsigned *__restrict__ D, long long count, int *y) {
    __shared__ ScaleShared<NP> sh;
    const long long j0 = ((long long)xcd_block() * (BLOCK / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * 32;
    scale_wave<NP>(c, tab, sh, x, smod, snum, D, count, j0, y);
}

}  // namespace grns
