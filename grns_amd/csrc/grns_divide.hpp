// grns_divide.hpp -- rns_div / rns_div_fast (src/rnsdiv.cuh:19-114) of 64 pairs per wave.
//
// Quotient and remainder of two integers are unique, so the pairs are divided on positional digits:
// x and d become 28-bit digits on the matrix cores, one lane divides one pair, and the quotient's and
// remainder's digits become residues on the matrix cores again.  The reference's one non-canonical
// output (a nonzero quotient divisible by an m_i keeps m_i where its reciprocal addition does, see
// group_div_words) is put back at the end.
//
// Long division with signed quotient digits in base 2^28.  The dividend's digits stay 64-bit sums
// without carries between them: a step subtracts q D, one v_mad_i64_i32 per digit of D, and adds
// less than 2^55.1 to a digit; 71 steps keep them below 2^62.  q is the nearest integer to (the
// window's top digits) / (the divisor's top three), in FP64 to 2^-15, so the new remainder is within
// (1/2 + 2^-15) of the divisor, |q| stays below 2^27 (1 + 2^-14), and no step needs a correction:
// one at the end makes the remainder nonnegative.  The wave-per-pair form pays a scalar quotient
// estimate and a carry resolution per word of one pair; here 64 pairs share a step.  2^20 pairs with
// divisors of uniform length: 4.42 -> 0.85 ms with 64 moduli, 2.19 -> 0.29 ms with 32, 0.54 -> 0.087
// ms with 8.  With 64 moduli two waves per SIMD fit (registers and LDS), and of a wave's 209
// thousand cycles 30% are in the division steps (at the multiply-adds' rate), 44% in the conversion
// of x and d (half of it matrix instructions) and 20% in the residues.
//
// Registers need constant indices while the lanes' divisors differ in length.  The dividend's digits
// W[t] (digit ND - 1 - t) stay in place; the divisor's are in LDS from the top down, D[i] = digit
// nd - 1 - i, and step t subtracts q D from W[t], W[t + 1], ... in every lane at once: it gives the
// lane's quotient digit of weight ND - nd - t, and a lane with no such weight is done and subtracts 0.
// Four steps make a block.  The block's head, the eight entries from W[4 b] on, is copied out (a
// branch per block picks the registers), gives the four quotient digits, and goes back; then the
// four are applied to the entries below, chunk by chunk, by divisor rows 4 b lower (zero rows on
// either side make every product right or 0).  Chunks above the head or past the longest divisor at
// work are skipped.  The loop over blocks is rolled: unrolled over all steps, the code was 90 KB and
// every wave waited for its instructions; moving the digits up by four places per block instead
// cost two register copies of the window.
#pragma once

#include "grns_matrix.hpp"

namespace grns {

// Four 7-bit pieces of a digit in (-2^28, 2^28): three in [0, 127] and a signed top one.
GRNS_D int digit_pieces(int d) {
    unsigned v = (unsigned)d;  // everything above a piece moves up by one bit, three times
    v += v & ~0x7fu;
    v += v & ~0x7fffu;
    v += v & ~0x7fffffu;
    return (int)v;
}

template <int NP>
struct DivShape {
    static constexpr int ND = Mat<NP>::ND, HEAD = 8, CHUNK = 8, BLOCKS = (ND + 3) / 4;
    static constexpr int PAD = 2;  // zero rows above D[0]: a chunk at work reads from row 4 b + 1 - 4 b - 3 on
    static constexpr int ROWS = 8 * Mat<NP>::DT > ND + PAD ? 8 * Mat<NP>::DT : ND + PAD;
};

// A move the compiler keeps as one (and behind its branch).
GRNS_D long long move_entry(long long v) {
    long long r;
    asm volatile("v_mov_b64_e32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
// The head of block b out of the window, and back.
template <int NP, int... B>
GRNS_D void head_out(int b, long long (&H)[DivShape<NP>::HEAD], const long long (&W)[Mat<NP>::ND],
                     std::integer_sequence<int, B...>) {
    auto copy = [&](auto blk) {
        constexpr int B0 = 4 * decltype(blk)::value;
#pragma unroll
        for (int i = 0; i < DivShape<NP>::HEAD; i++) H[i] = B0 + i < Mat<NP>::ND ? move_entry(W[B0 + i < Mat<NP>::ND ? B0 + i : 0]) : 0;
    };
    ((b == B ? copy(std::integral_constant<int, B>{}) : (void)0), ...);
}
template <int NP, int... B>
GRNS_D void head_in(int b, const long long (&H)[DivShape<NP>::HEAD], long long (&W)[Mat<NP>::ND],
                    std::integer_sequence<int, B...>) {
    auto copy = [&](auto blk) {
        constexpr int B0 = 4 * decltype(blk)::value;
#pragma unroll
        for (int i = 0; i < DivShape<NP>::HEAD; i++)
            if (B0 + i < Mat<NP>::ND) W[B0 + i < Mat<NP>::ND ? B0 + i : 0] = move_entry(H[i]);
    };
    ((b == B ? copy(std::integral_constant<int, B>{}) : (void)0), ...);
}

// What a lane keeps of its last step: the quotient's lowest digit, and v / D - 1/2 of that step.
struct DivLast {
    int q;
    double u;
};

// Step S of a block on its head: the quotient digit (negated) of weight `left` (the lane is done when
// it is negative) applied to the head.  The digit is the integer nearest to window / divisor, the
// last one that below it, ties aside.  The rounding is an addition of 1.5 2^52, whose low word is
// the integer: the chain from one digit to the next is what a step waits for.  Entry S then holds
// the quotient digit, or still the remainder's top digit in a lane that is done.
template <int NP, int S>
GRNS_D int div_digit(long long (&H)[DivShape<NP>::HEAD], const int (&D)[DivShape<NP>::HEAD], double ninv, int left,
                     DivLast &end) {
    constexpr double SHIFTER = 0x1.8p52;
    const double low = fma((double)(int)(H[S + 2] >> 32), 0x1p-24,
                           fma((double)(int)(H[S + 1] >> 32), 16.0, (double)(unsigned)H[S + 1] * 0x1p-28));
    const double v = fma((double)(int)(H[S] >> 32), 4294967296.0, (double)(unsigned)H[S] + low);
    const double u = fma(v, ninv, left == 0 ? 0.5 : 0.0), t = u + SHIFTER;
    const int n0 = (int)(unsigned)(unsigned long long)__double_as_longlong(t);
    const int nq = (int)lane_offset((unsigned)(left >= 0 ? n0 : 0));
    end.q = left == 0 ? -nq : end.q;
    end.u = left == 0 ? u : end.u;
#pragma unroll
    for (int i = 0; i < DivShape<NP>::HEAD - S; i++) H[S + i] += (long long)nq * D[i];
    H[S + 1] += left > 0 ? H[S] << 28 : 0;
    H[S] = left > 0 ? -(long long)nq : H[S];
    return nq;
}

// One block.  ninv: -1 / divisor; nda: the longest divisor still at work; left: ND - nd - 4 b.
template <int NP>
GRNS_D void div_block(long long (&W)[Mat<NP>::ND], const int *own, double ninv, int b, int nda, int left, DivLast &end) {
    using Sh = DivShape<NP>;
    constexpr auto cases = std::make_integer_sequence<int, Sh::BLOCKS>{};
    long long H[Sh::HEAD];
    head_out<NP>(b, H, W, cases);
    int top[Sh::HEAD];
#pragma unroll
    for (int i = 0; i < Sh::HEAD; i++) top[i] = own[(Sh::PAD + i) * 64];
    int nq[4];
    nq[0] = div_digit<NP, 0>(H, top, ninv, left, end);
    nq[1] = div_digit<NP, 1>(H, top, ninv, left - 1, end);
    nq[2] = div_digit<NP, 2>(H, top, ninv, left - 2, end);
    nq[3] = div_digit<NP, 3>(H, top, ninv, left - 3, end);
    // entries from 4 b + 8 on (those of the head are overwritten below)
#pragma unroll
    for (int j0 = 0; j0 < Sh::ND; j0 += Sh::CHUNK) {
        if (j0 + Sh::CHUNK > 4 * b + Sh::HEAD && j0 < 4 * b + 3 + nda) {
            const int *row = own + (Sh::PAD + j0 - 3 - 4 * b) * 64;
            int d[Sh::CHUNK + 3];  // D[j0 - 3 - 4 b] on
#pragma unroll
            for (int i = 0; i < Sh::CHUNK + 3; i++) d[i] = j0 + i - 3 < Sh::ND ? row[i * 64] : 0;
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int j = j0; j < j0 + Sh::CHUNK; j++)
                    if (j < Sh::ND)
                        W[j] = (long long)lane_pair((unsigned long long)(W[j] + (long long)nq[s] * d[j + 3 - s - j0]));
        }
    }
    head_in<NP>(b, H, W, cases);
}

GRNS_D int wave_max(int v) {
    for (int s = 1; s < 64; s <<= 1) {
        const int o = __shfl_xor(v, s, 64);
        v = o > v ? o : v;
    }
    return __builtin_amdgcn_readfirstlane(v);
}

// How a wave's residues are stored: STORE_ROWS all of them, one per modulus row; STORE_QUADS all of them,
// 16 bytes per four moduli; STORE_ANY with the checks of a partial wave and a partial set.
enum { STORE_ROWS, STORE_QUADS, STORE_ANY };

// Residues of the integers whose digits are in the B operands, row tile by row tile, to dst[t] (residue
// 4 h of tile t's number).  any[t]: the integer is not 0 and keeps m_i where a reciprocal addition
// would (quotients).  on[t]: the number is stored (STORE_ANY).
template <int NP, int STORE>
GRNS_D void residue_rows(const MatTab &tab, const ModRec *rec, int lane, int n, const v4i (&B)[2][Mat<NP>::KD],
                         const bool (&any)[2], const bool (&on)[2], int *const (&dst)[2], long long smod) {
    constexpr int KD = Mat<NP>::KD, RT = Mat<NP>::RT;
    const int h = lane >> 5;
    v4i a[KD];
    auto load_rows = [&](int mt) {
#pragma unroll
        for (int ks = 0; ks < KD; ks++) a[ks] = tab.res7[(mt * KD + ks) * 64 + lane];
    };
    load_rows(0);
    int *w[2] = {dst[0], dst[1]};
#pragma unroll 1
    for (int mt = 0; mt < RT; mt++) {
        v16i acc[2] = {};
#pragma unroll
        for (int ks = 0; ks < KD; ks++)
#pragma unroll
            for (int t = 0; t < 2; t++) acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[ks], B[t][ks], acc[t], 0, 0, 0);
        // The next rows are requested before this tile's stores, and the stores are not behind
        // conditions: memory operations are counted in order, so rows requested after them (or
        // after an unknown number of them) would wait until the stores are done.
        sched_stop();
        load_rows(mt + 1 < RT ? mt + 1 : 0);
        sched_stop();
        const int i0 = 8 * mt + 4 * h;
        v4i o[2];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const ModRec mr = rec[i0 + b];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const unsigned v = bytes_residue(acc[t][4 * b], acc[t][4 * b + 1], acc[t][4 * b + 2], acc[t][4 * b + 3], mr);
                o[t][b] = (int)(any[t] && v == 0 && mr.keeps_m ? mr.m : v);
            }
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if constexpr (STORE == STORE_QUADS) {
                *reinterpret_cast<v4i *>(w[t]) = o[t];
            } else {
#pragma unroll
                for (int b = 0; b < 4; b++)
                    if (STORE == STORE_ROWS || (on[t] && i0 + b < n)) w[t][(long long)b * smod] = o[t][b];
            }
            w[t] += 8 * smod;
        }
    }
}

constexpr int div_waves(int NP) { return NP == 64 ? 2 : NP == 8 ? 4 : 3; }  // per SIMD: registers and LDS allow these

// A block's LDS: digits of each wave's pairs, and the small tables.
template <int NP>
struct DivShared {
    int digits[BLOCK / 64][DivShape<NP>::ROWS * 64];
    __align__(16) int init[Mat<NP>::DT * 32];
    __align__(16) int mdig[8 * Mat<NP>::DT];
    ModRec rec[NP];
};

// The wave's pairs j0 .. j0 + 63 (those below count; all waves of a block call it).  rest(left, j): the
// lane's pair j if it is left to the reference loop (a residue outside [0, m), or a zero divisor).
template <int NP, class Rest>
GRNS_D void div_wave(const DevCtx *__restrict__ c, const MatTab &tab, DivShared<NP> &sh, const int *x, const int *d,
                     long long smod, long long snum, long long count, long long j0, int *q, int *r, Rest rest) {
    constexpr int KR = Mat<NP>::KR, ND = Mat<NP>::ND, DT = Mat<NP>::DT;
    int *init = sh.init, *mdig = sh.mdig;
    ModRec *rec = sh.rec;
    for (int i = threadIdx.x; i < DT * 32; i += BLOCK) init[i] = tab.crt7_init[i];
    for (int i = threadIdx.x; i < 8 * DT; i += BLOCK) mdig[i] = tab.m28[i];
    for (int i = threadIdx.x; i < NP; i += BLOCK) rec[i] = tab.rec[i];
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int n = c->n;
    int *lds = sh.digits[threadIdx.x >> 6], *own = lds + lane;
    const bool quad = quads(x, smod, snum) && quads(d, smod, snum);
    DigitColumn col[2];
    const int *p[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        unsigned *cp = reinterpret_cast<unsigned *>(lds) + 32 * t + (lane & 31);
        col[t] = {cp, cp, 64, 8 * DT};
    }
    auto number = [&](int t) {
        const long long j = j0 + 32 * t + (lane & 31);
        return (j < count ? j : count - 1) * snum;
    };
    unsigned long long bad = 0;  // bit l: pair j0 + l has a residue outside [0, m)
    auto convert = [&](const int *src, bool first) {
        v4i B[2][KR];
        int k[2];
        LaneAny nc[2];
#pragma unroll
        for (int t = 0; t < 2; t++) p[t] = src + number(t);
        load_residues<NP, 2>(p, smod, quad, n, h, B);
        if (first) __syncthreads();  // the tables; the first residues are on their way
        crt_operand<NP, 2>(rec, h, B, k, nc);
        bad |= ((nc[0].m | nc[0].m >> 32) & 0xffffffffull) | (nc[1].m | nc[1].m >> 32) << 32;
        crt_digits<NP, 7, DT, 1, 2>(tab.crt7, init, mdig, reinterpret_cast<const unsigned *>(mdig), B, k, lane, col);
        wave_lds_fence();
    };
    int nd = 0, D[ND] = {};
    bool zero = false;
    // pass 0: the divisor, its length and its digits from the top down; pass 1: the dividend
#pragma unroll 1
    for (int pass = 0; pass < 2; pass++) {
        convert(pass ? x : d, pass == 0);
        if (pass) break;
#pragma unroll
        for (int k = 0; k < ND; k++) nd = own[k * 64] != 0 ? k + 1 : nd;
        zero = nd == 0;
        if (zero) {  // left to the reference loop; any divisor will do here
            own[0] = 1;
            nd = 1;
        }
#pragma unroll
        for (int i = 0; i < ND; i++) {
            const int k = nd - 1 - i, v = own[(k > 0 ? k : 0) * 64];
            D[i] = k >= 0 ? v : 0;
        }
        wave_lds_fence();
    }
    const double ninv = -1.0 / ((double)D[0] + (double)D[1] * 0x1p-28 + (double)D[2] * 0x1p-56);
    const int ndmax = wave_max(nd), ndmin = -wave_max(-nd);
    long long W[ND];
#pragma unroll
    for (int t = 0; t < ND; t++) W[t] = own[(ND - 1 - t) * 64];
    wave_lds_fence();
    constexpr int PAD = DivShape<NP>::PAD;
#pragma unroll
    for (int i = 0; i < PAD; i++) own[i * 64] = 0;
#pragma unroll
    for (int i = 0; i < ND; i++) own[(PAD + i) * 64] = D[i];
    DivLast end = {0, 0.0};
    const int blocks = (ND - ndmin + 4) / 4;
#pragma unroll 1
    for (int b = 0; b < blocks; b++)
        div_block<NP>(W, own, ninv, b, ndmax < ND - 4 * b ? ndmax : ND - 4 * b, ND - nd - 4 * b, end);
    // the remainder's carries: its digit k is entry ND - 1 - k, k < nd; the other entries are quotient digits
    int R[ND];
    long long cy = 0;
    const int split = (int)lane_offset((unsigned)(ND - nd));  // compared afresh in each pass: ND lane masks are not kept
#pragma unroll
    for (int t = ND - 1; t >= 0; t--) {
        const bool rem = t >= split;
        const long long v = (rem ? W[t] : 0) + cy;
        R[t] = rem ? (int)v & 0xfffffff : (int)W[t];
        cy = rem ? v >> 28 : cy;
    }
    // 0 <= remainder < divisor but for about one lane in 2^13: those add or subtract the divisor
    const bool neg = cy < 0;
    const bool high = end.u + 0.5 - rint(end.u + 0.5) < 0x1p-14 && end.u + 0.5 - rint(end.u + 0.5) > -0x1p-14;
    if (__any(neg || high)) {
        const int *dig = own + (PAD + nd - ND) * 64;  // D[t - (ND - nd)] of entry t
        int c0 = 0;
#pragma unroll 1
        for (int pass = 0; pass < 2; pass++) {
            const int f = neg ? 1 : pass == 0 || c0 + (int)cy >= 0 ? -1 : 0;  // -1 only if that leaves no borrow (cy: at most 1)
            const bool apply = pass == 1 && (neg || (high && f != 0));
            c0 = 0;
            const int split1 = (int)lane_offset((unsigned)(ND - nd));
#pragma unroll
            for (int t = ND - 1; t >= 0; t--) {
                if (t >= split1) {
                    const int v = R[t] + f * dig[t * 64] + c0;
                    R[t] = apply ? v & 0xfffffff : R[t];
                    c0 = v >> 28;
                }
            }
            if (apply) end.q -= f;
        }
    }
    wave_lds_fence();
    // rows QTOP - e: the pieces of digit e of the quotient (e <= ND - nd); rows k < nd: of digit k of the
    // remainder
    constexpr int QTOP = 8 * DT - 1;
    static_assert(QTOP >= ND, "ND + 1 digits in all");
    own[QTOP * 64] = digit_pieces(end.q);
    const int split2 = (int)lane_offset((unsigned)(ND - nd));
#pragma unroll
    for (int t = 0; t < ND; t++) own[(t < split2 ? QTOP - ND + nd + t : ND - 1 - t) * 64] = digit_pieces(R[t]);
    wave_lds_fence();
    // residues of the quotient, then of the remainder
    const long long jl = j0 + lane;
    const bool ok = jl < count && !zero && !(bad >> lane & 1);
    const unsigned long long okm = __ballot(ok);
    int ndt[2];  // lengths of the tiles' divisors
#pragma unroll
    for (int t = 0; t < 2; t++) ndt[t] = __shfl(nd, 32 * t + (lane & 31), 64);
    const bool full = okm == ~0ull && (n & 7) == 0 && n == NP;
#pragma unroll 1
    for (int rem = 0; rem < 2; rem++) {
        int *out = rem ? r : q, *dst[2];
        v4i B[2][Mat<NP>::KD];
        bool any[2], on[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            // digit e is in row e or QTOP - e, for e below end
            const int len = (int)lane_offset((unsigned)ndt[t]), end = (rem ? len : ND + 1 - len) - 4 * h;
            const int step = rem ? 64 : -64;
            const int *row = lds + lane_offset(32 * t + (lane & 31)) + (rem ? 4 * h : QTOP - 4 * h) * 64;
            int nz = 0;
#pragma unroll
            for (int ks = 0; ks < Mat<NP>::KD; ks++) {
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const int v = row[b * step];
                    B[t][ks][b] = 8 * ks + b < end ? v : 0;
                    nz |= B[t][ks][b];
                }
                row += 8 * step;
                sched_stop();
            }
            any[t] = !rem && (nz | other_half(nz)) != 0;
            on[t] = okm >> (32 * t + (lane & 31)) & 1;
            dst[t] = out + number(t) + 4 * h * smod;
        }
        sched_stop();
        if (full && !quads(out, smod, snum)) residue_rows<NP, STORE_ROWS>(tab, rec, lane, n, B, any, on, dst, smod);
        else if (full) residue_rows<NP, STORE_QUADS>(tab, rec, lane, n, B, any, on, dst, smod);
        else residue_rows<NP, STORE_ANY>(tab, rec, lane, n, B, any, on, dst, smod);
    }
    rest(jl < count && !ok, jl);
}

template <int NP>
__global__ __launch_bounds__(BLOCK, div_waves(NP)) void k_div_mat(const DevCtx *__restrict__ c, MatTab tab,
                                                                  const int *x, const int *d, long long smod,
                                                                  long long snum, long long count, int *q, int *r,
                                                                  RareQ rq) {
    __shared__ DivShared<NP> sh;
    const long long j0 = ((long long)xcd_block() * (BLOCK / 64) + (threadIdx.x >> 6)) * 64;
    div_wave<NP>(c, tab, sh, x, d, smod, snum, count, j0, q, r, [&](bool left, long long j) {
        if (!rare_push(rq, left, j)) q[j * snum] = DIV_MARK;
    });
}

}  // namespace grns
