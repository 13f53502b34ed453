// grns_matrix.hpp -- conversions between residues and positional digits on the matrix cores.
//
// Both directions are products with constant tables.  The CRT value sum_i s_i (M / m_i) of a number
// (s_i = x_i w_i mod m_i) has as its column sums (bytes of the s_i) x (digits of 2^(8 a) M / m_i); the
// residues of an integer have as theirs (small digits of the integer) x (2^k mod m_i).  A wave takes
// 32 numbers per tile as the columns of v_mfma_i32_32x32x32_i8, whose operands are 8-bit and whose sums are
// exact in 32 bits; the tables are the rows.  Row order is chosen so that the four accumulator
// registers a lane holds side by side are the four 8-bit (or 7-bit) columns of one digit (or the four
// bytes of one residue's sum), so that what follows is lane arithmetic: lane l and lane l + 32 hold
// the lower and the upper half of number l's digits.
//
// For 64 moduli the products of one number are 64 x 62 word multiplications: a wave per number spent
// about 200 vector instructions on them, the matrix cores take 64 instructions for 32 numbers.
#pragma once

#include "grns_kernels.hpp"

namespace grns {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Per-modulus constants of the conversions.  Records past the set's n (up to the padded count) have
// m = 2^32 - 1 and zeros: any residue is canonical and its term is 0.
struct ModRec {
    unsigned m, w, wf;  // wf = floor(2^32 w / m)
    unsigned keeps_m;   // RN(m RN(1 / m)) < 1: a reciprocal addition leaves m where the sum is m
    double dinv, hdinv;      // RN(1 / m) and half of it
};

// Shapes for a set padded to NP in {8, 16, 32, 64} moduli (moduli below 2^31).
template <int NP>
struct Mat {
    static constexpr int KR = NP / 8;               // K steps over residues: 8 moduli of 4 bytes
    static constexpr int RT = NP / 8;               // row tiles of residues: 8 moduli of 4 bytes
    static constexpr int WT = NP / 8;               // row tiles of 32-bit words: 8 words of 4 bytes
    static constexpr int KW = NP / 8;               // K steps over words
    static constexpr int ND = (31 * NP + 27) / 28;  // 28-bit digits of M < 2^(31 NP); the top one stays below 2^27
    static constexpr int DT = (ND + 7) / 8;         // row tiles of digits: 8 digits of 4 columns of 7 bits
    static constexpr int KD = DT;                   // K steps over digits
};

// Device tables of one context (fragments in the order the wave loads them: 64 lanes x 16 bytes).
struct MatTab {
    const ModRec *rec;
    const v4i *crt8;       // [WT][KR][64]: digits of 2^(8 a) M / m_i, base 2^8 in [-128, 127]
    const int *crt8_init;  // [WT][2][16]: 128 x the row sums (the s bytes enter as b - 128)
    const int *m8;         // [2][4 WT]: M in base 2^32, digits in [-2^31, 2^31)
    const unsigned *m32;   // [2][4 WT]: M in base 2^32
    const v4i *res8;       // [RT][KW][64]: bytes in [-128, 127] of 2^(8 c) mod m_i, centred
    const int *res8_init;  // [RT][2][16]
    const unsigned *fold;  // [NP]: 2^(32 NP) mod m_i
    const v4i *crt7;       // [DT][KR][64]: digits of 2^(8 a) M / m_i, base 2^7
    const int *crt7_init;  // [DT][2][16]
    const int *m28;        // [2][4 DT]: M in base 2^28
    const v4i *res7;       // [RT][KD][64]: bytes in [-128, 127] of 2^(7 c) mod m_i, centred
};

// s_i = x_i w_i mod m_i, plus m_i at times: below 2 m_i < 2^32 for any 32-bit x_i.
GRNS_D unsigned rec_term(unsigned x, const ModRec &r) { return x * r.w - __umulhi(x, r.wf) * r.m; }

// The integer nearest below a value of the column sums in one residue's bytes (C0 .. C3), mod m:
// |C| < 2^23, so the halves fit 32 bits and the whole 2^48; (v + 1/2) / m is at least 1 / (2 m) from
// an integer, more than the product's error, so its floor is exact.
GRNS_D unsigned bytes_residue(int c0, int c1, int c2, int c3, const ModRec &r) {
    const double v = fma((double)(c2 + (c3 << 8)), 65536.0, (double)(c0 + (c1 << 8)));
    const double q = floor(fma(v, r.dinv, r.hdinv));
    return (unsigned)fma(-q, (double)r.m, v);
}

GRNS_D v16i load_init(const int *p) {
    v16i a;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const v4i t = *reinterpret_cast<const v4i *>(p + 4 * i);
        a[4 * i] = t[0]; a[4 * i + 1] = t[1]; a[4 * i + 2] = t[2]; a[4 * i + 3] = t[3];
    }
    return a;
}

// Value of another lane's register 32 lanes away.
GRNS_D int other_half(int v) { return __shfl_xor(v, 32, 64); }
GRNS_D double other_half_d(double v) { return __shfl_xor(v, 32, 64); }

// Whether four residues of consecutive moduli of one number are one aligned 16-byte word (number-major
// arrays whose number stride is a multiple of 4).
GRNS_D bool quads(const int *x, long long smod, long long snum) {
    return smod == 1 && (snum & 3) == 0 && ((uintptr_t)x & 15) == 0;
}

// Residues of the lane's moduli i = 8 ks + 4 h + b of T numbers (p[t]: residue 0 of tile t's number;
// those past n read residue 0), all in flight at once.  The rows are walked by a pointer: 32 row
// offsets per lane would otherwise be kept across the caller's loop.
template <int NP, int T>
GRNS_D void load_residues(const int *const (&p)[T], long long smod, bool quad, int n, int h,
                          v4i (&B)[T][Mat<NP>::KR]) {
#pragma unroll
    for (int t = 0; t < T; t++) {
        const int *r = p[t] + 4 * h * smod;
#pragma unroll
        for (int ks = 0; ks < Mat<NP>::KR; ks++) {
            r = lane_point(r);
            if (8 * ks + 8 <= n) {
                if (quad) {
                    B[t][ks] = *(const __attribute__((address_space(1))) v4i *)r;
                } else {
#pragma unroll
                    for (int b = 0; b < 4; b++)
                        B[t][ks][b] = __builtin_nontemporal_load((const global_int *)(r + b * smod));
                }
            } else {
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const int *q = 8 * ks + 4 * h + b < n ? r + b * smod : p[t];
                    B[t][ks][b] = *(const global_int *)q;
                }
            }
            r += 8 * smod;
        }
    }
    sched_stop();
}

// Residues to the B operand of the CRT product in place, and k = floor(sum_i s_i / m_i + 2^-30):
// sum_i s_i M_i - k M lies in [-2^-30 M, M) (the double sum is within 2^-40, so only a number within
// 2^-30 M of M may be taken for a negative one).  bad[t]: a residue of the lane's is not canonical.
template <int NP, int T>
GRNS_D void crt_operand(const ModRec *recs, int h, v4i (&B)[T][Mat<NP>::KR], int (&k)[T], LaneAny (&bad)[T]) {
    double sum[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
        sum[t] = 0.0;
    }
#pragma unroll
    for (int ks = 0; ks < Mat<NP>::KR; ks++) {
        const ModRec *rec = recs + lane_offset(4 * h);  // not hoisted out of the callers' loops
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const ModRec r = rec[8 * ks + b];
#pragma unroll
            for (int t = 0; t < T; t++) {
                const unsigned v = (unsigned)B[t][ks][b], s = rec_term(v, r);
                bad[t].set_if(v >= r.m);
                sum[t] = fma((double)s, r.dinv, sum[t]);
                B[t][ks][b] = (int)(s ^ 0x80808080u);
            }
        }
#pragma unroll
        for (int t = 0; t < T; t++) asm volatile("" : "+v"(sum[t]), "+s"(bad[t].m));  // summed here, not where they are used
        sched_stop();
    }
#pragma unroll
    for (int t = 0; t < T; t++) k[t] = (int)lane_offset((unsigned)(int)floor(sum[t] + other_half_d(sum[t]) + 0x1p-30));
}

// One number's digits in LDS: digit d < lim at p[d * sd], the others at q[d * sd].
struct DigitColumn {
    unsigned *p, *q;
    int sd, lim;
    GRNS_D unsigned &at(int d) const { return (d < lim ? p : q)[d * sd]; }
};

// Takes the carry out of the lower half's digits into the upper half's (usually one or two digits).
// Returns the carry out of the whole, -1 for a negative value, on both halves.
template <int CB>
GRNS_D int digits_join(const DigitColumn &col, int H, int h, int carry) {
    const int c0 = other_half(carry);
    int c = h ? c0 : 0;
#pragma unroll 1
    for (int k = 0; k < H && __any(c != 0); k++) {
        unsigned &d = col.at(h * H + k);
        const long long v = (long long)d + c;
        d = (unsigned)v & (unsigned)((1ull << (4 * CB)) - 1);
        c = (int)(v >> (4 * CB));
    }
    const int top = carry + c, o = other_half(top);
    return h ? top : o;
}

// The values sum_i s_i M_i - k M of the lane pair's numbers (one per tile), as digits in base 2^(4 CB)
// in LDS: lane half h writes digits 4 MT h + 0 .. 4 MT - 1 of col[t].  The column sums of one row tile
// are four digits of the half: with |C| < 2^23 the sums of two columns fit 32 bits.  MU row tiles at a
// time, so that the matrix core has independent sums to work on.  The loop over row tiles is rolled:
// unrolled, the code of a pass did not fit the instruction cache.
template <int NP, int CB, int MT, int MU, int T>
GRNS_D void crt_digits(const v4i *frags, const int *init, const int *mdig, const unsigned *mpos,
                       const v4i (&B)[T][Mat<NP>::KR], const int (&k)[T], int lane, const DigitColumn (&col)[T]) {
    constexpr int KR = Mat<NP>::KR, H = 4 * MT;
    const int h = lane >> 5;
    long long carry[T];
#pragma unroll
    for (int t = 0; t < T; t++) carry[t] = 0;
    v4i a[MU][KR];
    auto load_rows = [&](int m0) {
#pragma unroll
        for (int u = 0; u < MU; u++)
#pragma unroll
            for (int ks = 0; ks < KR; ks++) a[u][ks] = frags[((m0 + u) * KR + ks) * 64 + lane];
    };
    load_rows(0);
#pragma unroll 1
    for (int m0 = 0; m0 < MT; m0 += MU) {
        v16i acc[MU][T];
#pragma unroll
        for (int u = 0; u < MU; u++) {
            acc[u][0] = load_init(init + ((m0 + u) * 2 + h) * 16);
#pragma unroll
            for (int t = 1; t < T; t++) acc[u][t] = acc[u][0];
        }
#pragma unroll
        for (int ks = 0; ks < KR; ks++)
#pragma unroll
            for (int u = 0; u < MU; u++)
#pragma unroll
                for (int t = 0; t < T; t++)
                    acc[u][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u][ks], B[t][ks], acc[u][t], 0, 0, 0);
        sched_stop();
        load_rows(m0 + MU < MT ? m0 + MU : 0);  // the next rows arrive while the digits are formed
        sched_stop();
#pragma unroll
        for (int u = 0; u < MU; u++) {
            const v4i mw = *reinterpret_cast<const v4i *>(mdig + h * H + 4 * (m0 + u));
#pragma unroll
            for (int t = 0; t < T; t++) {
                const v16i &C = acc[u][t];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int lo = C[4 * q] + (C[4 * q + 1] << CB), hi = C[4 * q + 2] + (C[4 * q + 3] << CB);
                    const long long v = carry[t] + (long long)hi * (1 << (2 * CB)) + lo - (long long)k[t] * mw[q];
                    col[t].at(h * H + 4 * (m0 + u) + q) = (unsigned)v & (unsigned)((1ull << (4 * CB)) - 1);
                    carry[t] = v >> (4 * CB);
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < T; t++) {
        const bool neg = digits_join<CB>(col[t], H, h, (int)carry[t]) < 0;
        if (__any(neg)) {  // within 2^-30 M of M: M is added back
            long long c = 0;
#pragma unroll 1
            for (int d = h * H; d < h * H + H; d++) {
                const long long v = (long long)col[t].at(d) + (neg ? (long long)mpos[d] : 0) + c;
                col[t].at(d) = (unsigned)v & (unsigned)((1ull << (4 * CB)) - 1);
                c = v >> (4 * CB);
            }
            (void)digits_join<CB>(col[t], H, h, (int)c);
        }
    }
}

// rns_to_binary (src/rnsbase.cuh:277-287) of 32 numbers per wave and pass.  The words are formed in
// LDS; words that lie side by side in memory (word stride 1, numbers packed) leave as contiguous
// 16-byte stores: a lane's own words would touch 64 lines per store instruction.  The waves of a
// block share the table in LDS (64 KiB with 64 moduli, hence eight waves).  300007 numbers of 64 moduli:
// 308 -> 53 us; 2^20 numbers of 32 moduli 64 us, 4.1 TB/s, close to a copy's rate.
constexpr int to_binary_block(int NP) { return NP == 64 ? 512 : BLOCK; }
template <int NP>
__global__ __launch_bounds__(to_binary_block(NP), 2) void k_to_binary_mat(const DevCtx *__restrict__ c, MatTab tab,
                                                            const int *__restrict__ x, long long smod, long long snum,
                                                            long long count, unsigned *__restrict__ w, long long wst,
                                                            long long wsn) {
    constexpr int WT = Mat<NP>::WT, KR = Mat<NP>::KR, BS = to_binary_block(NP);
    __shared__ v4i table[WT * KR * 64];
    __shared__ __align__(16) int init[WT * 32], mdig[8 * WT];
    __shared__ ModRec rec[NP];
    __shared__ __align__(16) unsigned stage[BS / 64][32 * NP];
    for (int i = threadIdx.x; i < WT * KR * 64; i += BS) table[i] = tab.crt8[i];
    for (int i = threadIdx.x; i < WT * 32; i += BS) init[i] = tab.crt8_init[i];
    for (int i = threadIdx.x; i < 8 * WT; i += BS) mdig[i] = tab.m8[i];
    for (int i = threadIdx.x; i < NP; i += BS) rec[i] = tab.rec[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int n = c->n, nw = c->words - 1;
    const long long tiles = (count + 31) / 32;
    const long long wave = (long long)blockIdx.x * (BS / 64) + (threadIdx.x >> 6);
    const long long nwaves = (long long)gridDim.x * (BS / 64);
    const bool packed = wst == 1 && wsn == nw && ((uintptr_t)w & 15) == 0;
    const bool quad = quads(x, smod, snum);
    unsigned *st = stage[threadIdx.x >> 6];
    const DigitColumn col[1] = {{st + (lane & 31) * nw, st + 32 * nw + (lane & 31) * (NP - nw) - nw, 1, nw}};
    for (long long tile = wave; tile < tiles; tile += nwaves) {
        const long long j0 = tile * 32, j = j0 + (lane & 31);
        const int *p[1] = {x + (j < count ? j : count - 1) * snum};
        v4i B[1][KR];
        int k[1];
        LaneAny bad[1];
        load_residues<NP, 1>(p, smod, quad, n, h, B);
        crt_operand<NP, 1>(rec, h, B, k, bad);
        crt_digits<NP, 8, WT, WT >= 2 ? 2 : 1, 1>(table, init, mdig, tab.m32, B, k, lane, col);
        wave_lds_fence();
        const int valid = (int)(count - j0 < 32 ? count - j0 : 32);
        if (packed) {
            const int total = valid * nw;
            for (int i = 4 * lane; i < total; i += 256) {
                if (i + 4 <= total) {
                    *reinterpret_cast<uint4 *>(w + j0 * nw + i) = *reinterpret_cast<const uint4 *>(st + i);
                } else {
                    for (int e = i; e < total; e++) w[j0 * nw + e] = st[e];
                }
            }
        } else {
            for (int i = lane; i < valid * nw; i += 64) w[(j0 + i / nw) * wsn + (long long)(i % nw) * wst] = st[i];
        }
        // numbers with a residue outside [0, m_i): one after another by the whole wave
        const unsigned long long mb = bad[0].m & __ballot(j < count);
        unsigned both = (unsigned)mb | (unsigned)(mb >> 32);
        while (both) {
            const long long jb = j0 + __ffs((int)both) - 1;
            both &= both - 1;
            const Group g = make_group(64, n);
            const int xi = g.gl < n ? unsigned_long_residue(c, x[jb * snum + (long long)g.gl * smod], g.gl) : 0;
            const unsigned X = group_words<64>(c, g, xi);
            if (g.gl < nw) w[jb * wsn + (long long)g.gl * wst] = X;
        }
        wave_lds_fence();
    }
}

// rns_from_binary (src/rnsbase.cuh:253-261) of 64 numbers per wave and pass.  300007 numbers of 64
// moduli: 389 -> 64 us; 2^20 numbers of 32 moduli 64 us.  LONG: more than NP words,
// taken NP at a time, most significant first, combined by Horner's rule with 2^(32 NP) mod m.
template <int NP, bool LONG>
__global__ __launch_bounds__(BLOCK, 2) void k_from_binary_mat(const DevCtx *__restrict__ c, MatTab tab,
                                                              const unsigned *__restrict__ w, long long wst,
                                                              long long wsn, int nwords, const int *__restrict__ sign,
                                                              long long count, int *__restrict__ x, long long smod,
                                                              long long snum) {
    constexpr int RT = Mat<NP>::RT, KW = Mat<NP>::KW;
    __shared__ v4i table[RT * KW * 64];
    __shared__ __align__(16) int sinit[RT * 32];
    __shared__ ModRec rec[NP];
    for (int i = threadIdx.x; i < RT * KW * 64; i += BLOCK) table[i] = tab.res8[i];
    for (int i = threadIdx.x; i < RT * 32; i += BLOCK) sinit[i] = tab.res8_init[i];
    for (int i = threadIdx.x; i < NP; i += BLOCK) rec[i] = tab.rec[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int n = c->n;
    const int chunks = (nwords + NP - 1) / NP;
    const bool pairs = wst == 1 && (wsn & 1) == 0 && ((uintptr_t)w & 7) == 0;  // 8-byte loads
    const bool quad = quads(x, smod, snum);
    const long long tiles = (count + 63) / 64;
    const long long wave = (long long)blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    const long long nwaves = (long long)gridDim.x * (BLOCK / 64);
    for (long long tile = wave; tile < tiles; tile += nwaves) {
        long long j[2];
        j[0] = tile * 64 + (lane & 31);
        j[1] = j[0] + 32;
        bool ng[2];
        const unsigned *wp[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const long long jc = j[t] < count ? j[t] : count - 1;
            ng[t] = sign && sign[jc] != 0;
            wp[t] = w + jc * wsn;
        }
        // the residues of moduli i0 .. i0 + 3, negated for negative numbers
        auto store4 = [&](int t, int i0, const unsigned (&v)[4], const unsigned (&m)[4]) {
            v4i o;
#pragma unroll
            for (int q = 0; q < 4; q++) o[q] = (int)(ng[t] && v[q] != 0 ? m[q] - v[q] : v[q]);
            if (j[t] >= count) return;
            int *p = x + j[t] * snum + (long long)i0 * smod;
            if (quad && i0 + 4 <= n) {
                *reinterpret_cast<v4i *>(p) = o;
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (i0 + q < n) p[(long long)q * smod] = o[q];
            }
        };
        unsigned R[LONG ? 2 : 1][LONG ? 4 * RT : 1];
        for (int ch = LONG ? chunks - 1 : 0; ch >= 0; ch--) {
            v4i B[2][KW];
            const int c0 = LONG ? ch * NP : 0;
#pragma unroll
            for (int ks = 0; ks < KW; ks++) {
                const int k0 = c0 + 8 * ks + 4 * h;
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    if (pairs && k0 + 4 <= nwords) {
                        const uint2 a = *reinterpret_cast<const uint2 *>(wp[t] + k0);
                        const uint2 b = *reinterpret_cast<const uint2 *>(wp[t] + k0 + 2);
                        B[t][ks] = v4i{(int)a.x, (int)a.y, (int)b.x, (int)b.y};
                    } else {
#pragma unroll
                        for (int b = 0; b < 4; b++)
                            B[t][ks][b] = k0 + b < nwords ? (int)wp[t][(long long)(k0 + b) * wst] : 0;
                    }
                }
            }
            sched_stop();
#pragma unroll
            for (int ks = 0; ks < KW; ks++)
#pragma unroll
                for (int t = 0; t < 2; t++) B[t][ks] ^= (int)0x80808080u;
#pragma unroll LONG ? RT : 1
            for (int mt = 0; mt < RT; mt++) {
                const unsigned hl = lane_offset(h), ln = lane_offset(lane);  // no table load is hoisted
                const v16i init = load_init(sinit + (mt * 2 + hl) * 16);
                v16i acc[2] = {init, init};
#pragma unroll
                for (int ks = 0; ks < KW; ks++) {
                    const v4i a = table[(mt * KW + ks) * 64 + ln];
#pragma unroll
                    for (int t = 0; t < 2; t++)
                        acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, B[t][ks], acc[t], 0, 0, 0);
                }
const int i0 = 8 * mt + 4 * (int)hl;
                unsigned v[2][4], m[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const ModRec r = rec[i0 + q];
                    m[q] = r.m;
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        v[t][q] =
                            bytes_residue(acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3], r);
                        if constexpr (LONG) {
                            if (ch < chunks - 1)
                                v[t][q] = (unsigned)rem_trunc((long long)R[t][4 * mt + q] * tab.fold[i0 + q] + v[t][q],
                                                              (int)r.m, r.dinv);
                            R[t][4 * mt + q] = v[t][q];
                        }
                    }
                }
                if (ch == 0) {
#pragma unroll
                    for (int t = 0; t < 2; t++) store4(t, i0, v[t], m);
                }
                sched_stop();
            }
        }
    }
}

}  // namespace grns
