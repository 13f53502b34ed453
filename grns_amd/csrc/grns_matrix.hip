// grns_matrix.hip -- tables and launchers of the matrix-core conversions (grns_matrix.hpp).
#include <hip/hip_runtime.h>

#include <cstring>
#include <vector>

#include "grns_internal.hpp"
#include "grns_matrix.hpp"

using namespace grns;

namespace {

// Places of the tables in one device allocation, each on a 256-byte boundary.
struct Layout {
    size_t size = 0;
    size_t take(size_t bytes) {
        const size_t at = size;
        size = (size + bytes + 255) / 256 * 256;
        return at;
    }
};

// Digits of the words v (little-endian) in base 2^bits, `cols` of them; balanced: in
// [-2^(bits-1), 2^(bits-1)), else in [0, 2^bits).
void split_digits(const std::vector<unsigned> &v, int bits, int cols, bool balanced, std::vector<int> &out) {
    out.assign(cols, 0);
    int carry = 0;
    for (int k = 0; k < cols; k++) {
        const size_t b = (size_t)k * bits, w = b / 32;
        const unsigned long long lo = w < v.size() ? v[w] : 0u, hi = w + 1 < v.size() ? v[w + 1] : 0u;
        int d = (int)((((hi << 32) | lo) >> (b % 32)) & ((1u << bits) - 1u)) + carry;
        carry = 0;
        if (balanced && d >= (1 << (bits - 1))) {
            d -= 1 << bits;
            carry = 1;
        }
        out[k] = d;
    }
}

// Fragment order of an MFMA row operand: row r and K index kk of tile (mt, ks) at byte
// ((mt * KS + ks) * 64 + (kk / 16) * 32 + r) * 16 + kk % 16.
template <class Value>
void fill_fragments(signed char *dst, int tiles, int ksteps, Value value) {
    for (int mt = 0; mt < tiles; mt++)
        for (int ks = 0; ks < ksteps; ks++)
            for (int l = 0; l < 64; l++)
                for (int j = 0; j < 16; j++)
                    dst[((size_t)(mt * ksteps + ks) * 64 + l) * 16 + j] =
                        (signed char)value(mt, l % 32, ks * 32 + (l / 32) * 16 + j);
}
// 128 x the sum of row (mt, h, i) over K, in the order a lane of half h loads it.
template <class Value>
void fill_init(int *dst, int tiles, int ksteps, Value value) {
    for (int mt = 0; mt < tiles; mt++)
        for (int h = 0; h < 2; h++)
            for (int i = 0; i < 16; i++) {
                const int row = 8 * (i / 4) + 4 * h + i % 4;
                int sum = 0;
                for (int kk = 0; kk < ksteps * 32; kk++) sum += value(mt, row, kk);
                dst[(mt * 2 + h) * 16 + i] = 128 * sum;
            }
}

}  // namespace

// Tables for sets of up to 64 moduli below 2^31 (every int modulus).
grns_status matrix_tables_create(grns_ctx *c) {
    const int n = c->n;
    if (n > 64) return GRNS_OK;
    const int NP = n <= 8 ? 8 : n <= 16 ? 16 : n <= 32 ? 32 : 64;
    const int T8 = NP / 8, DT = ((31 * NP + 27) / 28 + 7) / 8, WW = c->h.words;
    Layout L;
    const size_t rec_at = L.take(sizeof(ModRec) * NP);
    const size_t crt8_at = L.take((size_t)T8 * T8 * 1024), crt8i_at = L.take((size_t)T8 * 32 * 4);
    const size_t m8_at = L.take((size_t)NP * 4), m32_at = L.take((size_t)NP * 4);
    const size_t res8_at = L.take((size_t)T8 * T8 * 1024), res8i_at = L.take((size_t)T8 * 32 * 4);
    const size_t fold_at = L.take((size_t)NP * 4);
    const size_t crt7_at = L.take((size_t)DT * T8 * 1024), crt7i_at = L.take((size_t)DT * 32 * 4);
    const size_t m28_at = L.take((size_t)DT * 8 * 4), res7_at = L.take((size_t)T8 * DT * 1024);
    std::vector<unsigned char> host(L.size, 0);

    ModRec *rec = reinterpret_cast<ModRec *>(host.data() + rec_at);
    for (int i = 0; i < NP; i++) {
        std::memset(&rec[i], 0, sizeof(ModRec));
        rec[i].m = 0xffffffffu;
        if (i < n) {
            rec[i].m = (unsigned)c->h.m[i];
            rec[i].w = (unsigned)c->h.w[i];
            rec[i].wf = c->h.wf_hi[i];
            rec[i].keeps_m = (double)c->h.m[i] * c->h.dinv[i] < 1.0;
            rec[i].dinv = c->h.dinv[i];
            rec[i].hdinv = 0.5 * c->h.dinv[i];
        }
    }
    // digits of 2^(8 a) M / m_i in base 2^bits, one vector per K index 4 i + a; row (mt, q, h, b) is
    // column b of digit 4 tiles h + 4 mt + q
    std::vector<std::vector<int>> crt((size_t)4 * NP);
    auto crt_digits_of = [&](int bits, int tiles, bool balanced) {
        for (int i = 0; i < n; i++)
            for (int a = 0; a < 4; a++) {
                std::vector<unsigned> v(WW + 1, 0u);
                for (int k = 0; k < WW; k++) {
                    const unsigned long long t = (unsigned long long)c->crt[(size_t)i * WW + k] << (8 * a);
                    v[k] |= (unsigned)t;
                    v[k + 1] = (unsigned)(t >> 32);
                }
                split_digits(v, bits, 32 * tiles, balanced, crt[(size_t)4 * i + a]);
            }
    };
    auto crt_value = [&](int tiles) {
        return [&crt, tiles](int mt, int row, int kk) {
            const std::vector<int> &d = crt[kk];
            const int q = row / 8, h = (row % 8) / 4, b = row % 4;
            return d.empty() ? 0 : d[4 * (4 * tiles * h + 4 * mt + q) + b];
        };
    };
    crt_digits_of(8, T8, true);
    fill_fragments(reinterpret_cast<signed char *>(host.data() + crt8_at), T8, T8, crt_value(T8));
    fill_init(reinterpret_cast<int *>(host.data() + crt8i_at), T8, T8, crt_value(T8));
    crt_digits_of(7, DT, false);
    fill_fragments(reinterpret_cast<signed char *>(host.data() + crt7_at), DT, T8, crt_value(DT));
    fill_init(reinterpret_cast<int *>(host.data() + crt7i_at), DT, T8, crt_value(DT));
    {
        int *m8 = reinterpret_cast<int *>(host.data() + m8_at);
        unsigned *m32 = reinterpret_cast<unsigned *>(host.data() + m32_at);
        unsigned carry = 0;
        for (int k = 0; k < NP; k++) {
            m32[k] = k < WW ? c->crt[(size_t)n * WW + k] : 0u;
            const unsigned long long v = (unsigned long long)m32[k] + carry;
            m8[k] = (int)(unsigned)v;
            carry = v >= 0x80000000ull ? 1u : 0u;  // the digit is v - 2^32
        }
        std::vector<int> d28;
        split_digits(std::vector<unsigned>(c->crt.begin() + (size_t)n * WW, c->crt.end()), 28, 8 * DT, false, d28);
        std::memcpy(host.data() + m28_at, d28.data(), d28.size() * 4);
    }
    // bytes of 2^(bits c) mod m_i, centred; K index c is byte (or 7-bit piece) c of the integer, row
    // (mt, q, h, b) byte b of modulus 8 mt + 4 h + q
    std::vector<std::vector<int>> pw(NP);
    auto powers = [&](int bits, int cols) {
        for (int i = 0; i < NP; i++) {
            pw[i].assign(cols, 0);
            if (i >= n) continue;
            const long long m = c->h.m[i];
            long long p = 1 % m;
            for (int k = 0; k < cols; k++) {
                pw[i][k] = (int)(p > m / 2 ? p - m : p);
                p = (p << bits) % m;
            }
            if (bits == 8) reinterpret_cast<unsigned *>(host.data() + fold_at)[i] = (unsigned)p;
        }
    };
    auto res_value = [&](int mt, int row, int kk) {
        const int q = row / 8, h = (row % 8) / 4, b = row % 4;
        const unsigned t = (unsigned)pw[8 * mt + 4 * h + q][kk] + 0x80808080u;
        return (int)((t >> (8 * b)) & 255u) - 128;
    };
    powers(8, 4 * NP);
    fill_fragments(reinterpret_cast<signed char *>(host.data() + res8_at), T8, T8, res_value);
    fill_init(reinterpret_cast<int *>(host.data() + res8i_at), T8, T8, res_value);
    powers(7, 32 * DT);
    fill_fragments(reinterpret_cast<signed char *>(host.data() + res7_at), T8, DT, res_value);

    if (hipMalloc(&c->d_mat, L.size) != hipSuccess) return GRNS_ERR_OOM;
    if (hipMemcpy(c->d_mat, host.data(), L.size, hipMemcpyHostToDevice) != hipSuccess) return GRNS_ERR_HIP;
    unsigned char *d = c->d_mat;
    c->mat.rec = reinterpret_cast<const ModRec *>(d + rec_at);
    c->mat.crt8 = reinterpret_cast<const v4i *>(d + crt8_at);
    c->mat.crt8_init = reinterpret_cast<const int *>(d + crt8i_at);
    c->mat.m8 = reinterpret_cast<const int *>(d + m8_at);
    c->mat.m32 = reinterpret_cast<const unsigned *>(d + m32_at);
    c->mat.res8 = reinterpret_cast<const v4i *>(d + res8_at);
    c->mat.res8_init = reinterpret_cast<const int *>(d + res8i_at);
    c->mat.fold = reinterpret_cast<const unsigned *>(d + fold_at);
    c->mat.crt7 = reinterpret_cast<const v4i *>(d + crt7_at);
    c->mat.crt7_init = reinterpret_cast<const int *>(d + crt7i_at);
    c->mat.m28 = reinterpret_cast<const int *>(d + m28_at);
    c->mat.res7 = reinterpret_cast<const v4i *>(d + res7_at);
    return GRNS_OK;
}

namespace {

// Persistent grid of the conversions: `per_cu` blocks per CU, or one per `numbers` numbers (a block's
// pass) when there are fewer.
unsigned grid_mat(const grns_ctx *c, size_t count, int numbers, int per_cu) {
    const long long need = (long long)((count + numbers - 1) / numbers);
    const long long most = (long long)c->cus * per_cu;
    return (unsigned)(need < most ? need : most);
}

}  // namespace

grns_status matrix_to_binary(grns_ctx *c, const int *x, long long smod, long long snum, size_t count, unsigned *w,
                             long long wst, long long wsn, hipStream_t s) {
    const long long cnt = (long long)count;
    const int NP = c->n <= 8 ? 8 : c->n <= 16 ? 16 : c->n <= 32 ? 32 : 64;
#define GRNS_TO_CASE(NN)                                                                                            \
    case NN:                                                                                                        \
        hipLaunchKernelGGL((k_to_binary_mat<NN>), dim3(grid_mat(c, count, to_binary_block(NN) / 2, NN == 64 ? 1 : 4)),  \
                           dim3(to_binary_block(NN)), 0, s, c->d, c->mat, x, smod, snum, cnt, w, wst, wsn);         \
        break;
    switch (NP) {
        GRNS_TO_CASE(8)
        GRNS_TO_CASE(16)
        GRNS_TO_CASE(32)
        GRNS_TO_CASE(64)
    }
#undef GRNS_TO_CASE
    return hipGetLastError() == hipSuccess ? GRNS_OK : GRNS_ERR_HIP;
}

grns_status matrix_from_binary(grns_ctx *c, const unsigned *w, long long wst, long long wsn, int nwords, const int *sign,
                               size_t count, int *x, long long smod, long long snum, hipStream_t s) {
    const dim3 grid(grid_mat(c, count, BLOCK, c->n <= 32 ? 4 : 2)), blk(BLOCK);
    const long long cnt = (long long)count;
    const int NP = c->n <= 8 ? 8 : c->n <= 16 ? 16 : c->n <= 32 ? 32 : 64;
#define GRNS_FROM_CASE(NN)                                                                                      \
    case NN:                                                                                                    \
        if (nwords <= NN) hipLaunchKernelGGL((k_from_binary_mat<NN, false>), grid, blk, 0, s, c->d, c->mat, w, wst, wsn, \
                                             nwords, sign, cnt, x, smod, snum);                                 \
        else hipLaunchKernelGGL((k_from_binary_mat<NN, true>), grid, blk, 0, s, c->d, c->mat, w, wst, wsn, nwords, sign,  \
                                cnt, x, smod, snum);                                                            \
        break;
    switch (NP) {
        GRNS_FROM_CASE(8)
        GRNS_FROM_CASE(16)
        GRNS_FROM_CASE(32)
        GRNS_FROM_CASE(64)
    }
#undef GRNS_FROM_CASE
    return hipGetLastError() == hipSuccess ? GRNS_OK : GRNS_ERR_HIP;
}
