// grns_internal.hpp -- library-internal declarations shared by the host translation units.
#pragma once

#include <mutex>
#include <vector>

#include "../../include/grns.h"
#include "grns_kernels.hpp"
#include "grns_matrix.hpp"

struct grns_ctx {
    int device = 0;
    int n = 0;
    int log2M = 0;
    grns::DevCtx h;                // host copy of the device constants
    grns::DevCtx *d = nullptr;     // device constants
    int *d_pow2 = nullptr;
    int *d_mrc = nullptr;
    int *d_mrc_acc = nullptr;     // DevCtx::mrc_acc
    int *d_status = nullptr;
    unsigned char *d_mat = nullptr;  // tables of the matrix-core conversions (sets of up to 64 moduli)
    grns::MatTab mat = {};           // their device addresses
    unsigned *d_crt = nullptr;      // DevCtx::crt_words
    int max_blocks = 2048;         // arg-max stage-1 grid, from the occupancy query (max_grid_for)
    int max_blocks_occ = 2048;     // the same as set at context creation (test hooks restore it)
    int max_blocks_nm = 1024;      // the most blocks of it over a number-major array (resident ones)
    // rare-item queues of the per-call eval / cmp kernels, one per stream (made on first use)
    struct RareQueue {
        void *stream;
        long long *items;
        unsigned *ctr;
        int *res;  // staged residues of the first queued items
    };
    std::mutex qmu;
    std::vector<RareQueue> queues;
    // optional timing of the first (streaming) kernel of eval / cmp / max: HIP events recorded on
    // the caller's stream around that kernel while enabled; pairs are reused round-robin and folded
    // into the total before reuse
    struct StageTimer {
        std::vector<void *> ev;    // 2 * slots events (start, end)
        std::vector<char> pending;  // slot holds an unread pair
        int next = 0;
        double ms = 0.0;
        long long launches = 0;
    };
    bool timing = false;
    bool reference_loops = false;  // division and scaling: the reference loops for every number (test hook)
    bool rare_staging = true;      // rare queues stage the residues of queued numbers (test hook)
    bool rare_spread = true;       // rare items spread over the sub-queues (test hook)
    int cus = 0;                   // compute units of the device
    int grid_cap = 0;              // streaming kernels: at most grid_cap x cus blocks (0: one per BLOCK numbers)
    StageTimer timers[3];
    std::vector<int> pow2;
    std::vector<int> mrc;
    std::vector<int> mrc_acc;
    std::vector<unsigned> crt;
};

namespace grns {
inline int groups_for(int n) {
    int G = 1;
    while (G < n) G <<= 1;
    return G;
}
}  // namespace grns

// Lanes per number of the word division: a power of two with room for every residue and every
// word of the CRT sum (0: no group of 64 lanes has room).
inline int words_group(const grns_ctx *c) {
    int G = grns::groups_for(c->n);
    while (G < c->h.words) G <<= 1;
    return G <= 64 ? G : 0;
}

// Conversions of at least this many numbers run on the matrix cores, shorter ones with a wave group per
// number.  A wave of the matrix form takes 32 or 64 numbers and first loads its tables, so short
// calls leave the chip idle: with 64 moduli 8192 numbers take 11-14 us by groups and 11-15 us on the
// matrix cores, 16384 take 21-25 us and 11-15 us; with 32 moduli both take 8.5-9.5 us at 8192
// numbers, and 16384 take 10-12 us and 8.5-9.5 us.
inline size_t matrix_min(const grns_ctx *c) { return c->n > 32 ? 16384 : 8192; }

// Matrix-core conversions (grns_matrix.hip): tables at context creation, and the launches.
grns_status matrix_tables_create(grns_ctx *c);
grns_status matrix_to_binary(grns_ctx *c, const int *x, long long smod, long long snum, size_t count, unsigned *w,
                             long long wst, long long wsn, hipStream_t s);
grns_status matrix_from_binary(grns_ctx *c, const unsigned *w, long long wst, long long wsn, int nwords, const int *sign,
                               size_t count, int *x, long long smod, long long snum, hipStream_t s);
// Divisions of at least this many pairs take a lane per pair (grns_divide.hip), shorter ones a wave
// group per pair: 64 pairs to a wave leave the chip idle below.  By groups and by lanes: 16384 pairs with
// divisors of uniform length 14 and 18 us (8 moduli), 34 and 24 us (16), 54 and 38 us (32), 103 and 82 us
// (64), with divisors as long as the dividend 12 and 16, 18 and 18, 22 and 30, 46 and 57 us; 32768 pairs of
// 32 moduli 91 and 40, 39 and 30 us, of 64 moduli 189 and 85, 84 and 57 us, of 8 moduli 25 and 18, 16 and
// 17 us.  Hence a higher line for the sets whose short quotients the groups finish sooner.
inline size_t div_lanes_min(const grns_ctx *c) { return c->n > 16 ? 32768 : c->n > 8 ? 16384 : 22528; }

// Lane-per-pair division (grns_divide.hip): pairs it does not take go to the rare queue.
grns_status matrix_div(grns_ctx *c, const int *x, const int *d, long long smod, long long snum, size_t count, int *q,
                       int *r, const grns::RareQ &rq, hipStream_t s);
// Scalings of at least this many numbers take their digits from the matrix cores (grns_scale.hip), 32
// numbers to a wave; shorter ones a wave group per number.  By groups and by 32s, 16384 numbers of 8,
// 16, 32, 64 moduli take 9, 16, 24, 54 us and 10, 18, 38, 83 us; 32768 take 12, 27, 39, 98 us and 10,
// 18, 38, 87 us.
constexpr size_t SCALE_MATRIX_MIN = 32768;
grns_status matrix_scale(grns_ctx *c, const int *x, long long smod, long long snum, const unsigned *D, size_t count,
                         int *y, hipStream_t s);
