// cse_internal.h -- layouts shared by the kernels and the host side of the
// engine (not part of the public C ABI).
#pragma once
#include <stdint.h>

#ifndef DEV
#define DEV __device__ __forceinline__
#endif

// Projector as kernel argument: generator g is i^phase[g] Z(zs[g]) X(xs[g]).
struct DevProjector {
    int nstabs;
    int phase[64];
    uint64_t xs[64];
    uint64_t zs[64];
};

// Record of a projected state: its form on the instance's slots (cse_tree.h),
// REC_WORDS uint64 words.
//   w[0] = n << 8 | Q << 16 | sexp << 24 | vanished << 40
//   w[1] = F, the slots that hold multipliers; w[2], w[3] = d1, d2
//   w[4 .. 68)   rows of J (symmetric, no diagonal), zero beyond n
// A word's slot x is bit 31 - x of its low half (x < 32), slot 32 + x bit
// 31 - x of its high half.
#define REC_ROWS 4
#define REC_WORDS 68

// Exact mode takes, for record r, the lanes (aligned blocks of ch = 2^G j)
// that reach the diagonal: c >= floor(r / ch), nch - floor(r / ch) of them.
// Block g (records g ch .. g ch + ch - 1) thus has ch (nch - g) lanes, and
// tri_before(g) lanes precede it (ch divides chi = ch nch).
inline __host__ __device__ long long tri_before(long long ch, long long nch, long long g) {
    return ch * (g * (2 * nch - g + 1) / 2);
}

// Slot order and tree of an instance (cse_tree.h).
#define TREE_MAXLOG 30      // largest log2 chi
#define TREE_MAXG 12        // largest log2 of the terms of one lane
// Words per lane of a wave's LDS stack: the most that leaves room for four
// blocks of four waves on a CU (160 KB), next to the exact sweep's histogram
#define TREE_LDS_WORDS0 38
#define TREE_LDS_WORDS1 34
// words of a saved form besides its rows, those it has beyond 32 slots, and all
// of one on c slots
#define TREE_STATE_WORDS 5
#define TREE_HIGH_WORDS 3
constexpr int tree_words(int c) { return TREE_STATE_WORDS + (c <= 32 ? c : TREE_HIGH_WORDS + 2 * c - 32); }

// largest flush_terms (and the default): 2^30 terms keep every 32-bit bin
// below 2^32
#define CSE_FLUSH_TERMS_MAX (1ll << 30)

// copies of an instance's sums where there are several (spread_sums)
#define TREE_COPIES 8

// Histogram bins per instance: P in [-(64 + 64), 0], 8 phases (the public
// CSE_HIST_BINS).
#define HIST_STRIDE (129 * 8)
struct InstDesc {
    int n;              // state dimension t
    int k;              // index bits: rows of L, or pairs (exact)
    int exact;          // 1: |H^t> decomposition, 0: |L>
    int G;              // a lane takes the 2^G terms of its low index bits
    long long chi;      // decomposition size, 2^k
    long long lanes;    // lanes of the instance
    long long rec_off;  // first record of this instance
    long long term_off; // first per-term output slot
    uint64_t seed;      // mode 0: Philox key of the random states
    long long first;    // mode 0: sample index of the first record
    int nlds;           // levels 1 .. nlds of the stack are in LDS
    int leaf;           // levels up to this one only move the looked-up slots, or pair
    int beyond;         // stack words (per lane) outside LDS
    int levels;         // most slots of a level (tree_levels)
    int pair;           // leaf is 1, and the terms of index bit 0 are summed in pairs
    uint8_t inv[64];    // column of each slot
    uint8_t ub[TREE_MAXG + 4];    // ub[g]: slots that index bits below g move
    uint16_t soff[TREE_MAXG + 4]; // first word of level g's part of its stack
    // per index bit: the slots it toggles and the slots whose sign it toggles
    // (|H^t>), bits as in a record, and both as columns of the state
    uint64_t LP[TREE_MAXLOG];
    uint64_t LT[TREE_MAXLOG];
    uint64_t col[TREE_MAXLOG];
    uint64_t sgn[TREE_MAXLOG];
    uint32_t jmap[TREE_MAXLOG];   // the reference's index j of each bit
};

struct SweepArgs {
    int ninst;
    long long nitems;           // blocks of 256 lanes
    const long long *item_off;  // ninst + 1 prefix of items
    // mode 1: a block flushes its partial histogram of an instance once it
    // has counted this many terms of it (its LDS bins are 32-bit and a term
    // adds at most 2 to one), so no bin can wrap however long the instance
    long long flush_terms;
    const InstDesc *inst;
    const uint64_t *recs;
    unsigned long long *queue;
    uint32_t *stack;          // levels beyond LDS: stack_words x 64 per wave
    long long stack_words;
    const uint8_t *leaf;      // table of the last slots (k_leaf_table)
    int32_t *terms;           // optional per-term output
    long long *zsum;          // mode 0: 4 per record
    double *kahan;            // mode 0: 2 per record; mode 1: 2 per instance
    unsigned long long *hist; // HIST_STRIDE per instance
    unsigned long long *ips;  // per instance
    unsigned long long *clock; // readings: records, sweep, results start
    int *err;                 // bit 1: an inner product left [-64, 0]
    // k_sweep_c*: the sums above are those of copy 0; block b adds to copy
    // b mod TREE_COPIES, copies being copy_words 8-byte words apart
    unsigned copy_words;
};

#ifdef __HIPCC__
namespace cse {

struct Rec {
    static DEV void store_vanished(uint64_t *rec, int n) {
        if (lane_id() == 0) {
            rec[0] = ((uint64_t)n << 8) | (1ull << 40);
            rec[1] = 0;
            rec[2] = 0;
            rec[3] = 0;
        }
    }
};

}  // namespace cse
#endif
