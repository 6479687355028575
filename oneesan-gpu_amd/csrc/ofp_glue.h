// ofp_glue.h -- launch interface of the half-row solve's last step (ofp_glue.hip).
#pragma once
#include "ofp_glue_impl.h"

namespace ofp {
namespace glue {

// The words of one strand count: G_m as sliced lists (see ofp_glue.hip) and how
// many occupancies of the row have m strands.
struct Seg {
    int m = 0;
    uint32_t rows = 0, slices = 0, count = 0;
    const uint32_t* labels = nullptr;  // label bits by label rank
    const uint32_t* rowlab = nullptr;  // label bits of each slice's rows (~0: none)
    const uint32_t* slot = nullptr;    // slice * 64 + lane of a row, by label rank
    const uint32_t* sptr = nullptr;    // first chunk of each slice
    const uint4* cols = nullptr;
};

// Device lists of consecutive strand counts (one allocation).
struct Tables {
    char* mem = nullptr;
    Seg seg[kTabStrands + 1];
};
constexpr int kTableSets = 2;  // up to kBaseStrands, and m = 19

// Accumulators of a sum: eight sets (one per XCD's workgroups) of three 64-bit parts.
constexpr int kCopies = 8;
constexpr int kAccWords = 3 * kCopies;

struct GlueLaunch {
    const uint32_t* main;   // the frontier after half of the cells, state-major, stride K
    const uint32_t* blk;
    const void* dp;         // packed height table (cell::Quad)
    const Ballot* ballot;
    const uint32_t* binom;  // C(p, q) at p * 32 + q
    uint64_t* acc;          // kAccWords sums per modulus, zero before the first launch
    const uint32_t* mods;   // k moduli on the device, or null: mod
    uint32_t* scratch;      // lower words of a batch (more than kTabStrands strands)
    int W, K, k;
    int center;             // the cut vertex of an odd row, -1 for even W
    int segs;
    uint32_t tasks, piece, ystride, task0, batch;
    uint32_t from, to, each;  // scratch entries of a task: of the level read, of the one written, in all
    int removed;              // arcs removed at the level read
    Seg seg[6];
    uint32_t mod[kMaxKC];
};

// Lists of m_lo, m_lo + 2, ..., m_hi strands (those of m_lo - 2: below); waits for s.
hipError_t build_tables(const Ballot& hb, const Ballot* dev_ballot, int m_lo, int m_hi, const Tables* below, Tables& out,
                        hipStream_t s);
void free_tables(Tables& t);
// Scratch bytes launch_glue needs at width W (0 up to kTabStrands positions).
size_t scratch_need(const Ballot& hb, int W, int K);
// All launches of one glue on s; word 0 of main_out takes the k residues.  tabs:
// kTableSets sets, made for every strand count of the row up to kTabStrands (W <=
// kSumStrands + 1);
// binom: the host copy of a.binom.
hipError_t launch_glue(const GlueLaunch& a, const Tables* tabs, const Ballot& hb, const uint32_t* binom, bool wide, int cus,
                       size_t scratch_bytes, uint32_t* main_out, hipStream_t s, int* launches);

}  // namespace glue
}  // namespace ofp
