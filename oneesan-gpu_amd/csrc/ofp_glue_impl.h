// ofp_glue_impl.h -- a solve from half of its rows: gluing the frontier in the
// middle of the grid to its own half-turned copy.
//
// A half turn of the grid exchanges the two ends of a corner-to-corner path.  So
// the frontier vector u in the middle (after half of the cells) describes both
// halves: a path is an upper part ending in some frontier word w and a lower
// part, half-turned, ending in some word w', that meet in the same frontier
// edges and together form one path.  With G(w, w') = 1 when they do,
//
//   count = sum over words w, w' of u[w] G(w, w') u[w'].
//
// Even W: u = the main words after W/2 rows.  Odd W: u = the main and blocked
// words after (W-1)/2 rows and the cells W-1..c+1 of the middle row, c =
// (W-1)/2: the cut passes through the middle vertex, whose four edges are two on
// either side.  It lies on no path (degrees 0 + 0: position c empty in both
// words), is crossed by the path (1 + 1: occupied in both), or has both its
// edges on one side (2 + 0: a blocked word there and a main word with position c
// empty on the other side, in either order).
//
// Words meet only when their occupancies (the positions that hold R or L) are
// each other's reversal.  A word of given occupancy o with m strands is its
// label sequence from the top (R before L: rank lambda among the
// ballot(m) sequences entered at height 1), the arcs it draws between the
// strands and the path's end (the entry height).  G depends on the two label
// ranks alone: G_m[lambda][lambda'], lambda' in the half-turned numbering, is 1
// when the arcs of both halves close no loop (then the m strands lie on one path
// from end to end).  Its ones are the open meanders with m crossings (1, 2, 8, 42,
// 262, ... 8152860 for m = 1, 3, 5, 7, 9, ... 19: about 5 % of the entries at m =
// 15).  At W = 23 they are 1.3e11 additions per modulus in all, as many as two rows
// of cells, for the 11.5 rows saved.
//
// Removing an arc.  Let the topmost L of the upper word w that an R follows at once
// be on strands b+1 and b (bit numbers); they are one arc.  Without them w is a
// word w2 of m - 2 strands, and the lower words that close no loop with w are those
// that make, when the same two strands are joined, a lower word that closes none
// with w2: row(w) = the preimages(v, j) of all v in row(w2), j = m-2-b the place in
// the lower word.  The lists are built that way, m from m - 2, and sums over rows
// of more strands than are listed first pull the lower words' residues down
// through the same preimages.
//
// By the half turn the pairs (o, reversed o) and (reversed o, o) contribute
// alike, so only one of them is summed, twice -- except the occupancies of an
// odd row with position c empty, where u[w] + 2 ublocked[w] takes the place of
// u[w] on one side and both orders are summed.
#pragma once
#include <algorithm>

#include "ofp_cell_impl.h"

namespace ofp {
namespace glue {

constexpr int kMaxStrands = 27;   // odd, <= kMaxW
constexpr int kTabStrands = 19;   // G_m is listed up to this m (16 MB); sums over up to kSumStrands
constexpr int kSumStrands = 23;   // strands go down to it by removing one or two arcs
constexpr int kBaseStrands = 17;  // tables made with the context: every solve up to n = 16
constexpr int kCols = 16;         // heights of a word: <= 14 at W <= 28

// Label sequences of r strands entered at height h, never below 0, ending at 0.
struct Ballot {
    uint32_t n[kMaxStrands + 1][kMaxStrands + 3];
};
inline void build_ballot(Ballot& b) {
    for (int r = 0; r <= kMaxStrands; ++r)
        for (int h = 0; h < kMaxStrands + 3; ++h)
            b.n[r][h] = r == 0 ? (h == 0) : (h > 0 ? b.n[r - 1][h - 1] : 0) + (h + 1 < kMaxStrands + 3 ? b.n[r - 1][h + 1] : 0);
}

// Labels of the sequence with rank lambda among those of m strands: bit m-1 is
// the top strand, 1 = L.
OFP_HD uint32_t labels_of(const Ballot& b, int m, uint32_t lambda) {
    uint32_t lab = 0;
    int h = 1;
    for (int i = m - 1; i >= 0; --i) {
        const uint32_t nr = h > 0 ? b.n[i][h - 1] : 0u;
        const bool L = lambda >= nr;
        lambda -= L ? nr : 0u;
        lab |= (uint32_t)L << i;
        h += L ? 1 : -1;
    }
    return lab;
}

// Rank of the word with occupancy occ and labels lab in a height table of
// (zn, zc) pairs.  skip = 31: the main numbering; skip = c: the blocked one with
// position c removed (positions above it move down by one).
template <typename Idx>
OFP_HD Idx word_rank(const cell::Pair<Idx> (*D)[kCols], uint32_t occ, uint32_t lab, int skip) {
    Idx r = 0;
    int h = 1;
    int i = __builtin_popcount(occ);
    while (occ) {
        const int pos = 31 - __builtin_clz(occ);
        occ ^= 1u << pos;
        --i;
        const bool L = (lab >> i) & 1u;
        const cell::Pair<Idx> e = D[pos - (pos > skip ? 1 : 0)][h];
        r += L ? e.c : e.n;
        h += L ? 1 : -1;
    }
    return r;
}

// Occupancy number idx among the C(W, m) masks with m of W positions (bin[p*32+q]
// = C(p, q)).
OFP_HD uint32_t mask_of(const uint32_t* bin, int W, int m, uint32_t idx) {
    uint32_t o = 0;
    for (int pos = W - 1; pos >= 0 && m > 0; --pos) {
        const uint32_t below = bin[pos * 32 + m];  // masks that leave pos empty
        const bool set = idx >= below;
        idx -= set ? below : 0u;
        o |= (uint32_t)set << pos;
        m -= set ? 1 : 0;
    }
    return o;
}
OFP_HD uint32_t reversed_mask(uint32_t o, int W) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __brev(o) >> (32 - W);
#else
    uint32_t r = 0;
    for (int i = 0; i < W; ++i) r |= ((o >> i) & 1u) << (W - 1 - i);
    return r;
#endif
}
// What occupancy o contributes: 0 = nothing (its reversal is summed twice), 1 =
// once, 2 = twice, 3 = once with the blocked words added twice (position c of an
// odd row empty; c < 0: even W).
OFP_HD int mask_weight(uint32_t o, int W, int c) {
    if (c >= 0 && !((o >> c) & 1u)) return 3;
    const uint32_t r = reversed_mask(o, W);
    return o > r ? 0 : (o == r ? 1 : 2);
}

// Rank of a label sequence of m strands (inverse of labels_of).
OFP_HD uint32_t rank_of(const Ballot& b, int m, uint32_t lab) {
    uint32_t r = 0;
    int h = 1;
    for (int i = m - 1; i >= 0; --i) {
        const bool L = (lab >> i) & 1u;
        r += L && h > 0 ? b.n[i][h - 1] : 0u;
        h += L ? 1 : -1;
    }
    return r;
}

// Bit b of the R of a word's topmost arc between neighbouring strands b+1, b (m >= 3).
OFP_HD int top_arc(uint32_t lab) { return 31 - __builtin_clz((lab >> 1) & ~lab); }
// A word without strands b+1, b, and with labels `two` (2 bits) put back there.
OFP_HD uint32_t without_pair(uint32_t lab, int b) { return ((lab >> (b + 2)) << b) | (lab & ((1u << b) - 1u)); }
OFP_HD uint32_t with_pair(uint32_t lab, int b, uint32_t two) {
    return ((lab >> b) << (b + 2)) | (two << b) | (lab & ((1u << b) - 1u));
}

// The lower words of m strands that become v (m - 2 strands) when their strands
// j+1 and j are joined: emit(labels) for each.  Where the new strands lie, v has a
// region of the half plane bounded by the arc around it (if any) and by arcs side
// by side within it; cutting one of these and leading its ends to the new strands
// gives one word each:
//   the arc around:                  R L
//   an arc below (its L at q < j):   L L, and q turns into R
//   an arc above (its R at q >= j):  R R, and q turns into L
template <class Emit>
OFP_HD void preimages(int m, uint32_t v, int j, Emit&& emit) {
    const int n = m - 2, above = n - j;
    const int h = 1 + 2 * __builtin_popcount(v >> j) - above;  // height at the new strands
    if (h > 0) emit(with_pair(v, j, 1u));
    int H = h;
    for (int q = j - 1; q >= 0; --q) {
        const bool L = (v >> q) & 1u;
        if (L && H == h) emit(with_pair(v & ~(1u << q), j, 3u));
        if (!L && H == h) break;  // the arc around ends here
        H += L ? 1 : -1;
    }
    H = h;
    for (int q = j; q < n; ++q) {
        const bool L = (v >> q) & 1u;
        if (!L && H == h) emit(with_pair(v | (1u << q), j, 0u));
        if (L && H == h) break;  // the arc around begins here
        H += L ? -1 : 1;
    }
}
OFP_HD uint32_t preimage_count(int m, uint32_t v, int j) {
    uint32_t n = 0;
    preimages(m, v, j, [&](uint32_t) { ++n; });
    return n;
}

// ---- strands beyond the lists: the scratch of a task ----
// Entries of a task of m strands whose words are listed at `tab` strands (m = tab + 2 or
// tab + 4): the lower words (n[m][1]), then one array of m - 2 strands per place b =
// 0..m-2 of the arc removed first, then, for m = tab + 4, one of m - 4 strands per pair
// (b, b2), b2 < b: the arc removed next lies below the first one's place or around it.
OFP_HD uint32_t pair_node(int b, int b2) { return (uint32_t)(b * (b - 1) / 2 + b2); }
OFP_HD uint32_t level_arrays(int m, int removed) { return removed == 0 ? (uint32_t)(m - 1) : pair_node(m - 1, 0); }
inline uint32_t task_entries(const Ballot& b, int m, int tab) {
    uint32_t n = b.n[m][1];
    for (int r = 0; r < (m - tab) / 2; ++r) n += level_arrays(m, r) * b.n[m - 2 * r - 2][1];
    return n;
}
// Entry l of array `node` one level down, `removed` (0 or 1) arcs being gone from the m
// strands of the level read, which begins at entry `from`: add(index) for each preimage
// there.  False: no such place, the entry is never read.
template <class Add>
OFP_HD bool pull_entry(const Ballot& b, int m, int removed, uint32_t from, uint32_t node, uint32_t l, Add&& add) {
    const int M = m - 2 * removed;  // strands of the level read
    int place = (int)node;
    if (removed) {
        int b1 = 1;
        while (pair_node(b1 + 1, 0) <= node) ++b1;
        place = (int)(node - pair_node(b1, 0));
        if (place > M - 2) return false;
        from += (uint32_t)b1 * b.n[M][1];
    }
    preimages(M, labels_of(b, M - 2, l), M - 2 - place, [&](uint32_t lab) { add(from + rank_of(b, M, lab)); });
    return true;
}
// The array (at the last level) in which an upper word's list is summed; lab becomes the
// labels left at `tab` strands.
OFP_HD uint32_t upper_node(int m, int tab, uint32_t& lab) {
    const int b1 = top_arc(lab);
    lab = without_pair(lab, b1);
    if (m <= tab + 2) return (uint32_t)b1;
    const int b2 = top_arc(lab);
    lab = without_pair(lab, b2);
    return pair_node(b1, b2);
}

// Ones of G_m (open meanders with m crossings) and the most in a row, m = 1, 3, ...
constexpr uint32_t kOnes[] = {1, 2, 8, 42, 262, 1828, 13820, 110954, 933458, 8152860};
constexpr uint32_t kLongest[] = {1, 1, 2, 4, 10, 24, 66, 174, 504, 1406};
// Chunks of 64 x 8 columns that hold the lists of m strands, rows sorted by length
// in slices of 64: a slice's longest row is no longer than the mean of the slice
// before it.
inline uint32_t chunk_bound(int m, uint32_t rows) {
    const uint32_t i = (uint32_t)(m - 1) / 2;
    return kOnes[i] / 512 + kLongest[i] / 8 + (rows + 63) / 64 + 2;
}

// ---- launches of the tasks in LDS (glue_kernel) ----
// The strand counts of one launch, the most strands (the longest tasks) first: waves of a
// workgroup, waves sharing a task, most moduli per pass, resident workgroups per CU.
struct Class {
    int lo, hi, waves, team;
    int most_kc;
    uint32_t per_cu;
};
constexpr Class kClasses[] = {{19, 19, 16, 16, 2, 2}, {17, 17, 16, 16, 4, 2}, {13, 15, 4, 4, 4, 8}, {1, 11, 4, 1, 4, 8}};
constexpr double kSumLimit = 18446744073709551616.0;  // 2^64: the sums are unsigned

// One launch: teams of a workgroup, moduli of a pass, tasks, tasks of a piece per team
// (pieces go to the 8 XCDs in turn), passes and blocks (per pass and XCD: blocks / 8 / passes).
struct Shape {
    uint32_t teams, kc, tasks, piece, passes, blocks;
};

// No more than this many of `count` consecutive tasks go to one XCD ...
inline uint64_t xcd_tasks(const Shape& s, uint64_t count) {
    const uint64_t P = (uint64_t)s.piece * s.teams;
    return std::min<uint64_t>(count, ((count + 8 * P - 1) / (8 * P) + 1) * P);
}
// ... and this many of them to one of its blocks of a pass, which takes a round of `teams`
// neighbouring ones in every (blocks / 8 / passes).
inline uint64_t block_tasks(const Shape& s, uint64_t count) {
    const uint64_t round = (uint64_t)(s.blocks / 8 / s.passes) * s.teams;
    return std::min<uint64_t>(xcd_tasks(s, count), ((xcd_tasks(s, count) + round - 1) / round + 1) * s.teams);
}
// Greatest sum of the high halves of a block's products: a task of m strands adds
// kOnes[m / 2] products of two residues, whose high halves are below 2^32 each.  (The low
// halves are fewer, one per word.)
inline double block_sum(const Shape& s, const Class& c, int W, const uint32_t* bin) {
    double sum = 0;
    for (int m = c.lo; m <= c.hi && m <= W; m += 2)
        sum += (double)block_tasks(s, bin[W * 32 + m]) * kOnes[(m - 1) / 2] * 4294967296.0;
    return sum;
}

// The launch of class c at width W with records of K moduli on cus CUs: the resident
// workgroups (the LDS and registers of a class), fewer where a team would get less than
// two tasks per pass, more where a block's 64-bit sums could wrap (few CUs, or many passes:
// with 256 CUs at W = 24 from 11 moduli on).
inline Shape class_shape(const Class& c, int W, int K, int cus, const uint32_t* bin) {
    Shape s{};
    s.teams = (uint32_t)(c.waves / c.team);
    s.kc = (uint32_t)std::min(c.most_kc, K >= 4 ? 4 : (K >= 2 ? 2 : 1));
    for (int m = c.lo; m <= c.hi && m <= W; m += 2) s.tasks += bin[W * 32 + m];
    s.piece = std::min(32u, std::max(1u, s.tasks / (64u * s.teams)));
    s.passes = ((uint32_t)K + s.kc - 1) / s.kc;
    const uint32_t few = (s.tasks + 2 * s.teams - 1) / (2 * s.teams) * (((uint32_t)K + 3) / 4);
    const uint32_t blocks = std::min((uint32_t)cus * c.per_cu, std::max((uint32_t)cus, few));
    // whole rounds of 8 XCDs and all passes
    s.blocks = std::max(1u, blocks / (8 * s.passes)) * 8 * s.passes;
    while (block_sum(s, c, W, bin) >= kSumLimit) s.blocks *= 2;
    return s;
}

}  // namespace glue
}  // namespace ofp
