// ofp_glue.hip -- the sum over meeting word pairs that ends a solve after half of
// its rows (the identity, G_m and its tables: ofp_glue_impl.h), for gfx950.
//
// A task is one occupancy o with m strands.  Its lower words' residues (occupancy
// reversed, label ranks 0..B-1) are loaded into LDS once; then each lane takes an
// upper word lambda, adds the lower words of its list (row lambda of G_m) and
// multiplies the sum by its own residue.  Every word of the state is loaded once
// as an upper and once as a lower word, the additions are LDS gathers: at W = 23
// one task of m = 17 is 933,458 of them per modulus on 4862 loaded words.
//
//  * Lists: rows sorted by length, slices of 64 rows (one wave), 8 columns of 16
//    bits per lane and chunk, so a wave reads its lists as whole 1 KB chunks.
//    Shorter rows are filled up with column B, a zero entry.
//  * LDS: KC moduli per pass, KC chosen so that the B entries fit: 4 up to m = 17
//    (78 KB), 2 at m = 19 (134 of the 160 KB).  A team
//    of waves shares one task: one wave up to m = 11 (132 rows), a workgroup of 4
//    waves for m = 13 and 15, of 16 above.
//  * m = 21 (58786 words, 235 KB at one modulus) and 23: the lower words are
//    gathered into a scratch array in HBM and pulled down to 19 strands, one array
//    per place of the removed arc (two arcs: per pair of places); each upper word
//    then sums the list of what is left of it in its own array, from the L2s.
//  * Sums of residues stay below 2^46 and are multiplied in two halves into 64-bit
//    sums, reduced once per lane at the end: no division per word.
#include <algorithm>

#include "ofp_glue.h"

namespace ofp {
namespace glue {

namespace {

using cell::addm;
using cell::Pair;
using cell::Quad;

template <int KC>
__device__ __forceinline__ void load_rec(const uint32_t* base, uint64_t i, int K, int off, uint32_t (&v)[KC]) {
    const uint32_t* q = base + i * (uint64_t)(uint32_t)K + (uint32_t)off;
    if (off + KC <= K) {
        cell::load_words<KC>(q, v);
    } else {
#pragma unroll
        for (int j = 0; j < KC; ++j) v[j] = off + j < K ? q[j] : 0u;
    }
}

// The moduli of lanes off..off+KC-1 (lanes past the k moduli: a valid one).
template <int KC>
__device__ __forceinline__ void load_mods(const GlueLaunch& a, int off, uint32_t (&mod)[KC]) {
#pragma unroll
    for (int j = 0; j < KC; ++j) {
        const int i = off + j < a.k ? off + j : 0;
        mod[j] = a.mods ? a.mods[i] : a.mod[i];
    }
}

template <typename Idx>
__device__ void load_height(Pair<Idx> (*D)[kCols], const void* dp) {
    const Quad<Idx>* g = static_cast<const Quad<Idx>*>(dp);
    for (int t = threadIdx.x; t < kMaxW * kCols; t += blockDim.x) {
        const Quad<Idx> e = g[(t / kCols) * kDpCols + t % kCols];
        D[t / kCols][t % kCols] = Pair<Idx>{e.zn, e.zc};
    }
}

// Products x * (sum of residues), summed over words: lo collects the low 32 bits
// of the low-half products, hi everything above.
template <int KC>
struct Sum {
    uint64_t lo[KC], hi[KC];
    __device__ __forceinline__ void init() {
#pragma unroll
        for (int j = 0; j < KC; ++j) lo[j] = hi[j] = 0;
    }
    __device__ __forceinline__ void add(const uint32_t (&x)[KC], const uint64_t (&acc)[KC]) {
#pragma unroll
        for (int j = 0; j < KC; ++j) {
            const uint64_t p = (uint64_t)x[j] * (uint32_t)acc[j];
            lo[j] += (uint32_t)p;
            hi[j] += (p >> 32) + (uint64_t)x[j] * (uint32_t)(acc[j] >> 32);
        }
    }
    // The workgroup's sums (of moduli off..) into one of the kCopies sets of
    // accumulators: per modulus the low sums, and the high sums in two halves (a
    // workgroup's cannot wrap: block_sum), reduced by the last kernel.
    template <int NT>
    __device__ void flush(const GlueLaunch& a, int off) {
        __shared__ unsigned long long part[NT / 64][2 * KC];
        const int wave = (int)threadIdx.x >> 6;
#pragma unroll
        for (int j = 0; j < KC; ++j) {
            for (int d = 32; d >= 1; d >>= 1) {
                lo[j] += __shfl_xor((unsigned long long)lo[j], d);
                hi[j] += __shfl_xor((unsigned long long)hi[j], d);
            }
            if ((threadIdx.x & 63) == 0) {
                part[wave][j] = lo[j];
                part[wave][KC + j] = hi[j];
            }
        }
        __syncthreads();
        const int j = (int)threadIdx.x;
        if (j < KC && off + j < a.k) {
            unsigned long long l = 0, h = 0;
            for (int w = 0; w < NT / 64; ++w) {
                l += part[w][j];
                h += part[w][KC + j];
            }
            unsigned long long* acc =
                reinterpret_cast<unsigned long long*>(a.acc) + (size_t)(blockIdx.x & (kCopies - 1)) * 3 * a.k + off + j;
            atomicAdd(acc, l);
            atomicAdd(acc + a.k, h & 0xffffffffull);
            atomicAdd(acc + 2 * a.k, h >> 32);
        }
    }
};

// Residue of the upper word (occ, lab) with the weight of its occupancy.
template <int KC, typename Idx>
__device__ __forceinline__ void load_upper(const GlueLaunch& a, const Pair<Idx> (*D)[kCols], uint32_t occ, uint32_t lab,
                                           int weight, int off, const uint32_t (&mod)[KC], uint32_t (&x)[KC]) {
    load_rec<KC>(a.main, (uint64_t)word_rank<Idx>(D, occ, lab, 31), a.K, off, x);
    if (weight == 3) {
        uint32_t z[KC];
        load_rec<KC>(a.blk, (uint64_t)word_rank<Idx>(D, occ, lab, a.center), a.K, off, z);
#pragma unroll
        for (int j = 0; j < KC; ++j) x[j] = addm(addm(x[j], z[j], mod[j]), z[j], mod[j]);
    } else if (weight == 2) {
#pragma unroll
        for (int j = 0; j < KC; ++j) x[j] = addm(x[j], x[j], mod[j]);
    }
}

template <int KC>
struct alignas(KC * 4) Entry {
    uint32_t v[KC];
};

// Sum over the chunks of one slice's lists for this lane, entries at y.
template <int KC, class Y>
__device__ __forceinline__ void add_lists(const Seg& g, uint32_t slice, const Y& y, uint64_t (&acc)[KC]) {
#pragma unroll
    for (int j = 0; j < KC; ++j) acc[j] = 0;
    const uint32_t c1 = g.sptr[slice + 1];
    const uint4* cols = g.cols + (size_t)(threadIdx.x & 63);
    uint32_t c = g.sptr[slice];
    uint4 next = cols[(size_t)c * 64];  // the next chunk is loaded while one is added
    for (; c < c1; ++c) {
        const uint32_t w[4] = {next.x, next.y, next.z, next.w};
        if (c + 1 < c1) next = cols[(size_t)(c + 1) * 64];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const Entry<KC> e0 = y(w[i] & 0xffffu), e1 = y(w[i] >> 16);
#pragma unroll
            for (int j = 0; j < KC; ++j) acc[j] += (uint64_t)e0.v[j] + e1.v[j];
        }
    }
}

// Tasks in LDS: teams of TW waves, one occupancy per team at a time.  The words of
// one occupancy lie scattered, but next to those of the occupancies that differ in
// the lowest positions -- the tasks with the next numbers -- and a record's moduli
// are read by different passes.  So block b works on XCD b % 8 (round-robin
// dispatch), the passes of a task are neighbouring blocks of one XCD, and the tasks
// go to the XCDs in pieces of a.piece per team (32, fewer where an XCD would get less
// than eight pieces): what one fetches from HBM the others find in that XCD's L2.
template <int KC, typename Idx, int NT, int TW>
__global__ __launch_bounds__(NT) void glue_kernel(GlueLaunch a) {
    constexpr int kTeams = NT / 64 / TW;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ Pair<Idx> D[kMaxW][kCols];
    __shared__ uint32_t binom[kMaxW * 32];
    load_height<Idx>(D, a.dp);
    for (int t = threadIdx.x; t < a.W * 32; t += NT) binom[t] = a.binom[t];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int team = wave / TW, tlane = (int)threadIdx.x - team * TW * 64;
    Entry<KC>* y = reinterpret_cast<Entry<KC>*>(lds + (size_t)team * a.ystride);
    const uint32_t xcd = blockIdx.x & 7u, local = blockIdx.x >> 3, passes = (uint32_t)(a.K + KC - 1) / KC;
    const uint32_t nw = (gridDim.x >> 3) / passes;  // blocks of one pass on one XCD
    const int off = (int)(local % passes) * KC;
    uint32_t mod[KC];
    load_mods<KC>(a, off, mod);
    Sum<KC> sum;
    sum.init();
    __syncthreads();
    const uint32_t P = a.piece * kTeams;
    for (uint32_t q = local / passes * kTeams;; q += nw * kTeams) {
        const uint32_t first = (q / P * 8 + xcd) * P + q % P;
        if (first >= a.tasks) break;  // later rounds lie higher
        const uint32_t t = first + (uint32_t)team;
        if (t >= a.tasks) continue;   // (one-wave teams only: no barrier in their rounds)
        int gi = 0;
        uint32_t idx = t;
        while (idx >= a.seg[gi].count) idx -= a.seg[gi++].count;
        const Seg& g = a.seg[gi];
        const uint32_t occ = __builtin_amdgcn_readfirstlane((int)mask_of(binom, a.W, g.m, idx));
        const int weight = mask_weight(occ, a.W, a.center);
        if (!weight) continue;
        const uint32_t rocc = reversed_mask(occ, a.W);
        for (uint32_t l = tlane; l <= g.rows; l += TW * 64) {
            Entry<KC> e{};
            if (l < g.rows) load_rec<KC>(a.main, (uint64_t)word_rank<Idx>(D, rocc, g.labels[l], 31), a.K, off, e.v);
            y[l] = e;
        }
        if constexpr (TW > 1) __syncthreads();
        else __threadfence_block();
        for (uint32_t s = wave - team * TW; s < g.slices; s += TW) {
            const uint32_t lab = g.rowlab[s * 64 + (threadIdx.x & 63)];
            const bool valid = lab != ~0u;
            uint32_t x[KC] = {};
            if (valid) load_upper<KC, Idx>(a, D, occ, lab, weight, off, mod, x);
            uint64_t acc[KC];
            add_lists<KC>(g, s, [&](uint32_t c) { return y[c]; }, acc);
            sum.add(x, acc);
        }
        if constexpr (TW > 1) __syncthreads();
        else __threadfence_block();
    }
    sum.template flush<NT>(a, off);
}

// ---- strands beyond the lists ----
// Entry i of a task's scratch (a.each of K residues; laid out as pull_entry says).
__device__ __forceinline__ uint32_t* entry(const GlueLaunch& a, uint32_t task, uint32_t i) {
    return a.scratch + ((uint64_t)task * a.each + i) * (uint32_t)a.K;
}
__device__ void load_ballot(Ballot& b, const Ballot* g) {
    for (int t = threadIdx.x; t < (int)(sizeof(Ballot) / 4); t += blockDim.x) (&b.n[0][0])[t] = (&g->n[0][0])[t];
}

template <typename Idx>
__global__ __launch_bounds__(256) void glue_gather_kernel(GlueLaunch a) {
    __shared__ Pair<Idx> D[kMaxW][kCols];
    __shared__ Ballot b;
    load_height<Idx>(D, a.dp);
    load_ballot(b, a.ballot);
    __syncthreads();
    const Seg& g = a.seg[0];
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t t = (uint32_t)(i / g.rows), l = (uint32_t)(i - (uint64_t)t * g.rows);
    if (t >= a.batch) return;
    const uint32_t occ = mask_of(a.binom, a.W, g.m, a.task0 + t);
    if (!mask_weight(occ, a.W, a.center)) return;
    uint32_t* out = entry(a, t, l);
    const uint64_t r = (uint64_t)word_rank<Idx>(D, reversed_mask(occ, a.W), labels_of(b, g.m, l), 31);
    const uint32_t* src = a.main + r * (uint64_t)(uint32_t)a.K;
    for (int j = 0; j < a.K; ++j) out[j] = src[j];
}

// One level down: entry v of every array of M - 2 strands = the sum over the
// preimages of v in its array of M strands.  One thread per (task, array, v).
template <int KC>
__global__ __launch_bounds__(256) void glue_pull_kernel(GlueLaunch a, uint32_t arrays) {
    __shared__ Ballot b;
    load_ballot(b, a.ballot);
    __syncthreads();
    const int m = a.seg[0].m;
    const uint32_t rows = b.n[m - 2 * a.removed - 2][1];
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t ta = (uint32_t)(i / rows), l = (uint32_t)(i - (uint64_t)ta * rows);
    const uint32_t t = ta / arrays, node = ta - t * arrays;
    if (t >= a.batch) return;
    if (!mask_weight(mask_of(a.binom, a.W, m, a.task0 + t), a.W, a.center)) return;
    const int off = (int)blockIdx.y * KC;
    uint32_t mod[KC], sum[KC] = {};
    load_mods<KC>(a, off, mod);
    const bool place = pull_entry(b, m, a.removed, a.from, node, l, [&](uint32_t src) {
        uint32_t e[KC];
        load_rec<KC>(entry(a, t, src), 0, a.K, off, e);
#pragma unroll
        for (int j = 0; j < KC; ++j) sum[j] = addm(sum[j], e[j], mod[j]);
    });
    if (!place) return;
    uint32_t* out = entry(a, t, a.to + node * rows + l) + off;
#pragma unroll
    for (int j = 0; j < KC; ++j)
        if (off + j < a.K) out[j] = sum[j];
}

// One thread per (task, upper word): its arcs removed down to kTabStrands, its list
// summed in the array of their places (at a.from).
template <int KC, typename Idx>
__global__ __launch_bounds__(256) void glue_big_kernel(GlueLaunch a) {
    __shared__ Pair<Idx> D[kMaxW][kCols];
    __shared__ Ballot b;
    load_height<Idx>(D, a.dp);
    load_ballot(b, a.ballot);
    __syncthreads();
    const Seg &g = a.seg[0], &lists = a.seg[1];
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t t = (uint32_t)(i / g.rows), l = (uint32_t)(i - (uint64_t)t * g.rows);
    const int off = (int)blockIdx.y * KC;
    uint32_t mod[KC];
    load_mods<KC>(a, off, mod);
    Sum<KC> sum;
    sum.init();
    uint32_t occ = 0;
    int weight = 0;
    if (t < a.batch) {
        occ = mask_of(a.binom, a.W, g.m, a.task0 + t);
        weight = mask_weight(occ, a.W, a.center);
    }
    if (weight) {
        uint32_t lab = labels_of(b, g.m, l);
        uint32_t x[KC];
        load_upper<KC, Idx>(a, D, occ, lab, weight, off, mod, x);
        const uint32_t node = upper_node(g.m, kTabStrands, lab);
        const uint32_t* y = entry(a, t, a.from + node * lists.rows);
        const uint32_t slot = lists.slot[rank_of(b, kTabStrands, lab)], s = slot >> 6;
        const uint4* cols = lists.cols + (slot & 63u);
        uint64_t acc[KC] = {};
        for (uint32_t c = lists.sptr[s]; c < lists.sptr[s + 1]; ++c) {
            const uint4 q = cols[(size_t)c * 64];
            const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                const uint32_t col = (w[p >> 1] >> (16 * (p & 1))) & 0xffffu;
                if (col >= lists.rows) break;  // the filling after the row's end
                uint32_t e[KC];
                load_rec<KC>(y, col, a.K, off, e);
#pragma unroll
                for (int j = 0; j < KC; ++j) acc[j] += e[j];
            }
        }
        sum.add(x, acc);
    }
    sum.template flush<256>(a, off);
}

// The answer word (index 0) takes the sums, one wave per modulus: low + 2^32 (mid +
// 2^32 high), each below 2^64 over all waves.
__global__ __launch_bounds__(64) void glue_finish_kernel(GlueLaunch a, uint32_t* main) {
    const int j = (int)blockIdx.x, lane = (int)threadIdx.x;
    const uint64_t m = a.mods ? a.mods[j] : a.mod[j];
    uint64_t v = lane < kAccWords ? a.acc[(size_t)lane * a.k + j] % m : 0;  // lane = copy * 3 + part
    const uint64_t two32 = (1ull << 32) % m;
    const int part = lane % 3;
    if (part >= 1) v = v * two32 % m;
    if (part == 2) v = v * two32 % m;
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor((unsigned long long)v, d);
    if (lane == 0) main[j] = (uint32_t)(v % m);
}

// ---- lists, m strands from m - 2 ----
// Labels and row lengths of m strands (one thread per row).
__global__ __launch_bounds__(64) void glue_count_kernel(const Ballot* ballot, Seg g, Seg below, uint32_t* labels,
                                                        uint32_t* counts) {
    __shared__ Ballot b;
    load_ballot(b, ballot);
    __syncthreads();
    const uint32_t l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= g.rows) return;
    const uint32_t lab = labels_of(b, g.m, l);
    labels[l] = lab;
    if (g.m == 1) {
        counts[l] = 1;
        return;
    }
    const int p = top_arc(lab), j = g.m - 2 - p;
    const uint32_t slot = below.slot[rank_of(b, g.m - 2, without_pair(lab, p))], s = slot >> 6;
    const uint16_t* cols = reinterpret_cast<const uint16_t*>(below.cols + (slot & 63u));
    uint32_t n = 0;
    for (uint32_t i = 0; i < (below.sptr[s + 1] - below.sptr[s]) * 8; ++i) {
        const uint32_t c = cols[((size_t)(below.sptr[s] + (i >> 3)) * 64) * 8 + (i & 7u)];
        if (c >= below.rows) break;
        n += preimage_count(g.m, below.labels[c], j);
    }
    counts[l] = n;
}

// Rows by falling length (a counting sort in one workgroup): slot of each row, row
// of each slot, first chunk of each slice.
constexpr int kLengths = 2048;  // > kLongest
__global__ __launch_bounds__(1024) void glue_order_kernel(uint32_t rows, uint32_t chunk0, const uint32_t* counts,
                                                          uint32_t* slot, uint32_t* order, uint32_t* sptr) {
    __shared__ uint32_t at[kLengths], part[1024];
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < kLengths; i += 1024) at[i] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < rows; i += 1024) atomicAdd(&at[kLengths - 1 - counts[i]], 1u);
    __syncthreads();
    // exclusive prefix over the lengths, longest first (two bins per thread)
    const uint32_t n0 = at[2 * tid], n1 = at[2 * tid + 1];
    part[tid] = n0 + n1;
    __syncthreads();
    for (uint32_t d = 1; d < 1024; d <<= 1) {
        const uint32_t v = tid >= d ? part[tid - d] : 0;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    at[2 * tid] = part[tid] - n0 - n1;
    at[2 * tid + 1] = part[tid] - n1;
    __syncthreads();
    for (uint32_t i = tid; i < rows; i += 1024) {
        const uint32_t p = atomicAdd(&at[kLengths - 1 - counts[i]], 1u);
        slot[i] = p;
        order[p] = i;
    }
    __syncthreads();
    __threadfence_block();
    // chunks of a slice: its first row's; slices <= 263, one per thread
    const uint32_t slices = (rows + 63) / 64;
    const uint32_t mine = tid < slices ? (counts[order[tid * 64]] + 7) / 8 : 0;
    part[tid] = mine;
    __syncthreads();
    for (uint32_t d = 1; d < 1024; d <<= 1) {
        const uint32_t v = tid >= d ? part[tid - d] : 0;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    if (tid < slices) sptr[tid] = chunk0 + part[tid] - mine;
    if (tid == slices) sptr[slices] = chunk0 + part[tid];
}

__global__ __launch_bounds__(64) void glue_fill_kernel(const Ballot* ballot, Seg g, Seg below, const uint32_t* order,
                                                       uint32_t* rowlab, uint4* cols) {
    __shared__ Ballot b;
    load_ballot(b, ballot);
    __syncthreads();
    const uint32_t slot = blockIdx.x * 64 + threadIdx.x, s = blockIdx.x;
    uint4* out = cols + (size_t)g.sptr[s] * 64 + threadIdx.x;
    const uint32_t chunks = g.sptr[s + 1] - g.sptr[s];
    uint64_t lo = 0, hi = 0;  // the chunk being filled
    uint32_t n = 0;
    auto put = [&](uint32_t c) {
        lo = (lo >> 16) | (hi << 48);
        hi = (hi >> 16) | ((uint64_t)c << 48);
        if ((++n & 7u) == 0) {
            *out = make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
            out += 64;
        }
    };
    uint32_t lab = ~0u;
    if (slot < g.rows) {
        lab = g.labels[order[slot]];
        if (g.m == 1) {
            put(0);
        } else {
            const int p = top_arc(lab), j = g.m - 2 - p;
            const uint32_t q = below.slot[rank_of(b, g.m - 2, without_pair(lab, p))], qs = q >> 6;
            const uint16_t* src = reinterpret_cast<const uint16_t*>(below.cols + (q & 63u));
            for (uint32_t i = 0; i < (below.sptr[qs + 1] - below.sptr[qs]) * 8; ++i) {
                const uint32_t c = src[((size_t)(below.sptr[qs] + (i >> 3)) * 64) * 8 + (i & 7u)];
                if (c >= below.rows) break;
                preimages(g.m, below.labels[c], j, [&](uint32_t w) { put(rank_of(b, g.m, w)); });
            }
        }
    }
    rowlab[slot] = lab;
    while (n < chunks * 8) put(g.rows);
}

uint32_t round_up(uint32_t x, uint32_t q) { return (x + q - 1) / q * q; }

}  // namespace

hipError_t build_tables(const Ballot& hb, const Ballot* dev_ballot, int m_lo, int m_hi, const Tables* below, Tables& out,
                        hipStream_t s) {
    // labels, row labels, slots, slice offsets and chunks of every m; row lengths and
    // orders only while the lists are made
    size_t words = 0, most = 0;
    uint32_t chunks = 0;
    for (int m = m_lo; m <= m_hi; m += 2) {
        const uint32_t rows = hb.n[m][1], slots = round_up(rows, 64);
        words += 3 * (size_t)slots + round_up(slots / 64 + 1, 64);
        chunks += chunk_bound(m, rows);
        most = std::max<size_t>(most, slots);
    }
    char *mem = nullptr, *tmp = nullptr;
    hipError_t e = hipMalloc(&mem, words * 4 + (size_t)chunks * 64 * sizeof(uint4));
    if (e == hipSuccess && (e = hipMalloc(&tmp, most * 8)) != hipSuccess) (void)hipFree(mem);
    if (e != hipSuccess) return e;
    uint4* cols = reinterpret_cast<uint4*>(mem + words * 4);  // words: a multiple of 64
    uint32_t* w = reinterpret_cast<uint32_t*>(mem);
    uint32_t *counts = reinterpret_cast<uint32_t*>(tmp), *order = counts + most;
    uint32_t chunk0 = 0;
    Tables t{};
    t.mem = mem;
    for (int m = m_lo; m <= m_hi; m += 2) {
        const uint32_t rows = hb.n[m][1], slots = round_up(rows, 64);
        Seg g{};
        g.m = m;
        g.rows = rows;
        g.slices = slots / 64;
        uint32_t *labels = w, *rowlab = w + slots, *slot = w + 2 * (size_t)slots, *sptr = w + 3 * (size_t)slots;
        w += 3 * (size_t)slots + round_up(slots / 64 + 1, 64);
        g.labels = labels;
        g.rowlab = rowlab;
        g.slot = slot;
        g.sptr = sptr;
        g.cols = cols;
        const Seg prev = m == 1 ? Seg{} : (m == m_lo ? below->seg[m - 2] : t.seg[m - 2]);
        hipLaunchKernelGGL(glue_count_kernel, dim3(g.slices), dim3(64), 0, s, dev_ballot, g, prev, labels, counts);
        hipLaunchKernelGGL(glue_order_kernel, dim3(1), dim3(1024), 0, s, rows, chunk0, counts, slot, order, sptr);
        hipLaunchKernelGGL(glue_fill_kernel, dim3(g.slices), dim3(64), 0, s, dev_ballot, g, prev, order, rowlab, cols);
        chunk0 += chunk_bound(m, rows);
        t.seg[m] = g;
    }
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(tmp);
    if (e != hipSuccess) {
        (void)hipFree(mem);
        return e;
    }
    out = t;
    return hipSuccess;
}

void free_tables(Tables& t) {
    if (t.mem) (void)hipFree(t.mem);
    t = Tables{};
}

namespace {

template <int KC, typename Idx, int NT, int TW>
hipError_t launch_lds(const GlueLaunch& a, uint32_t blocks, hipStream_t s) {
    const size_t bytes = (size_t)a.ystride * (NT / 64 / TW);
    auto* k = glue_kernel<KC, Idx, NT, TW>;
    if (bytes > (32u << 10)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)bytes);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k, dim3(blocks), dim3(NT), bytes, s, a);
    return hipGetLastError();
}

template <typename Idx, int NT, int TW>
hipError_t launch_lds_kc(GlueLaunch a, const Shape& sh, hipStream_t s) {
    uint32_t rows = 0;
    for (int i = 0; i < a.segs; ++i) rows = std::max(rows, a.seg[i].rows);
    a.tasks = sh.tasks;
    a.piece = sh.piece;
    a.ystride = round_up((rows + 1) * sh.kc * 4, 16);
    switch (sh.kc) {
        case 1: return launch_lds<1, Idx, NT, TW>(a, sh.blocks, s);
        case 2: return launch_lds<2, Idx, NT, TW>(a, sh.blocks, s);
        default: return launch_lds<4, Idx, NT, TW>(a, sh.blocks, s);
    }
}

template <int KC, typename Idx>
hipError_t launch_big_kc(GlueLaunch a, const Ballot& hb, hipStream_t s, int* launches) {
    const int m = a.seg[0].m;
    const unsigned passes = (unsigned)((a.K + KC - 1) / KC);
    auto grid = [](uint64_t n) { return (unsigned)((n + 255) / 256); };
    hipLaunchKernelGGL((glue_gather_kernel<Idx>), dim3(grid((uint64_t)a.batch * hb.n[m][1])), dim3(256), 0, s, a);
    a.from = 0;
    a.to = hb.n[m][1];
    const int levels = (m - kTabStrands) / 2;  // 1 or 2
    for (int r = 0; r < levels; ++r) {
        const uint32_t arrays = level_arrays(m, r), rows = hb.n[m - 2 * r - 2][1];
        a.removed = r;
        hipLaunchKernelGGL((glue_pull_kernel<KC>), dim3(grid((uint64_t)a.batch * arrays * rows), passes), dim3(256), 0, s, a,
                           arrays);
        a.from = a.to;
        a.to += arrays * rows;
    }
    hipLaunchKernelGGL((glue_big_kernel<KC, Idx>), dim3(grid((uint64_t)a.batch * hb.n[m][1]), passes), dim3(256), 0, s, a);
    if (launches) *launches += 2 + levels;
    return hipGetLastError();
}

template <typename Idx>
hipError_t launch_idx(GlueLaunch a, const Tables* tabs, const Ballot& hb, const uint32_t* binom, int cus, size_t scratch_bytes,
                      hipStream_t s, int* launches) {
    auto seg_of = [&](int m) {
        Seg g{};
        if (m <= kTabStrands) g = tabs[m > kBaseStrands ? 1 : 0].seg[m];
        g.m = m;
        g.rows = hb.n[m][1];
        g.count = binom[a.W * 32 + m];
        return g;
    };
    const int top = a.W % 2 ? a.W : a.W - 1;
    hipError_t e = hipSuccess;
    for (int m = top; m > kTabStrands && e == hipSuccess; m -= 2) {
        a.segs = 1;
        a.seg[0] = seg_of(m);
        a.seg[1] = seg_of(kTabStrands);
        a.each = task_entries(hb, m, kTabStrands);
        const Seg& g = a.seg[0];
        const uint32_t most =
            (uint32_t)std::min<uint64_t>(256, std::max<uint64_t>(1, scratch_bytes / ((uint64_t)a.each * a.K * 4)));
        for (uint32_t t = 0; t < g.count && e == hipSuccess; t += most) {
            a.task0 = t;
            a.batch = std::min(most, g.count - t);
            if (a.K == 1) e = launch_big_kc<1, Idx>(a, hb, s, launches);
            else if (a.K == 2) e = launch_big_kc<2, Idx>(a, hb, s, launches);
            else e = launch_big_kc<4, Idx>(a, hb, s, launches);
        }
    }
    for (const Class& c : kClasses) {
        if (e != hipSuccess) break;
        a.segs = 0;
        for (int m = std::min(c.hi, top); m >= c.lo; m -= 2) a.seg[a.segs++] = seg_of(m);
        const Shape sh = class_shape(c, a.W, a.K, cus, binom);
        if (!sh.tasks) continue;
        if (c.lo >= 17) e = launch_lds_kc<Idx, 1024, 16>(a, sh, s);
        else if (c.lo >= 13) e = launch_lds_kc<Idx, 256, 4>(a, sh, s);
        else e = launch_lds_kc<Idx, 256, 1>(a, sh, s);
        if (launches) ++*launches;
    }
    return e;
}

}  // namespace

size_t scratch_need(const Ballot& hb, int W, int K) {
    const int top = W % 2 ? W : W - 1;
    if (top <= kTabStrands) return 0;
    return std::max<size_t>((size_t)64 << 20, (size_t)task_entries(hb, top, kTabStrands) * K * 4);
}

hipError_t launch_glue(const GlueLaunch& a, const Tables* tabs, const Ballot& hb, const uint32_t* binom, bool wide, int cus,
                       size_t scratch_bytes, uint32_t* main_out, hipStream_t s, int* launches) {
    const hipError_t e = wide ? launch_idx<uint64_t>(a, tabs, hb, binom, cus, scratch_bytes, s, launches)
                              : launch_idx<uint32_t>(a, tabs, hb, binom, cus, scratch_bytes, s, launches);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(glue_finish_kernel, dim3(a.k), dim3(64), 0, s, a, main_out);
    if (launches) ++*launches;
    return hipGetLastError();
}

}  // namespace glue
}  // namespace ofp
