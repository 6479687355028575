// ofp_pair.hip -- the pair pass: cells p and p-1 of a row applied in place,
// one launch per window height change d, or one for d = -1, 0 and 1 (body and design
// in ofp_pair_impl.h; which one: reader_pieces in ofp_api.hip).
//
// Each thread takes one class (P', d, S'), decoded from its class number with
// the class completion table of (p, d) and the height table, both in LDS; the
// classes are dealt to the XCDs in pieces exactly as the cell kernels deal
// their blocked words (cell::Sched).  Every word belongs to one class and only
// that class's thread writes it; the words a class reads from other classes
// still hold their values from before the pass when it reads them (launch
// order d = -1, 0, 1, then -2, 2), so the launches need no atomics and no
// second copy of the state.
#include <algorithm>

#include "ofp_pair_impl.h"

namespace ofp {

namespace {

using namespace cell;

// Whether the closure sums are gathered before the class's words are loaded (pair_body's
// GF).  Loading the words first, so that the scans run while they are in flight, keeps up to
// 14 records per thread live (d = 0: ten words, two sums and, in the scans, four sources):
// from 14 moduli, or 13 with 64-bit ranks, that is more than the 256 VGPRs two workgroups
// per CU leave each thread, and up to 65 of them spill.  Gathered first none does.  ms of a
// full row, words first and sums first: n=20 at 16 moduli 116.5, 113.0; 15 114.1, 112.5; 14
// 105.6, 105.4; n=21 at 16 310.1, 303.9; 14 277.9, 278.2; with 64-bit ranks n=20 at 16
// 119.2, 113.4; 14 108.8, 106.1; 13 103.3, 102.1; 12 (two spilled in pair_readers_kernel)
// 89.2, 89.7.
template <int KC, typename Idx>
constexpr int kSumsFirst = KC >= (sizeof(Idx) == 8 ? 13 : 14) ? 1 : 0;

// MB: workgroups of 256 per CU the register allocation must allow (2: at most
// 256 VGPRs, no spills; 3: at most 168, with spills).
// Capped: the classes of a height-capped pass (a.cap).
template <int KC, typename Idx, int D, int GF, int MB, bool Capped>
__global__ __launch_bounds__(256, MB) void pair_kernel(pair::PairLaunch a) {
    constexpr int C = LdsCols<Idx>::value;
    __shared__ Quad<Idx> tab[kLdsRows][C];
    __shared__ Pair<Idx> ctab[kLdsRows][C];
    const Quad<Idx>* g = (const Quad<Idx>*)a.dp;
    load_table<C, kDpCols>(&tab[0][0], g, a.W);
    load_table<C, C>(&ctab[0][0], (const Pair<Idx>*)a.ct, a.W);
    __syncthreads();
    Tab<Idx> T{tab};
    const pair::Io<KC, Idx> io{a.main_in, a.blk_in, a.main_out, a.blk_out, a.K, a.off};
    const Sched sc(a.classes, blockDim.x, gridDim.x, blockIdx.x, a.xcd_shift);
    for (uint64_t t = sc.slot; t < sc.count; t += sc.nx) {
        const uint64_t c = sc.chunk(t) * blockDim.x + threadIdx.x;
        if (c < a.classes) {
            const pair::Class<Idx> k = Capped ? pair::decode_class_capped<Idx>(T, ctab, a.W, a.p, D, c)
                                              : pair::decode_class<Idx>(T, ctab, a.W, a.p, c);
            pair::pair_body<KC, Idx, D, GF>(a, T, k, io);
        }
    }
}

// The classes of d = -1, 0 and 1 in one launch, a piece of the prefixes P' at a time: a
// workgroup takes a.group chunks of d = 0's classes and, with them, the d = -1 and 1
// classes of the same P' (from the first P' of its chunks to that of the next ones).
template <int KC, typename Idx, bool Capped>
__global__ __launch_bounds__(256, 2) void pair_readers_kernel(pair::PairLaunch a) {
    constexpr int C = LdsCols<Idx>::value;
    __shared__ Quad<Idx> tab[kLdsRows][C];
    __shared__ Pair<Idx> ctab[kLdsRows][C];
    __shared__ uint64_t at[2], word[2];  // the piece's ends: classes of one d; P' (all ones: past the last)
    load_table<C, kDpCols>(&tab[0][0], (const Quad<Idx>*)a.dp, a.W);
    const Tab<Idx> T{tab};
    const pair::Io<KC, Idx> io{a.main_in, a.blk_in, a.main_out, a.blk_out, a.K, a.off};
    const uint64_t piece = (uint64_t)blockDim.x * (uint32_t)a.group;
    const Sched sc(a.classes, (uint32_t)piece, gridDim.x, blockIdx.x, a.xcd_shift);
    auto table = [&](int d) {
        __syncthreads();  // the last one's readers
        load_table<C, C>(&ctab[0][0], (const Pair<Idx>*)((const char*)a.ct + (size_t)(d + 3) * a.ct_bytes), a.W);
        __syncthreads();
    };
    auto decode = [&](int d, uint64_t c) {
        return Capped ? pair::decode_class_capped<Idx>(T, ctab, a.W, a.p, d, c)
                      : pair::decode_class<Idx>(T, ctab, a.W, a.p, c);
    };
    for (uint64_t t = sc.slot; t < sc.count; t += sc.nx) {
        const uint64_t lo = sc.chunk(t) * piece, hi = lo + piece < a.classes ? lo + piece : a.classes;
        if (lo >= a.classes) continue;  // the whole workgroup
        table(0);
        if (threadIdx.x < 2) {
            const uint64_t c = threadIdx.x ? hi : lo;
            word[threadIdx.x] = c < a.classes ? pair::decode_class<Idx>(T, ctab, a.W, a.p, c).word : ~0ull;
        }
        for (uint64_t c = lo + threadIdx.x; c < hi; c += blockDim.x)
            pair::pair_body<KC, Idx, 0, kSumsFirst<KC, Idx>>(a, T, decode(0, c), io);
        for (int side = 0; side < 2; ++side) {
            table(2 * side - 1);
            if (threadIdx.x < 2)
                at[threadIdx.x] = threadIdx.x == 0 && lo == 0 ? 0
                                  : word[threadIdx.x] == ~0ull
                                      ? a.sides[side]
                                      : (uint64_t)pair::classes_before<Idx>(ctab, a.W, a.p, word[threadIdx.x]);
            __syncthreads();
            const uint64_t b = at[0], e = at[1];
            for (uint64_t c = b + threadIdx.x; c < e; c += blockDim.x) {
                if (side == 0) pair::pair_body<KC, Idx, -1, kSumsFirst<KC, Idx>>(a, T, decode(-1, c), io);
                else pair::pair_body<KC, Idx, 1, kSumsFirst<KC, Idx>>(a, T, decode(1, c), io);
            }
        }
    }
}

// The classes with d = -3, 3 change nothing and get no launch.
template <int KC, typename Idx, int GF, int MB, bool Capped = false>
hipError_t launch_d(const pair::PairLaunch& a, int threads, int blocks, hipStream_t s) {
    switch (a.d) {
#define OFP_D(d) \
    case d: hipLaunchKernelGGL((pair_kernel<KC, Idx, d, GF, MB, Capped>), dim3(blocks), dim3(threads), 0, s, a); break;
        OFP_D(-2) OFP_D(-1) OFP_D(0) OFP_D(1) OFP_D(2)
#undef OFP_D
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Pair-kernel variant (PairLaunch::variant): bit 1 = the three-workgroups-per-CU register
// budget; only the whole-state 14- and 16-moduli kernels carry it (the others run variant 0).
template <int KC, typename Idx>
hipError_t launch_gf(const pair::PairLaunch& a, int threads, int blocks, hipStream_t s) {
    constexpr int GF = kSumsFirst<KC, Idx>;
    if (a.cap > 0) return launch_d<KC, Idx, GF, 2, true>(a, threads, blocks, s);
    if constexpr (KC == 14 || KC == 16)
        if (a.variant & 2) return launch_d<KC, Idx, GF, 3>(a, threads, blocks, s);
    return launch_d<KC, Idx, GF, 2>(a, threads, blocks, s);
}

// Class tables of every (cap, p, d), cap 0 = none, one wave each (lane = height):
// the height table's rows from the bottom up to p-2, then the class counts above p
// (pair::build_class_table with the cap), packed as pair::pack_class_table does.
template <typename Idx>
__global__ __launch_bounds__(64) void class_tables_kernel(Pair<Idx>* out) {
    constexpr int C = LdsCols<Idx>::value;
    const int d = (int)(blockIdx.x % 7) - 3, p = (int)(blockIdx.x / 7) % kMaxW, cap = (int)(blockIdx.x / 7) / kMaxW;
    const int h = (int)threadIdx.x, top = cap > 0 ? cap : kDpCols - 1;
    const bool in = h <= top;
    Pair<Idx>* t = out + (size_t)blockIdx.x * kLdsRows * C;
    const auto at = [&](uint64_t v, int q) -> uint64_t {  // the value at height q, 0 outside 0..top
        const uint64_t x = __shfl(v, q & 63);
        return q >= 0 && q <= top ? x : 0;
    };
    const auto put = [&](int row, uint64_t v) {
        const uint64_t below = at(v, h - 1);
        if (h < C) t[row * C + h] = Pair<Idx>{(Idx)v, (Idx)(v + below)};
    };
    uint64_t v = h == 0 ? 1 : 0;  // the height table's row w
    for (int w = 0; w < p - 2; ++w) {
        put(w, cap > 0 ? v : 0);
        const uint64_t dn = at(v, h - 1), up = at(v, h + 1);
        v = in ? v + dn + up : 0;
    }
    v = p >= 2 ? at(v, h + d) : 0;  // row p-2 at height h + d
    v = in ? v : 0;
    for (int m = p < 2 ? 0 : p - 2; m <= p && m < kLdsRows; ++m) put(m, 0);
    for (int m = p + 1; m < kLdsRows; ++m) {
        put(m, v);
        const uint64_t dn = at(v, h - 1), up = at(v, h + 1);
        v = in ? v + dn + up : 0;
    }
}

}  // namespace

size_t class_table_bytes(bool wide) {
    return (wide ? sizeof(Pair<uint64_t>) * LdsCols<uint64_t>::value : sizeof(Pair<uint32_t>) * LdsCols<uint32_t>::value) *
           kLdsRows;
}

hipError_t launch_class_tables(bool wide, void* out, hipStream_t s) {
    const dim3 grid((kPairCaps + 1) * kMaxW * 7);
    if (wide) hipLaunchKernelGGL((class_tables_kernel<uint64_t>), grid, dim3(64), 0, s, (Pair<uint64_t>*)out);
    else hipLaunchKernelGGL((class_tables_kernel<uint32_t>), grid, dim3(64), 0, s, (Pair<uint32_t>*)out);
    return hipGetLastError();
}

// The prefixes P' that end at height h, times the suffixes S' entered at h + d, summed
// over h: pair::class_count without a table of its own per launch (seven a pass).
uint64_t pair_class_count(int W, int p, int d, int cap) {
    struct Words {
        uint64_t down[kPairCaps + 1][kDpRows][kDpCols];  // words of w positions from h to 0
        uint64_t up[kPairCaps + 1][kDpRows][kDpCols];    // words of w positions from 1 to h
        Words() {
            for (int c = 0; c <= kPairCaps; ++c) {
                if (c > 0) build_capped_table(c, down[c]);
                else build_height_table(down[c]);
                const int top = c > 0 ? c : kDpCols - 1;
                for (int w = 0; w < kDpRows; ++w)
                    for (int h = 0; h < kDpCols; ++h)
                        up[c][w][h] = h > top ? 0
                                      : w == 0 ? (h == 1)
                                               : up[c][w - 1][h] + (h > 0 ? up[c][w - 1][h - 1] : 0) +
                                                     (h < top ? up[c][w - 1][h + 1] : 0);
            }
        }
    };
    static const Words words;  // the same for every context
    uint64_t n = 0;
    if (p < 2 || p > W - 1) return 0;
    for (int h = std::max(0, -d); h + std::max(0, d) < kDpCols; ++h)
        n += words.up[cap][W - 1 - p][h] * words.down[cap][p - 2][h + d];
    return n;
}

hipError_t launch_pair_readers(const pair::PairLaunch& a, bool wide, int threads, int blocks, hipStream_t s) {
    if (a.p < 2 || a.p > a.W - 1 || a.kc < 1 || a.off + a.kc > a.K || a.cap < 0 || a.cap > kPairCaps || !a.classes ||
        a.group < 1 || threads <= 0 || threads > 256 || (threads & 63) || blocks <= 0 || (blocks & 7))
        return hipErrorInvalidValue;
#define OFP_R(n, I)                                                                                                \
    if (a.cap > 0) hipLaunchKernelGGL((pair_readers_kernel<n, I, true>), dim3(blocks), dim3(threads), 0, s, a);     \
    else hipLaunchKernelGGL((pair_readers_kernel<n, I, false>), dim3(blocks), dim3(threads), 0, s, a);
    switch (a.kc) {
#define OFP_KC(n)                                      \
    case n:                                            \
        if (wide) { OFP_R(n, uint64_t) }               \
        else { OFP_R(n, uint32_t) }                    \
        break;
        OFP_KC(1) OFP_KC(2) OFP_KC(3) OFP_KC(4) OFP_KC(5) OFP_KC(6) OFP_KC(7) OFP_KC(8)
        OFP_KC(9) OFP_KC(10) OFP_KC(11) OFP_KC(12) OFP_KC(13) OFP_KC(14) OFP_KC(15) OFP_KC(16)
#undef OFP_KC
#undef OFP_R
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_pair(const pair::PairLaunch& a, bool wide, int threads, int blocks, hipStream_t s) {
    if (a.p < 2 || a.p > a.W - 1 || a.d < -3 || a.d > 3 || a.kc < 1 || a.off + a.kc > a.K || a.cap < 0 || a.cap > kPairCaps)
        return hipErrorInvalidValue;
    switch (a.kc) {
#define OFP_KC(n) \
    case n: return wide ? launch_gf<n, uint64_t>(a, threads, blocks, s) : launch_gf<n, uint32_t>(a, threads, blocks, s);
        OFP_KC(1) OFP_KC(2) OFP_KC(3) OFP_KC(4) OFP_KC(5) OFP_KC(6) OFP_KC(7) OFP_KC(8)
        OFP_KC(9) OFP_KC(10) OFP_KC(11) OFP_KC(12) OFP_KC(13) OFP_KC(14) OFP_KC(15) OFP_KC(16)
#undef OFP_KC
        default: return hipErrorInvalidValue;
    }
}

}  // namespace ofp
