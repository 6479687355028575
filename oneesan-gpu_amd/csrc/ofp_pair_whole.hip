// ofp_pair_whole.hip -- the pair pass of a small state in one launch, for gfx950.
//
// A small state's solve is bound by its launches: about 4 us each before the first
// word is touched, and up to 3 us of table loads and dependent index math (n=12: 72
// cells in 0.49 ms of a 0.64 ms solve).  In place a pair pass needs up to five
// launches in two steps; from one pair of arrays to another (pair_body's Whole) every
// class reads only the old state, so the classes of all seven window changes go in one
// launch, two cells at a time -- d = +-3, the words both cells keep, among them.  The
// workgroups of one launch take the window changes one after another (a.block).
// Measured against one launch per cell (n=12, one modulus: 81 launches of 6.4 us, 42 of
// 11) and against passes in place: see kWholeWords in ofp_api.hip.
#include <algorithm>

#include "ofp_pair_impl.h"

namespace ofp {

namespace {

using namespace cell;

template <int KC, int D, bool Capped>
__device__ __forceinline__ void whole_class(const pair::PairLaunch& a, const Tab<uint32_t>& T,
                                            const Pair<uint32_t> (*ct)[LdsCols<uint32_t>::value],
                                            const pair::Io<KC, uint32_t>& io, uint32_t c) {
    const pair::Class<uint32_t> k = Capped ? pair::decode_class_capped<uint32_t>(T, ct, a.W, a.p, D, c)
                                           : pair::decode_class<uint32_t>(T, ct, a.W, a.p, c);
    pair::pair_body<KC, uint32_t, D, 0, true>(a, T, k, io);
}

template <int KC, bool Capped>
__global__ __launch_bounds__(256) void pair_whole_kernel(pair::PairLaunch a) {
    constexpr int C = LdsCols<uint32_t>::value;
    __shared__ Quad<uint32_t> tab[kLdsRows][C];
    __shared__ Pair<uint32_t> ctab[kLdsRows][C];
    int di = 0;
    while (blockIdx.x >= a.block[di + 1]) ++di;
    load_table<C, kDpCols>(&tab[0][0], (const Quad<uint32_t>*)a.dp, a.W);
    load_table<C, C>(&ctab[0][0], (const Pair<uint32_t>*)((const char*)a.ct + (size_t)di * a.ct_bytes), a.W);
    __syncthreads();
    const Tab<uint32_t> T{tab};
    const pair::Io<KC, uint32_t> io{a.main_in, a.blk_in, a.main_out, a.blk_out, a.K, a.off};
    const uint32_t c = (blockIdx.x - a.block[di]) * blockDim.x + threadIdx.x;
    if (c >= a.count[di]) return;
    switch (di) {
        case 0: whole_class<KC, -3, Capped>(a, T, ctab, io, c); break;
        case 1: whole_class<KC, -2, Capped>(a, T, ctab, io, c); break;
        case 2: whole_class<KC, -1, Capped>(a, T, ctab, io, c); break;
        case 3: whole_class<KC, 0, Capped>(a, T, ctab, io, c); break;
        case 4: whole_class<KC, 1, Capped>(a, T, ctab, io, c); break;
        case 5: whole_class<KC, 2, Capped>(a, T, ctab, io, c); break;
        default: whole_class<KC, 3, Capped>(a, T, ctab, io, c); break;
    }
}

// The words of a fresh state, both pairs of arrays (16-byte pieces), in one launch:
// zero, but 1 mod each modulus at the start word; and the accs sums zero.
__global__ __launch_bounds__(256) void init_whole_kernel(WholeInit a) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x, t0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (int i = 0; i < 4; ++i)
        for (uint64_t t = t0; t < a.words[i] / 4; t += stride) {
            uint32_t v[4] = {0, 0, 0, 0};
            if (i == 0 && 4 * t + 3 >= a.start && 4 * t < a.start + (uint32_t)a.k)
                for (int q = 0; q < 4; ++q) {
                    const uint64_t j = 4 * t + q - a.start;
                    if (j < (uint64_t)a.k) v[q] = 1u % (a.mods ? a.mods[j] : a.mod[j]);
                }
            reinterpret_cast<uint4*>(a.array[i])[t] = make_uint4(v[0], v[1], v[2], v[3]);
        }
    if (a.acc)
        for (uint64_t t = t0; t < (uint64_t)a.accs; t += stride) a.acc[t] = 0;
}

}  // namespace

hipError_t launch_pair_whole(const pair::PairLaunch& a, int threads, hipStream_t s) {
    if (a.p < 2 || a.p > a.W - 1 || a.kc < 1 || a.kc > kWholeKC || a.off + a.kc > a.K || a.cap < 0 || a.cap > kPairCaps ||
        a.main_in == a.main_out || threads <= 0 || threads > 256 || (threads & 63))
        return hipErrorInvalidValue;
    if (!a.block[7]) return hipSuccess;
    switch (a.kc) {
#define OFP_KC(n)                                                                                              \
    case n:                                                                                                    \
        if (a.cap > 0) hipLaunchKernelGGL((pair_whole_kernel<n, true>), dim3(a.block[7]), dim3(threads), 0, s, a); \
        else hipLaunchKernelGGL((pair_whole_kernel<n, false>), dim3(a.block[7]), dim3(threads), 0, s, a);      \
        break;
        OFP_KC(1) OFP_KC(2) OFP_KC(3) OFP_KC(4) OFP_KC(5) OFP_KC(6) OFP_KC(7) OFP_KC(8)
#undef OFP_KC
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_init_whole(const WholeInit& a, hipStream_t s) {
    const uint64_t most = (a.words[0] / 4 + 255) / 256;
    hipLaunchKernelGGL(init_whole_kernel, dim3((unsigned)std::min<uint64_t>(std::max<uint64_t>(most, 1), 2048)), dim3(256), 0,
                       s, a);
    return hipGetLastError();
}

}  // namespace ofp
