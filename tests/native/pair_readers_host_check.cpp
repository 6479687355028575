// Host check of the pieces that a launch over a pair pass's readers is cut into
// (pair_readers_kernel in oneesan-gpu_amd/csrc/ofp_pair.hip): the classes of d = -1 and 1
// from classes_before of a piece's first P' to that of the next piece's are, piece by
// piece, all classes of that d once and in order, and exactly those whose P' lies
// between the two.  Both rank widths, whole and capped, pieces of several sizes.
// Built and run by tests/test_pair_readers.py; "ALL OK" at the end.
#include <cstdio>
#include <cstdlib>

#include "../../oneesan-gpu_amd/csrc/ofp_pair_impl.h"

using namespace ofp;

template <typename Idx>
static int check(int n, int p, int cap, uint64_t piece) {
    constexpr int C = cell::LdsCols<Idx>::value;
    static cell::Quad<Idx> q[kDpRows][C];
    static cell::Pair<Idx> ct[3][kDpRows][C];
    uint64_t d0[kDpRows][kDpCols], full[kDpRows][kDpCols], count[3];
    for (int pass = 0; pass < 2; ++pass) {
        uint64_t(*t)[kDpCols] = pass ? full : d0;
        const int top = !pass && cap ? cap : kDpCols - 1;
        for (int w = 0; w < kDpRows; ++w)
            for (int h = 0; h < kDpCols; ++h)
                t[w][h] = h > top ? 0
                                  : (w == 0 ? (h == 0)
                                            : t[w - 1][h] + (h > 0 ? t[w - 1][h - 1] : 0) + (h + 1 <= top ? t[w - 1][h + 1] : 0));
    }
    static cell::Quad<Idx> qf[kDpRows][kDpCols];
    cell::pack_quads<Idx>(full, qf);
    for (int r = 0; r < kDpRows; ++r)
        for (int h = 0; h < C; ++h) q[r][h] = qf[r][h];
    const cell::Tab<Idx> T{q};
    const int W = n + 1;
    for (int i = 0; i < 3; ++i) {
        pair::pack_class_table<Idx, C>(d0, p, i - 1, ct[i], cap);
        count[i] = pair::class_count(d0, W, p, i - 1, cap);
    }
    for (int i = 0; i < 3; i += 2) {
        uint64_t next = 0;
        for (uint64_t lo = 0; lo < count[1]; lo += piece) {
            const uint64_t hi = lo + piece < count[1] ? lo + piece : count[1];
            const uint64_t w0 = pair::decode_class<Idx>(T, ct[1], W, p, lo).word;
            const uint64_t w1 = hi < count[1] ? pair::decode_class<Idx>(T, ct[1], W, p, hi).word : ~0ull;
            const uint64_t b = lo == 0 ? 0 : (uint64_t)pair::classes_before<Idx>(ct[i], W, p, w0);
            const uint64_t e = w1 == ~0ull ? count[i] : (uint64_t)pair::classes_before<Idx>(ct[i], W, p, w1);
            if (b != next || e < b) return printf("GAP n=%d p=%d cap=%d d=%d piece=%llu\n", n, p, cap, i - 1, (unsigned long long)piece);
            next = e;
            for (uint64_t c = b; c < e; ++c) {
                const uint64_t w = pair::decode_class<Idx>(T, ct[i], W, p, c).word;
                if ((lo > 0 && w < w0) || w >= w1)
                    return printf("OUTSIDE n=%d p=%d cap=%d d=%d class=%llu\n", n, p, cap, i - 1, (unsigned long long)c);
            }
        }
        if (count[1] && next != count[i]) return printf("MISSING n=%d p=%d cap=%d d=%d\n", n, p, cap, i - 1);
    }
    return 0;
}

int main() {
    for (int n = 3; n <= 11; ++n)
        for (int p = 2; p < n; ++p)
            for (int cap = 0; cap <= 4; ++cap)
                for (uint64_t piece : {1ull, 7ull, 64ull, 256ull, 512ull})
                    if (check<uint32_t>(n, p, cap, piece) || check<uint64_t>(n, p, cap, piece)) return 1;
    printf("ALL OK\n");
    return 0;
}
