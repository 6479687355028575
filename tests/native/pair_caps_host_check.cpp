// Host check of height-capped pair passes (oneesan-gpu_amd/csrc/ofp_pair_impl.h):
// the first rows of a solve swept IN PLACE on the CPU by pair passes over only the
// classes whose P' and S' stay at the row's height bound, against the CPU oracle's
// whole rows from the same start: every main word after each pass, and every blocked
// word while there are any.  Classes in rank order and reversed, 32- and 64-bit ranks.
// Built and run by tests/test_pair_caps_host.py; "ALL OK" at the end.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../oneesan-gpu_amd/csrc/ofp_pair_impl.h"

extern "C" int or_apply_cells(int n, uint32_t mod, uint32_t* main, uint32_t* blk, int p_hi, int p_lo, int blk_valid,
                              int use_pull);

using namespace ofp;

static uint64_t D0[kDpRows][kDpCols];

static void table(int cap, uint64_t (*d)[kDpCols]) {
    const int top = cap > 0 ? cap : kDpCols - 1;
    for (int w = 0; w < kDpRows; ++w)
        for (int h = 0; h < kDpCols; ++h)
            d[w][h] = h > top ? 0
                              : (w == 0 ? (h == 0)
                                        : d[w - 1][h] + (h > 0 ? d[w - 1][h - 1] : 0) + (h + 1 <= top ? d[w - 1][h + 1] : 0));
}

template <typename Idx, int D>
static void run_d(const pair::PairLaunch& a, const cell::Tab<Idx>& T, const pair::Io<1, Idx>& io, bool rev) {
    constexpr int C = cell::LdsCols<Idx>::value;
    static cell::Pair<Idx> ct[kDpRows][C];
    static uint64_t dc[kDpRows][kDpCols];
    table(a.cap, dc);
    pair::pack_class_table<Idx, C>(dc, a.p, D, ct, a.cap);
    const uint64_t n = pair::class_count(dc, a.W, a.p, D, a.cap);
    for (uint64_t t = 0; t < n; ++t) {
        const pair::Class<Idx> k = pair::decode_class_capped<Idx>(T, ct, a.W, a.p, D, rev ? n - 1 - t : t);
        pair::pair_body<1, Idx, D, 0>(a, T, k, io);
    }
}

template <typename Idx>
static int check(int n, uint32_t mod, bool rev) {
    const int W = n + 1;
    constexpr int C = cell::LdsCols<Idx>::value;
    static cell::Quad<Idx> qfull[kDpRows][kDpCols], q[kDpRows][C];
    cell::pack_quads<Idx>(D0, qfull);
    for (int r = 0; r < kDpRows; ++r)
        for (int h = 0; h < C; ++h) q[r][h] = qfull[r][h];
    cell::Tab<Idx> T{q};
    std::vector<uint32_t> m(D0[W][1], 0), b(D0[W - 1][1], 0);
    m[D0[W - 1][1]] = 1 % mod;
    std::vector<uint32_t> em = m, eb = b;
    for (int r = 0; r < W - 2; ++r)
        for (int p = W - 1; p >= 1;) {
            const int bound = std::max(p >= W - r ? r : r + 1, p - 1 >= W - r ? r : r + 1), cap = r == 0 ? 1 : bound;
            if (p == 1 || cap > 13) {  // a last single cell: taken from the oracle
                or_apply_cells(n, mod, m.data(), b.data(), p, p, p != W - 1, 1);
                or_apply_cells(n, mod, em.data(), eb.data(), p, p, p != W - 1, 1);
                --p;
            } else {
                pair::PairLaunch a{};
                a.W = W;
                a.p = p;
                a.cap = cap;
                a.read_blk = p != W - 1;
                a.K = a.kc = 1;
                a.mod[0] = mod;
                pair::Io<1, Idx> io{m.data(), b.data(), m.data(), b.data(), 1, 0};
                run_d<Idx, -1>(a, T, io, rev);
                run_d<Idx, 0>(a, T, io, rev);
                run_d<Idx, 1>(a, T, io, rev);
                run_d<Idx, -2>(a, T, io, rev);
                run_d<Idx, 2>(a, T, io, rev);
                or_apply_cells(n, mod, em.data(), eb.data(), p, p - 1, p != W - 1, 1);
                if (m != em || (p - 1 >= 2 && b != eb)) {
                    printf("MISMATCH n=%d row=%d p=%d cap=%d %s\n", n, r, p, cap, m != em ? "main" : "blocked");
                    return 1;
                }
                p -= 2;
            }
        }
    printf("ok n=%d idx=%d order=%s\n", n, (int)sizeof(Idx) * 8, rev ? "reverse" : "forward");
    return 0;
}

int main(int argc, char** argv) {
    const int nmax = argc > 1 ? atoi(argv[1]) : 10;
    table(0, D0);
    for (int n = 3; n <= nmax; ++n)
        for (int rev = 0; rev < 2; ++rev)
            if (check<uint32_t>(n, 4294967291u, rev) || check<uint64_t>(n, 65537u, rev)) return 1;
    printf("ALL OK\n");
    return 0;
}
