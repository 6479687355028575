// Host check of pair passes that go from one pair of arrays to another
// (oneesan-gpu_amd/csrc/ofp_pair_impl.h, pair_body's Whole): a solve's rows, first over
// only the classes whose P' and S' stay at the row's height bound, then whole, and two
// rows from arbitrary residues in every word, against the CPU oracle's whole rows: every
// main word after each pass, and every blocked word while there are any.  What a whole
// pass leaves unwritten keeps a value no residue has.  Window changes and classes in
// order and reversed, at one and three moduli.
// Built and run by tests/test_pair_whole_host.py; "ALL OK" at the end.
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

template <int KC, int D>
static void run_d(const pair::PairLaunch& a, const cell::Tab<uint32_t>& T, const pair::Io<KC, uint32_t>& io, bool rev) {
    constexpr int C = cell::LdsCols<uint32_t>::value;
    static cell::Pair<uint32_t> ct[kDpRows][C];
    static uint64_t dc[kDpRows][kDpCols];
    table(a.cap, dc);
    pair::pack_class_table<uint32_t, C>(dc, a.p, D, ct, a.cap);
    const uint64_t n = pair::class_count(dc, a.W, a.p, D, a.cap);
    for (uint64_t t = 0; t < n; ++t) {
        const uint64_t c = rev ? n - 1 - t : t;
        const pair::Class<uint32_t> k = a.cap > 0 ? pair::decode_class_capped<uint32_t>(T, ct, a.W, a.p, D, c)
                                                  : pair::decode_class<uint32_t>(T, ct, a.W, a.p, c);
        pair::pair_body<KC, uint32_t, D, 0, true>(a, T, k, io);
    }
}

template <int KC>
static void pass(const pair::PairLaunch& a, const cell::Tab<uint32_t>& T, const pair::Io<KC, uint32_t>& io, bool rev) {
    for (int i = 0; i < 7; ++i) switch (rev ? 3 - i : i - 3) {
        case -3: run_d<KC, -3>(a, T, io, rev); break;
        case -2: run_d<KC, -2>(a, T, io, rev); break;
        case -1: run_d<KC, -1>(a, T, io, rev); break;
        case 0: run_d<KC, 0>(a, T, io, rev); break;
        case 1: run_d<KC, 1>(a, T, io, rev); break;
        case 2: run_d<KC, 2>(a, T, io, rev); break;
        default: run_d<KC, 3>(a, T, io, rev); break;
    }
}

// rows from `first`: capped by their bound from the start state, whole where the bound
// is no cap (row -1: arbitrary residues, two whole rows)
template <int KC>
static int check(int n, int first, bool rev) {
    static const uint32_t mods[3] = {4294967291u, 65537u, 4294967279u};
    const int W = n + 1;
    constexpr int C = cell::LdsCols<uint32_t>::value;
    static cell::Quad<uint32_t> qfull[kDpRows][kDpCols], q[kDpRows][C];
    cell::pack_quads<uint32_t>(D0, qfull);
    for (int r = 0; r < kDpRows; ++r)
        for (int h = 0; h < C; ++h) q[r][h] = qfull[r][h];
    cell::Tab<uint32_t> T{q};
    const size_t nm = D0[W][1], nb = D0[W - 1][1];
    std::vector<uint32_t> m(nm * KC, 0), b(nb * KC, 0), m2, b2, em[KC], eb[KC];
    uint64_t x = 88172645463325252ull;
    for (int j = 0; j < KC; ++j) {
        if (first < 0)
            for (size_t i = 0; i < nm; ++i) m[i * KC + j] = (uint32_t)((x = x * 6364136223846793005ull + 1) >> 33) % mods[j];
        else
            m[D0[W - 1][1] * KC + j] = 1;
        em[j].resize(nm);
        eb[j].assign(nb, 0);
        for (size_t i = 0; i < nm; ++i) em[j][i] = m[i * KC + j];
    }
    m2.assign(m.size(), first < 0 ? 0xffffffffu : 0);
    b2.assign(b.size(), first < 0 ? 0xffffffffu : 0);
    const int rows = first < 0 ? 2 : W - 1;
    for (int r = 0; r < rows; ++r)
        for (int p = W - 1; p >= 1;) {
            const int bound = std::max(p >= W - r ? r : r + 1, p - 1 >= W - r ? r : r + 1);
            const int cap = first < 0 || r == W - 2 ? 0 : (r == 0 ? 1 : bound);
            const int lo = p >= 2 ? p - 1 : p;
            for (int j = 0; j < KC; ++j) or_apply_cells(n, mods[j], em[j].data(), eb[j].data(), p, lo, p != W - 1, 1);
            if (p == 1) {  // a last single cell: taken from the oracle
                for (int j = 0; j < KC; ++j)
                    for (size_t i = 0; i < nm; ++i) m[i * KC + j] = em[j][i];
            } else {
                pair::PairLaunch a{};
                a.W = W;
                a.p = p;
                a.cap = cap;
                a.read_blk = p != W - 1;
                a.K = a.kc = KC;
                for (int j = 0; j < KC; ++j) a.mod[j] = mods[j];
                pass<KC>(a, T, pair::Io<KC, uint32_t>{m.data(), b.data(), m2.data(), b2.data(), KC, 0}, rev);
                m.swap(m2);
                b.swap(b2);
                for (int j = 0; j < KC; ++j) {
                    for (size_t i = 0; i < nm; ++i)
                        if (m[i * KC + j] != em[j][i]) return printf("MISMATCH main n=%d row=%d p=%d cap=%d\n", n, r, p, cap);
                    for (size_t i = 0; p - 1 >= 2 && i < nb; ++i)
                        if (b[i * KC + j] != eb[j][i]) return printf("MISMATCH blocked n=%d row=%d p=%d cap=%d\n", n, r, p, cap);
                }
            }
            p -= 2;
        }
    printf("ok n=%d k=%d %s order=%s\n", n, KC, first < 0 ? "arbitrary" : "from the start", rev ? "reverse" : "forward");
    return 0;
}

int main(int argc, char** argv) {
    const int nmax = argc > 1 ? atoi(argv[1]) : 9;
    table(0, D0);
    for (int n = 2; n <= nmax; ++n)
        for (int rev = 0; rev < 2; ++rev)
            for (int first = -1; first < 1; ++first)
                if (check<1>(n, first, rev) || check<3>(n, first, rev)) return 1;
    printf("ALL OK\n");
    return 0;
}
