// Host check of the half-row solve (oneesan-gpu_amd/csrc/ofp_glue_impl.h): the
// CPU oracle sweeps half of a row sweep's cells, the header's functions built for
// the host sum over the meeting word pairs (every table index range-checked), and
// the result is compared with the oracle's whole solve; and the lists of open
// meanders are compared with a walk along the arcs of every pair of words.
// Built and run by tests/test_glue_host.py; "ALL OK" at the end.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../oneesan-gpu_amd/csrc/ofp_glue_impl.h"

extern "C" int or_apply_cells(int n, uint32_t mod, uint32_t* main, uint32_t* blk, int p_hi, int p_lo, int blk_valid,
                              int use_pull);
extern "C" uint32_t or_solve(int n, uint32_t mod, int use_pull, int* err);

using namespace ofp;
using namespace ofp::glue;

static Ballot B;
static uint64_t H[kDpRows][kDpCols];
static uint32_t bin[kMaxW * 32];

// Row lambda of G_m by removing arcs, and through the arrays of the removed arcs'
// places as the sums over many strands go.
static std::vector<uint32_t> row_of(int m, uint32_t lambda) {
    if (m == 1) return {0};
    const uint32_t lab = labels_of(B, m, lambda);
    const int p = top_arc(lab);
    std::vector<uint32_t> r;
    for (uint32_t v : row_of(m - 2, rank_of(B, m - 2, without_pair(lab, p))))
        preimages(m, labels_of(B, m - 2, v), m - 2 - p, [&](uint32_t w) { r.push_back(rank_of(B, m, w)); });
    return r;
}

// arcs of a word from its labels: partner of strand i (m-1 = top), m = the path's end
static void arcs(int m, uint32_t lab, std::vector<int>& par) {
    par.assign(m + 1, -1);
    std::vector<int> st{m};
    for (int i = m - 1; i >= 0; --i) {
        if ((lab >> i) & 1u) {
            st.push_back(i);
        } else {
            const int t = st.back();
            st.pop_back();
            par[i] = t;
            par[t] = i;
        }
    }
}

static int check_lists(int m) {
    const uint32_t rows = B.n[m][1];
    std::vector<int> up, lo;
    long ones = 0;
    uint32_t longest = 0;
    for (uint32_t l = 0; l < rows; ++l) {
        arcs(m, labels_of(B, m, l), up);
        std::vector<uint32_t> want;
        for (uint32_t c = 0; c < rows; ++c) {
            arcs(m, labels_of(B, m, c), lo);  // strand i of the lower word is strand m-1-i of the upper one
            int at = up[m], seen = 1;
            while (true) {
                const int t = lo[m - 1 - at];
                if (t == m) break;
                at = up[m - 1 - t];
                ++seen;
                if (at == m) break;  // back at the upper end: cannot happen
                ++seen;
            }
            if (seen == m) want.push_back(c);
        }
        std::vector<uint32_t> got = row_of(m, l);
        std::sort(got.begin(), got.end());
        if (got != want) {
            printf("MISMATCH list m=%d row=%u\n", m, l);
            return 1;
        }
        ones += (long)got.size();
        longest = std::max(longest, (uint32_t)got.size());
        if (rank_of(B, m, labels_of(B, m, l)) != l) return 1;
        if (m >= 5) {  // the second arc's place lies below the first one's or around it
            const int b1 = top_arc(labels_of(B, m, l));
            if (top_arc(without_pair(labels_of(B, m, l), b1)) >= b1) return 1;
        }
    }
    if (ones != (long)kOnes[m / 2] || longest != kLongest[m / 2]) {
        printf("MISMATCH constants m=%d: %ld ones, longest %u\n", m, ones, longest);
        return 1;
    }
    printf("ok lists m=%d ones=%ld\n", m, ones);
    return 0;
}

template <typename Idx>
static int check_solve(int n, uint32_t mod) {
    const int W = n + 1, c = (W & 1) ? (W - 1) / 2 : -1;
    std::vector<uint32_t> u(H[W][1], 0), z(H[W - 1][1], 0);
    u[H[W - 1][1]] = 1 % mod;  // R at position W-1
    for (int r = 0; r < W / 2; ++r) or_apply_cells(n, mod, u.data(), z.data(), W - 1, 1, 0, 1);
    if (c >= 0) or_apply_cells(n, mod, u.data(), z.data(), W - 1, c + 1, 0, 1);
    cell::Pair<Idx> D[kMaxW][kCols];
    for (int p = 0; p < kMaxW; ++p)
        for (int h = 0; h < kCols; ++h)
            D[p][h] = cell::Pair<Idx>{(Idx)H[p][h], (Idx)(H[p][h] + (h > 0 ? H[p][h - 1] : 0))};
    std::vector<char> hit(u.size(), 0);
    unsigned __int128 total = 0;
    for (int m = 1; m <= W; m += 2) {
        std::vector<std::vector<uint32_t>> rows;
        for (uint32_t l = 0; l < B.n[m][1]; ++l) rows.push_back(row_of(m, l));
        for (uint32_t i = 0; i < bin[W * 32 + m]; ++i) {
            const uint32_t o = mask_of(bin, W, m, i);
            if ((o >> W) || __builtin_popcount(o) != m) return 2;
            const int w = mask_weight(o, W, c);
            const uint32_t ro = reversed_mask(o, W);
            for (uint32_t l = 0; l < rows.size(); ++l) {
                const uint64_t iu = word_rank<Idx>(D, o, labels_of(B, m, l), 31);
                if (iu >= u.size()) return 3;
                hit[iu]++;
                if (!w) continue;
                uint64_t x = u[iu];
                if (w == 2) x *= 2;
                if (w == 3) {
                    const uint64_t ib = word_rank<Idx>(D, o, labels_of(B, m, l), c);
                    if (ib >= z.size()) return 4;
                    x += 2ull * z[ib];
                }
                uint64_t sum = 0;
                for (uint32_t k : rows[l]) sum += u[word_rank<Idx>(D, ro, labels_of(B, m, k), 31)];
                total += (unsigned __int128)(x % mod) * sum;
            }
        }
    }
    for (char h : hit)
        if (h != 1) return 5;  // every main word is a (occupancy, label rank) once
    int err = 0;
    const uint32_t want = or_solve(n, mod, 1, &err), got = (uint32_t)(total % mod);
    printf("%s n=%d mod=%u idx=%d got=%u want=%u\n", got == want && !err ? "ok" : "MISMATCH", n, mod, (int)sizeof(Idx) * 8, got,
           want);
    return got == want && !err ? 0 : 1;
}

int main(int argc, char** argv) {
    const int nmax = argc > 1 ? atoi(argv[1]) : 10;
    build_ballot(B);
    H[0][0] = 1;
    for (int w = 1; w < kDpRows; ++w)
        for (int h = 0; h < kDpCols; ++h)
            H[w][h] = H[w - 1][h] + (h > 0 ? H[w - 1][h - 1] : 0) + (h + 1 < kDpCols ? H[w - 1][h + 1] : 0);
    for (int p = 0; p < kMaxW; ++p)
        for (int q = 0; q < 32; ++q) bin[p * 32 + q] = q == 0 ? 1 : (p == 0 ? 0 : bin[(p - 1) * 32 + q] + bin[(p - 1) * 32 + q - 1]);
    for (int m = 1; m <= 13; m += 2)
        if (check_lists(m)) return 1;
    for (int n = 3; n <= nmax; ++n)
        for (uint32_t mod : {4294967291u, 2u, 4294966997u}) {
            const int e = n % 2 ? check_solve<uint32_t>(n, mod) : check_solve<uint64_t>(n, mod);
            if (e) {
                printf("FAILED n=%d (%d)\n", n, e);
                return 1;
            }
        }
    printf("ALL OK\n");
    return 0;
}
