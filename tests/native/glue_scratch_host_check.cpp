// Host check of a half-row solve's sums over words of more strands than are listed
// (pull_entry, upper_node and task_entries in oneesan-gpu_amd/csrc/ofp_glue_impl.h): the
// levels of a task's scratch filled as the kernels fill them, with smaller list limits,
// every entry index range-checked and written before it is read, against sums over the
// words' own lists.  And the sizes of the lists (kOnes, kLongest, chunk_bound) up to 19
// strands.  Built and run by tests/test_glue_scratch.py; "ALL OK" at the end.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "../../oneesan-gpu_amd/csrc/ofp_glue_impl.h"

using namespace ofp;
using namespace ofp::glue;

static Ballot B;
using Rows = std::vector<std::vector<uint32_t>>;

// The lists of m strands from those of m - 2, as the list kernels make them.
static Rows next_rows(int m, const Rows& below) {
    Rows out(B.n[m][1]);
    for (uint32_t l = 0; l < out.size(); ++l) {
        const uint32_t lab = labels_of(B, m, l);
        const int p = top_arc(lab);
        for (uint32_t v : below[rank_of(B, m - 2, without_pair(lab, p))])
            preimages(m, labels_of(B, m - 2, v), m - 2 - p, [&](uint32_t w) { out[l].push_back(rank_of(B, m, w)); });
    }
    return out;
}

static int check_scratch(int m, int tab, const Rows& listed, const Rows& own) {
    const uint32_t each = task_entries(B, m, tab);
    std::vector<uint64_t> s(each, 0);
    std::vector<char> set(each, 0);
    uint64_t x = 0x9e3779b97f4a7c15ull;
    for (uint32_t l = 0; l < B.n[m][1]; ++l) {
        x = x * 6364136223846793005ull + 1442695040888963407ull;
        s[l] = x >> 44;
        set[l] = 1;
    }
    uint32_t from = 0, to = B.n[m][1];
    for (int r = 0; r < (m - tab) / 2; ++r) {
        const uint32_t arrays = level_arrays(m, r), rows = B.n[m - 2 * r - 2][1];
        for (uint32_t node = 0; node < arrays; ++node)
            for (uint32_t l = 0; l < rows; ++l) {
                int bad = 0;
                uint64_t sum = 0;
                const bool place = pull_entry(B, m, r, from, node, l, [&](uint32_t i) {
                    if (i < from || i >= to || !set[i]) bad = 1;
                    else sum += s[i];
                });
                if (bad) return 1;
                const uint32_t o = to + node * rows + l;
                if (o >= each || set[o]) return 2;
                if (!place) continue;
                s[o] = sum;
                set[o] = 1;
            }
        from = to;
        to += arrays * rows;
    }
    if (to != each) return 3;
    const uint32_t rows = B.n[tab][1];
    for (uint32_t l = 0; l < B.n[m][1]; ++l) {
        uint32_t lab = labels_of(B, m, l);
        const uint32_t node = upper_node(m, tab, lab), y = from + node * rows;
        uint64_t got = 0, want = 0;
        for (uint32_t c : listed[rank_of(B, tab, lab)]) {
            if (y + c >= each || !set[y + c]) return 4;
            got += s[y + c];
        }
        for (uint32_t c : own[l]) want += s[c];
        if (got != want) return 5;
    }
    return 0;
}

int main() {
    build_ballot(B);
    std::vector<Rows> g(kTabStrands + 1);
    g[1] = {{0}};
    for (int m = 3; m <= 17; m += 2) g[m] = next_rows(m, g[m - 2]);
    for (int m = 1; m <= kTabStrands; m += 2) {
        std::vector<uint32_t> len(B.n[m][1], 0);
        for (uint32_t l = 0; l < len.size(); ++l) {
            if (m <= 17) {
                len[l] = (uint32_t)g[m][l].size();
                continue;
            }
            const uint32_t lab = labels_of(B, m, l);
            const int p = top_arc(lab);
            for (uint32_t v : g[m - 2][rank_of(B, m - 2, without_pair(lab, p))])
                len[l] += preimage_count(m, labels_of(B, m - 2, v), m - 2 - p);
        }
        std::sort(len.rbegin(), len.rend());
        uint64_t ones = 0, chunks = 0;
        for (uint32_t v : len) ones += v;
        for (size_t i = 0; i < len.size(); i += 64) chunks += (len[i] + 7) / 8;
        if (ones != kOnes[m / 2] || len[0] != kLongest[m / 2] || chunks > chunk_bound(m, (uint32_t)len.size())) {
            printf("MISMATCH sizes m=%d: %lu ones, longest %u, %lu chunks\n", m, ones, len[0], chunks);
            return 1;
        }
    }
    for (int tab = 3; tab <= 9; tab += 2)
        for (int m = tab + 2; m <= tab + 4; m += 2)
            if (const int e = check_scratch(m, tab, g[tab], g[m])) {
                printf("MISMATCH scratch m=%d listed to %d (%d)\n", m, tab, e);
                return 1;
            }
    printf("ALL OK\n");
    return 0;
}
