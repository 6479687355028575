// Host check of the launches of a half-row solve's last step (class_shape and block_sum in
// oneesan-gpu_amd/csrc/ofp_glue_impl.h): no 64-bit sum can wrap at any width, moduli count
// and CU count, and the bounds hold for the kernel's own walk over its tasks.
// Built and run by tests/test_glue_sums.py; "ALL OK" at the end.
#include <cstdio>
#include <vector>

#include "../../oneesan-gpu_amd/csrc/ofp_glue_impl.h"

using namespace ofp;
using namespace ofp::glue;

static uint32_t bin[kMaxW * 32];

// glue_kernel's walk: tasks of each strand count per block of one pass, each task once.
static int walk(const Class& c, int W, int K, int cus) {
    const Shape s = class_shape(c, W, K, cus, bin);
    if (!s.tasks) return 0;
    std::vector<int> ms;
    std::vector<uint64_t> end;
    uint64_t total = 0;
    for (int m = c.hi; m >= c.lo; m -= 2)
        if (m <= W) {
            ms.push_back(m);
            end.push_back(total += bin[W * 32 + m]);
        }
    const uint32_t nw = (s.blocks >> 3) / s.passes, P = s.piece * s.teams;
    std::vector<char> hit(s.tasks, 0);
    for (uint32_t xcd = 0; xcd < 8; ++xcd) {
        std::vector<uint64_t> onx(ms.size(), 0);
        for (uint32_t b = 0; b < nw; ++b) {
            std::vector<uint64_t> mine(ms.size(), 0);
            for (uint32_t q = b * s.teams;; q += nw * s.teams) {
                const uint32_t first = (q / P * 8 + xcd) * P + q % P;
                if (first >= s.tasks) break;
                for (uint32_t t = first; t < first + s.teams && t < s.tasks; ++t) {
                    if (hit[t]++) return 1;
                    size_t g = 0;
                    while (t >= end[g]) ++g;
                    ++mine[g];
                    ++onx[g];
                }
            }
            for (size_t g = 0; g < ms.size(); ++g)
                if (mine[g] > block_tasks(s, bin[W * 32 + ms[g]])) return 2;
        }
        for (size_t g = 0; g < ms.size(); ++g)
            if (onx[g] > xcd_tasks(s, bin[W * 32 + ms[g]])) return 3;
    }
    for (char h : hit)
        if (h != 1) return 4;
    return 0;
}

int main() {
    Ballot B;
    build_ballot(B);
    for (int p = 0; p < kMaxW; ++p)
        for (int q = 0; q < 32; ++q) bin[p * 32 + q] = q == 0 ? 1 : (p == 0 ? 0 : bin[(p - 1) * 32 + q] + bin[(p - 1) * 32 + q - 1]);
    int raised = 0, launches = 0;
    double most = 0;
    for (int W = 4; W <= kSumStrands + 1; ++W) {
        for (int cus : {1, 4, 16, 64, 80, 128, 256, 304})
            for (int K = 1; K <= 1024; K = K < 40 ? K + 1 : K + K / 3)
                for (const Class& c : kClasses) {
                    const Shape s = class_shape(c, W, K, cus, bin);
                    if (!s.tasks) continue;
                    const double sum = block_sum(s, c, W, bin);
                    if (!(sum < kSumLimit) || s.blocks % (8 * s.passes)) {
                        printf("MISMATCH W=%d K=%d cus=%d m=%d..%d\n", W, K, cus, c.lo, c.hi);
                        return 1;
                    }
                    ++launches;
                    raised += (uint64_t)s.blocks > 8ull * s.passes && s.blocks > (uint32_t)cus * c.per_cu;
                    if (cus == 256 && K <= 16 && sum > most) most = sum;
                }
        // the low halves: one product per word, in the sums of an XCD's blocks
        double low = 0;
        for (int m = 1; m <= W; m += 2) {
            uint64_t tasks = bin[W * 32 + m];
            if (m <= kTabStrands) {
                for (const Class& c : kClasses)
                    if (m >= c.lo && m <= c.hi) tasks = xcd_tasks(class_shape(c, W, 1, 256, bin), tasks);
                low += (double)tasks * B.n[m][1];
            } else {  // workgroups of 256 words, in turn, of each batch
                low += (double)tasks * B.n[m][1] / 8 + 256.0 * (double)tasks;
            }
        }
        if (!(low * 4294967296.0 < kSumLimit)) {
            printf("MISMATCH low sums W=%d\n", W);
            return 1;
        }
    }
    if (!raised) return 1;  // some launch needed more blocks than are resident
    for (int W : {4, 5, 9, 12, 13, 16, 17, 20, 23})
        for (int cus : {2, 60, 256})
            for (int K : {1, 3, 8, 25, 190})
                for (const Class& c : kClasses)
                    if (const int e = walk(c, W, K, cus)) {
                        printf("MISMATCH walk W=%d K=%d cus=%d m=%d..%d (%d)\n", W, K, cus, c.lo, c.hi, e);
                        return 1;
                    }
    printf("%d launches, %d raised, most %.3g of 2^64 at 256 CUs and up to 16 moduli\nALL OK\n", launches, raised, most / kSumLimit);
    return 0;
}
