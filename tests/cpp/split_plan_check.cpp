// The device split plan's arithmetic (mugen_amd/csrc/split_plan.h) on the host:
// over batches, kv heads, split caps and lengths, the planned work list never
// has more items than the launch has workgroups, and no sequence more splits
// than the workspace has slots.  The reciprocal is taken exact and one unit in
// the last place to either side, as the device's may be.
//
// Usage: split_plan_check SEED DRAWS.  Prints every violation; exit status 1 if
// there is one.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

static int g_ulp = 0;
static float host_rcp(float x) {
    const float r = 1.0f / x;
    return g_ulp == 0 ? r : std::nextafter(r, g_ulp > 0 ? 2.0f * r : 0.0f);
}
#define MUGEN_PLAN_RCP(x) host_rcp(x)
#define MUGEN_PLAN_SQRT(x) std::sqrt(x)
#include "split_plan.h"

using namespace mugen_attn;

namespace {

int units(int t) { return (t + 31) / 32; }
int exact_ceil(int a, int b) { return (a + b - 1) / b; }

struct Case {
    int kinds, mult, budget, cmin, cap;
    bool empty_counts;         // (GQA, where cmin is fixed; else MLA) an empty sequence still has one split
    std::vector<int> T, nq;    // tokens, of which quantised (kinds 2)
    int longest = 1 << 30;     // the longest chunk that is good enough
};

int run_of(const Case& c, int j, int kind) {  // units of one run of a sequence
    return c.kinds == 1 ? units(c.T[j]) : kind == 0 ? units(c.nq[j]) : units(c.T[j] - c.nq[j]);
}

int violations = 0;
void check(const Case& c, const char* what) {
    const int B = (int)c.T.size();
    int sum = 0, mx = 0;
    for (int j = 0; j < B; j++) {
        int u = 0;
        for (int k = 0; k < c.kinds; k++) u += run_of(c, j, k);
        sum += u;
        mx = u > mx ? u : mx;
    }
    auto total = [&](int x, float rx) {
        int n = 0;
        for (int j = 0; j < B; j++) {
            int s = 0;
            for (int k = 0; k < c.kinds; k++) s += ceil_div_f(run_of(c, j, k), x, rx);
            n += c.empty_counts && s == 0 ? 1 : s;
        }
        return n;
    };
    // MLA: mult blocks of 64 query rows
    const int cmin = c.empty_counts ? c.cmin : plan_mla_least(sum, 64 * c.mult);
    const int c0 = plan_by_cap(mx, cmin, c.cap);
    int chunk;
    if (B <= 8)
        chunk = c.kinds == 1 ? plan_few<1>(B, c.mult, c.budget, c0, c.cap, sum, mx, total)
                             : plan_few<2>(B, c.mult, c.budget, c0, c.cap, sum, mx, total);
    else
        chunk = c.kinds == 1 ? plan_many<1>(B, c.mult, c.budget, c0, sum, mx, total)
                             : plan_many<2>(B, c.mult, c.budget, c0, sum, mx, total);
    long items = 0;
    int most = 0;
    for (int j = 0; j < B; j++) {
        int s = 0;
        for (int k = 0; k < c.kinds; k++) s += exact_ceil(run_of(c, j, k), chunk);
        most = s > most ? s : most;
        items += c.empty_counts && s == 0 ? 1 : s;
    }
    items *= c.mult;
    // workgroups of the launch: one round, or every slot of every sequence
    const long slots = c.cap + c.kinds - 1, wgs = std::min<long>(c.budget, (long)B * c.mult * slots);
    if (chunk < cmin || items > wgs || most > slots || chunk > c.longest) {
        violations++;
        if (violations <= 20) {
            std::printf("%s: kinds %d batch %d mult %d budget %d cap %d ulp %d: chunk %d, %ld items for %ld workgroups, "
                        "%d splits for %ld slots; lengths", what, c.kinds, B, c.mult, c.budget, c.cap, g_ulp, chunk,
                        items, wgs, most, slots);
            for (int j = 0; j < B && j < 8; j++) std::printf(" %d", c.T[j]);
            std::printf("\n");
        }
    }
}

void store(std::vector<int> T, int mult, int budget, int cap, int keep, const char* what) {
    Case c{2, mult, budget, 2, cap, true, T, T};
    for (int& n : c.nq) n = std::max(0, n - keep);
    check(c, what);
}

}  // namespace

// MLA's least chunk: 128 rows, 8 ragged sequences of up to 1638 tokens (64-token
// chunks there have more partials to merge than tiles to walk), 3 full ones of 8192,
// whose 32 even splits stay, and a short one
void least(int sum, int R, int lo, int hi) {
    const int c = plan_mla_least(sum, R);
    if (c < lo || c > hi) {
        violations++;
        std::printf("least chunk of %d units, %d rows: %d, not %d..%d\n", sum, R, c, lo, hi);
    }
}

int main(int argc, char** argv) {
    least(225, 128, 4, 6);
    least(768, 128, 1, 8);
    least(8, 128, 1, 1);
    least(225, 16, 1, 2);
    std::mt19937 rng(argc > 1 ? (unsigned)std::atoi(argv[1]) : 1u);
    const int draws = argc > 2 ? std::atoi(argv[2]) : 20000;
    auto pick = [&](int lo, int hi) { return (int)(lo + rng() % (unsigned)(hi - lo + 1)); };
    for (g_ulp = -1; g_ulp <= 1; g_ulp++) {
        // batches that lost items to the two roundings of the store
        store({4600, 5853, 3424, 4723, 5733, 5020, 4463, 3623}, 8, 512, 32, 256, "8 sequences x 8 kv heads");
        store({3054, 3054, 3054, 3054}, 4, 512, 32, 256, "4 equal sequences x 4 kv heads");
        store({7168, 7168, 7168, 7168}, 4, 512, 32, 256, "4 equal sequences x 4 kv heads");
        store({8000, 1024, 1024, 1024, 1024, 1024, 1024, 1024}, 32, 512, 32, 256, "8 sequences x 32 kv heads");
        store(std::vector<int>(6, 5000), 8, 512, 32, 256, "6 equal sequences x 8 kv heads");
        // equal sequences that fill the round exactly, cut in halves
        check({1, 8, 512, 2, 32, true, std::vector<int>(32, 8192), {}, 128}, "32 full sequences x 8 kv heads");
        check({1, 8, 256, 2, 32, true, std::vector<int>(16, 4096), {}, 64}, "16 full sequences x 8 kv heads");
        check({1, 4, 512, 2, 32, true, std::vector<int>(32, 4096), {}, 32}, "32 full sequences x 4 kv heads");
        // every batch up to 64 that plans on the device, equal lengths and drawn
        // ones, every split cap that a workspace can leave
        const int budgets[] = {256, 512, 256};  // GQA above head_dim 128 and up to it, MLA
        for (int bi = 0; bi < 3; bi++)
            for (int B = 1; B <= 64; B++)
                for (int mult = 1; mult <= 32; mult++) {
                    if (B * mult * 2 > budgets[bi]) continue;
                    for (int T : {0, 1, 31, 33, 700, 3054, 4097, 7168, 8191, 32768}) {
                        if (bi < 2) store(std::vector<int>(B, T), mult, budgets[bi], 32, pick(0, 600), "equal");
                        check({1, mult, budgets[bi], bi == 2 ? 1 : 2, 32, bi < 2, std::vector<int>(B, T), {}}, "equal");
                    }
                }
        for (int i = 0; i < draws; i++) {
            const int bi = pick(0, 2), budget = budgets[bi], room = budget / 2;
            const int B = pick(0, 1) ? pick(1, 8) : pick(1, 64);
            const int mult = pick(1, std::max(1, room / B));
            if (B * mult > room) continue;
            const int hi = pick(1, pick(0, 3) ? 8191 : 200000), lo = std::max(0, hi / pick(1, 16) - pick(0, 1));
            std::vector<int> T(B);
            for (int& t : T) t = pick(0, 15) ? pick(lo, hi) : 0;
            if (bi < 2) store(T, mult, budget, pick(0, 1) ? 32 : pick(1, 32), pick(0, 1000), "drawn");
            check({1, mult, budget, bi == 2 ? 1 : 2, pick(0, 1) ? 32 : pick(2, 33), bi < 2, T, {}}, "drawn");
        }
    }
    std::printf("%d violations\n", violations);
    return violations != 0;
}
