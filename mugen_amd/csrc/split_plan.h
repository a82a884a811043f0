// split_plan.h -- arithmetic of the context-split plan made on the device
// (plan_chunk_device, common.h): which chunk cuts the sequences of a batch into
// a work list that the launch's workgroups cover.  Plain integer and float C++,
// so that tests/cpp/split_plan_check.cpp runs the same code on the host.
#pragma once

#ifdef __HIPCC__
#define MUGEN_PLAN_FN __device__ __forceinline__
#else
#define MUGEN_PLAN_FN inline
#endif
// 1 / x to one unit in the last place (v_rcp_f32)
#ifndef MUGEN_PLAN_RCP
#define MUGEN_PLAN_RCP(x) __builtin_amdgcn_rcpf(x)
#endif
#ifndef MUGEN_PLAN_SQRT
#define MUGEN_PLAN_SQRT(x) __builtin_amdgcn_sqrtf(x)
#endif

namespace mugen_attn {

MUGEN_PLAN_FN int plan_max(int a, int b) { return a > b ? a : b; }
MUGEN_PLAN_FN float plan_rcp(int d) { return MUGEN_PLAN_RCP((float)d); }

// ceil(n / d) for 0 <= n < 2^23, 1 <= d, rd = 1.0f / d to one ulp: the product
// is within one of the quotient, the remainder tells which
MUGEN_PLAN_FN int ceil_div_f(int n, int d, float rd) {
    const int x = n + d - 1;
    const int q = (int)((float)x * rd);
    const int r = x - q * d;
    return r < 0 ? q - 1 : r >= d ? q + 1 : q;
}

// an upper bound of ceil(n / d), at most one above it
MUGEN_PLAN_FN int plan_div_up(int n, int d) { return (int)((float)n * plan_rcp(d) * (1.0f + 4e-6f)) + 1; }

// the smallest chunk (in units, at least cmin) that cuts mx units into at most
// cap splits
MUGEN_PLAN_FN int plan_by_cap(int mx, int cmin, int cap) {
    return plan_max(cmin, cap == 32 ? (mx + 31) >> 5 : ceil_div_f(mx, cap, plan_rcp(cap)));
}

// c, raised by a sixteenth at a time until its work list -- mult items for each
// of the total(c, 1 / c) splits -- fits `budget`.  It ends at mx, where every
// sequence is one split of each kind: the callers see to it that those fit
template <typename Total>
MUGEN_PLAN_FN int plan_grow(int c, int mx, int mult, int budget, Total total) {
    while (c < mx && total(c, plan_rcp(c)) * mult > budget) c += plan_max(1, c >> 4);
    return c;
}

// The plan of a few sequences from their units' sum and maximum mx.  KINDS: how
// many runs of a sequence are split on their own (2: the 4-bit store's Q4 and
// f16 tokens), each rounded up, so that a sequence has up to ceil(units / c) +
// KINDS - 1 splits.  c0 = plan_by_cap.  KINDS B mult <= budget.
template <int KINDS, typename Total>
MUGEN_PLAN_FN int plan_few(int B, int mult, int budget, int c0, int cap, int sum, int mx, Total total) {
    // work lists that fit however the sequences are cut: the split cap alone
    if (B * mult * (cap + KINDS - 1) <= budget || mx == 0) return c0;
    // one guess: half a split's tokens lost per rounding; the longest sequence
    // cut evenly, where that still fits
    int c = plan_max(c0, plan_div_up(sum * mult, budget - KINDS * B * mult / 2) - 1);
    const int ns = ceil_div_f(mx, c, plan_rcp(c));
    c = plan_max(c0, ceil_div_f(mx, ns, plan_rcp(ns)));
    // the store: its two roundings leave no room for a closed bound where the
    // batch fills half the round (budget = KINDS B mult), so the count decides
    if (KINDS > 1) return plan_grow(c, mx, mult, budget, total);
    // else the bound sum mult / (budget - B mult): one rounding per sequence, so
    // it always fits (one sequence: a search cost 0.8 us of a 7 us call)
    if (total(c, plan_rcp(c)) * mult > budget) c = plan_max(c0, plan_div_up(sum * mult, budget - B * mult));
    return c;
}

// The plan of more sequences, a search: the longest sequence cut evenly at the
// guess of half a split lost per sequence, where that fits (32 equal sequences
// fill the round exactly with two halves each: 32 / 8 heads d128, full caches of
// 8192, 222 -> 200 us against two thirds and one), else the smallest chunk to 1/16
// from that guess.  A store whose two runs per sequence leave room for less than
// half a split more each takes one split of each at once (32 / 8 heads, 32
// sequences: the search took 4.7 of 42 us)
template <int KINDS, typename Total>
MUGEN_PLAN_FN int plan_many(int B, int mult, int budget, int c0, int sum, int mx, Total total) {
    if (KINDS > 1 && (2 * KINDS + 1) * B * mult > 2 * budget) return plan_max(c0, mx);
    const int c = plan_max(c0, plan_div_up(sum * mult, budget - KINDS * B * mult / 2) - 1);
    const int ns = ceil_div_f(mx, c, plan_rcp(c));
    if (mx > 0) {
        const int even = plan_max(c0, ceil_div_f(mx, ns, plan_rcp(ns)));
        if (total(even, plan_rcp(even)) * mult <= budget) return even;
    }
    return plan_grow(c, mx, mult, budget, total);
}

// MLA decode: the least chunk (units) for `sum` units of R query rows.  A unit is
// ~0.4 us of a workgroup's time, and a split's partials (R x 512 x 2 bytes there and
// back) ~0.1 us of the call at 128 rows, so the sum of both is least around
// sqrt(sum R / 600) (128 heads, caches of 8192, us at 64 / 128 / 192 / 256 tokens: 8
// sequences of 200..1638 23.3 / 16.9 / 16.4 / 16.9, 4 19.0 / 15.3 / 15.3 / 16.1, 8 of
// 80..400 13.3 / 13.5 / 14.6 / 15.9).  Less than that: full caches keep their 32 even
// splits (3 of 8192 tokens 20.3 us at 8 units, 22.4 at 9)
MUGEN_PLAN_FN int plan_mla_least(int sum, int R) {
    return plan_max(1, (int)(MUGEN_PLAN_SQRT((float)sum * (float)R * (1.0f / 1400.0f)) + 0.5f));
}

}  // namespace mugen_attn
