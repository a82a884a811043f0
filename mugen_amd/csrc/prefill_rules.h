// prefill_rules.h -- which prefill kernel takes a prompt, and where a split call's partials lie.  Plain integer C++, so that
// tests/cpp/prefill_rules_check.cpp prints the same on the host.
#pragma once
#include <cstddef>
#include <cstdint>

namespace mugen_attn {

// The warp-specialised kernel (else the per-block one), below the flattened-row
// kernel's sizes: above head_dim 64 and for more than 4 heads per kv head (graph
// replays, us: Qwen2.5-7B shape N = 16 / 256 / 768 5.9 / 10.7 / 21.6 against 7.5 /
// 11.9 / 22.4 per-block, H32 Hk8 d128 N = 768 18.0 against 26.5; H16 Hk2 d64 N = 256
// 7.4 against 8.0); 4-head blocks at head_dim 64 from 1024 to 4096 tokens (below,
// the per-block and short-prompt kernels lead: N = 512 7.7 against 9.2; above,
// where few kv heads make too few flattened-row blocks, f16, per-block /
// warp-specialised: 8 / 2 heads N = 4200 46.0 / 48.0, 6500 68 / 79, 9900 157 / 170;
// 9 / 3 heads 6000 86 / 89; 4 / 1 heads 4200 33 / 47, 8192 65 / 88, 20000 277 / 345)
inline bool prefill_ws_default(int n_tokens, int G, int head_dim) {
    return head_dim > 64 || G > 4 || (n_tokens >= 1024 && n_tokens <= 4096);
}

// The flattened-row kernel where its 128-row blocks make enough workgroups (two
// share a CU, three at head_dim 64) that the longest causal rows' chain does not
// set the time, by how full the other kernels' head slots are: us, the faster
// of those two / flattened.
//  * head_dim above 64.  One or two heads per kv head (4-head blocks half full)
//    256 workgroups: 8 / 8 heads 129 / 83, 16 / 8 47 / 44, 2 / 1 315 / 313, 128
//    workgroups 40 / 44.  Up to 4: 512: 32 / 8 52.5 / 50.7, 8 / 2 191 / 182, 4 / 1
//    375 / 360, 16 / 2 (8 heads each) 77 / 94.  More: 640: 28 / 4 heads 88 / 78,
//    448 workgroups 42 / 48.  Where few kv heads make the blocks few and long, or
//    all are equally long, 8-head slots full or one short need more: 8 / 1 640 243 /
//    254, 768 333 / 324; after as many tokens 28 / 4 640 221 / 233, 768 321 / 296;
//    32 / 4 640 185 / 187, 768 244 / 261 or 278 / 259 (where the other kernel's last
//    round is full, or not), 1028 474 / 473, 1284 709 / 677.
//  * head_dim 64.  One head per kv head 256: 16 / 16 43 / 34.  Two: more with fewer,
//    longer chains, for which the per-block kernel's steps are shorter: 16 / 8 256
//    27.3 / 34.0, 320 43.0 / 41.3; 8 / 4 320 77.2 / 77.4; 4 / 2 256 89 / 120, 384 182 /
//    179; 2 / 1 384 334 / 356, 448 446 / 415; equally long 256: 16 / 8 after 8000 181 /
//    150, 8 / 4 131 / 122, 2 / 1 448 / 477.  More: 640: 32 / 8 512 34 / 37, 768 66 / 58;
//    14 / 2 448 49 / 63, 656 105 / 98; with full slots and one kv head 800: 4 / 1 640
//    290 / 325, 750 388 / 399, 813 452 / 446; 8 / 1 640 158 / 166, 800 233 / 226.
inline bool prefill_rows_default(int n_tokens, int start_pos, bool causal, int G, int n_kv_heads, int head_dim) {
    if ((int64_t)n_tokens * G > INT32_MAX - 127) return false;  // the kernel numbers the rows in 32 bits
    const int64_t wgs = ((int64_t)n_tokens * G + 127) / 128 * n_kv_heads;
    const bool level = !causal || start_pos >= n_tokens;  // blocks of about the same key count
    int least = 640;
    if (head_dim > 64) {
        if (G <= 4) least = G <= 2 ? 256 : 512;
        else if (G % 8 == 0) least = level ? 1088 : n_kv_heads <= 2 ? 768 : 640;
        else if (G % 8 == 7 && level) least = 768;
    } else if (G == 1) {
        least = 256;
    } else if (G == 2) {
        least = level ? (n_kv_heads > 1 ? 256 : 320) : n_kv_heads >= 4 ? 320 : n_kv_heads > 1 ? 384 : 448;
    } else if (!level && n_kv_heads == 1 && G % 4 == 0) {
        least = 800;
    }
    return wgs >= least;
}

// head_dim above 128, keys not split: up to one round of (token, kv head) pairs,
// at head_dim below 256 two, run one pair to a workgroup, whose four waves share
// the pair's keys; past it the flattened-row kernel, which pads every head to 256
// columns where a pair moves head_dim.  us, per pair / flattened: 16 / 8 heads d256
// N = 32 5.4 / 7.1, 64 9.9 / 8.5, 256 53 / 14.8; d256 260 to 512 pairs 0.75 to 1.0 of
// the pairs' time at 1 to 16 kv heads.  d136: 1 / 1 heads N = 290 15.9 / 19.7, 600
// 32 / 28; 4 / 4 110 10.5 / 13.0, 150 19 / 15; d192: 4 / 4 110 11.1 / 13.5, 150 20 / 16.
// With 64 heads and more the blocks fill sooner: 128 / 16 heads d136 N = 17 11.8 /
// 10.5, 64 / 8 33 11.8 / 11.2, 64 / 16 17 10.7 / 10.1 (after as many tokens 11.1 / 11.4)
inline bool prefill_wide_rows_default(int n_tokens, int start_pos, bool causal, int G, int n_kv_heads, int head_dim) {
    const bool level = !causal || start_pos >= n_tokens;
    const bool early = head_dim == 256 || (G * n_kv_heads >= 64 && (G >= 8 || !level));
    return (int64_t)n_tokens * n_kv_heads > (early ? 256 : 512);
}

// Key splits: floats from the (max, sum) pairs, at a 256-byte boundary of the
// workspace, to the partials, which are read and written 16 bytes at a time: the
// pairs of an odd number of (row, split) slots end between two such words
inline size_t prefill_partials_at(size_t slots) { return (slots * 2 + 63) / 64 * 64; }
// bytes for that many slots of `part` bytes, with both roundings
inline size_t prefill_split_bytes(size_t slots, size_t part) { return slots * (part + 2 * sizeof(float)) + 512; }

}  // namespace mugen_attn
