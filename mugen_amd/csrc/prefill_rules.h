// prefill_rules.h -- which prefill kernel takes a prompt at head_dim up to 128.
// Plain integer C++, so that tests/cpp/prefill_rules_check.cpp prints the same
// choices on the host.
#pragma once
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

}  // namespace mugen_attn
