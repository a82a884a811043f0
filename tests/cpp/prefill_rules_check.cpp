// The prefill kernel that the rules (mugen_amd/csrc/prefill_rules.h) choose:
// reads lines "n_tokens n_heads n_kv_heads head_dim", prints one name each.
#include <cstdio>

#include "prefill_rules.h"

using namespace mugen_attn;

int main() {
    int n, h, hk, d;
    while (std::scanf("%d %d %d %d", &n, &h, &hk, &d) == 4)
        std::puts(prefill_ws_default(n, h / hk, d) ? "ws" : "block");
    return 0;
}
