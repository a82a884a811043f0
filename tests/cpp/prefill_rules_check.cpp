// The prefill kernel that the rules (mugen_amd/csrc/prefill_rules.h) choose:
// reads lines "n_tokens start_pos causal n_heads n_kv_heads head_dim", prints one
// name each (the short-prompt kernel and key splits, tested elsewhere, come first).
#include <cstdio>

#include "prefill_rules.h"

using namespace mugen_attn;

int main() {
    int n, start, causal, h, hk, d;
    while (std::scanf("%d %d %d %d %d %d", &n, &start, &causal, &h, &hk, &d) == 6)
        std::puts(prefill_rows_default(n, start, causal != 0, h / hk, hk, d) ? "rows"
                  : prefill_ws_default(n, h / hk, d)                         ? "ws"
                                                                             : "block");
    return 0;
}
