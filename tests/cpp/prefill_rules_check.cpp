// The prefill kernel that the rules (mugen_amd/csrc/prefill_rules.h) choose:
// reads lines "n_tokens start_pos causal n_heads n_kv_heads head_dim", prints one
// name each (the short-prompt kernel and key splits, tested elsewhere, come first).
// With an argument: reads "slots part", prints the byte offset of a split call's
// partials from its (max, sum) pairs and the bytes that its workspace has.
#include <cstdio>

#include "prefill_rules.h"

using namespace mugen_attn;

int main(int argc, char**) {
    if (argc > 1) {
        size_t slots, part;
        while (std::scanf("%zu %zu", &slots, &part) == 2)
            std::printf("%zu %zu\n", prefill_partials_at(slots) * sizeof(float), prefill_split_bytes(slots, part));
        return 0;
    }
    int n, start, causal, h, hk, d;
    while (std::scanf("%d %d %d %d %d %d", &n, &start, &causal, &h, &hk, &d) == 6)
        if (d > 128)
            std::puts(prefill_wide_rows_default(n, start, causal != 0, h / hk, hk, d) ? "rows" : "pairs");
        else
            std::puts(prefill_rows_default(n, start, causal != 0, h / hk, hk, d) ? "rows"
                  : prefill_ws_default(n, h / hk, d)                         ? "ws"
                                                                             : "block");
    return 0;
}
