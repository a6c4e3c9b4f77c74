// Evaluates the launch rules (gemma4-webgpu_amd/csrc/launch_rules.h) for tests/test_launch_rules.py: reads
// "<rule> <arguments>" lines and prints one value a line.
#include <stdio.h>

#include <iostream>
#include <string>

#include "../gemma4-webgpu_amd/csrc/launch_rules.h"

int main() {
    std::string rule;
    while (std::cin >> rule) {
        uint32_t a = 0, b = 0, c = 0;
        if (rule == "token_merge_shift" && std::cin >> a)
            printf("%u\n", g4::token_merge_shift(a));
        else if (rule == "softmax_scores_per_thread" && std::cin >> a >> b)
            printf("%u\n", g4::softmax_scores_per_thread(a, b));
        else if (rule == "attn_output_chain" && std::cin >> a >> b >> c)
            printf("%d\n", (int)g4::attn_output_chain(a, b, c));
        else if (rule == "argmax_small" && std::cin >> a)
            printf("%d\n", (int)g4::argmax_small(a));
        else
            return fprintf(stderr, "unknown rule %s\n", rule.c_str()), 1;
    }
    return 0;
}
