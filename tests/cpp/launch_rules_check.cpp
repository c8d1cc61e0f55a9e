// Prints the launch choices of apbf_amd/csrc/launch_rules.h: one line per
// request "walk n long_rows" "walks" (the walk's lane counts), "few n"
// or "sort cap upper_bound shape_bits keys_below".
#include <cstdio>
#include <cstring>

#include "../../apbf_amd/csrc/launch_rules.h"

int main() {
    char what[16];
    while (std::scanf("%15s", what) == 1) {
        if (!std::strcmp(what, "walk")) {
            unsigned n, long_rows;
            if (std::scanf("%u %u", &n, &long_rows) != 2) return 1;
            std::printf("%d\n", apbf::walk_lanes_for(n, long_rows != 0));
        } else if (!std::strcmp(what, "few")) {
            unsigned n;
            if (std::scanf("%u", &n) != 1) return 1;
            std::printf("%d\n", apbf::solve_few_rows(n) ? 1 : 0);
        } else if (!std::strcmp(what, "sort")) {
            unsigned cap, upper, bits, below;
            if (std::scanf("%u %u %u %u", &cap, &upper, &bits, &below) != 4) return 1;
            const apbf::SortPlan p = apbf::sort_plan(cap, upper, bits, below != 0);
            std::printf("%u %u %d\n", p.bits, p.passes, p.one_block ? 1 : 0);
        } else if (!std::strcmp(what, "walks")) {
            for (int lanes : apbf::WALK_LANES) std::printf("%d ", lanes);
            std::printf("\n");
        } else {
            return 1;
        }
    }
    return 0;
}
