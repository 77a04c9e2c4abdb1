// The dispatch rules of homelab_amd/csrc/dispatch.hpp as a program: one query a line on stdin,
// one answer a line.
//   tiled N K w_off s_off n_experts max_n exact  ->  rows | wide | narrow
//   step T E k hidden inter                      ->  step | staged
//   turbo kv_len kv_heads fp32                   ->  waves blocks
#include <iostream>
#include <string>

#include "../homelab_amd/csrc/dispatch.hpp"

int main() {
    std::string what;
    while (std::cin >> what) {
        if (what == "tiled") {
            int64_t n, k, w, s, e, m;
            bool exact;
            std::cin >> n >> k >> w >> s >> e >> m >> exact;
            const oom::TiledRoute r = oom::tiled_route(n, k, w, s, e, m, exact);
            std::cout << (r == oom::TiledRoute::rows ? "rows" : r == oom::TiledRoute::wide ? "wide" : "narrow") << "\n";
        } else if (what == "step") {
            int t, e, k;
            int64_t h, i;
            std::cin >> t >> e >> k >> h >> i;
            std::cout << (oom::gate_up_step_ok(t, e, k, h, i) ? "step" : "staged") << "\n";
        } else if (what == "turbo") {
            int n, h;
            bool fp32;
            std::cin >> n >> h >> fp32;
            const oom::TurboSplit s = oom::turbo_split(n, h, fp32);
            std::cout << s.waves << " " << s.blocks << "\n";
        } else {
            return 1;
        }
    }
    return 0;
}
