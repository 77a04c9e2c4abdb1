// The dispatch rules of homelab_amd/csrc/dispatch.hpp as a program: one query a line on stdin,
// one answer a line.
//   tiled N K w_off s_off n_experts max_n exact  ->  rows | wide | narrow | rows+wide | rows+narrow
//   counted N K wide exact max_n n_experts n..   ->  rows | tiles (n: each expert's assignments)
//   step T E k hidden inter                      ->  step | staged
//   attn kv_len heads kv_heads ws_bytes (-1: all) ->  pairs of tiles a wave
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
            std::cout << (r.rows ? "rows" : "") << (r.rows && r.tiles ? "+" : "")
                      << (!r.tiles ? "" : r.wide ? "wide" : "narrow") << "\n";
        } else if (what == "counted") {
            int64_t n, k, m;
            int e, t16 = 0;
            bool wide, exact;
            std::cin >> n >> k >> wide >> exact >> m >> e;
            const oom::TiledGrid g = oom::tiled_grid(n, m, wide);
            oom::XcdBlocks blocks;
            for (int i = 0; i < e; i++) {
                int64_t c;
                std::cin >> c;
                t16 += (int)oom::cdiv(c, oom::NR_M);
                blocks.add((uint32_t)g.nx * g.ny * i, g.nx * (int32_t)oom::cdiv(c, g.rows));
            }
            std::cout << (oom::tiled_cost(n, k, wide, exact).rows_faster(t16, blocks) ? "rows" : "tiles") << "\n";
        } else if (what == "step") {
            int t, e, k;
            int64_t h, i;
            std::cin >> t >> e >> k >> h >> i;
            std::cout << (oom::gate_up_step_ok(t, e, k, h, i) ? "step" : "staged") << "\n";
        } else if (what == "attn") {
            int n, h, hk;
            int64_t ws;
            std::cin >> n >> h >> hk >> ws;
            std::cout << oom::attn_pairs(n, h, hk, 128, ws < 0 ? oom::attn_ws(n, hk, 128).total : (size_t)ws) << "\n";
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
