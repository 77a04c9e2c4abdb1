// Which kernel or split a call takes: the host rules of the entry points that have more than
// one, as functions of sizes alone. No HIP here, so that a CPU test compiles them by themselves
// (tests/dispatch_rules.cpp).
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>

namespace oom {

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- oom_moe_tiled_nvfp4 (nvfp4_tiled.hip, nvfp4_rows.hpp) -------------------------------

constexpr int T4_BN = 128;  // 128-row tiles: weight rows a block,
constexpr int T4_BM = 64;   // assignments a block
constexpr int T4_BK = 32;   // and the K step

constexpr int TW_BN = 640;  // wide tiles
constexpr int TW_BM = 48;
constexpr int TW_BK = 128;

constexpr int NR_WAVES = 8;    // few-row kernel: waves a block,
constexpr int NR_BATCH = 8;    // 16-row subtiles a wave between two meetings of the slices,
constexpr int NR_MAXK = 2560;  // 8 slices of 10 steps: 120 registers of activation terms,
constexpr int NR_M = 16;       // and activation rows

// How the few-row kernel splits K: KS = 1 << ks_log slices of 32 ST columns, the other waves on
// other weight rows.
struct RowsSplit {
    int ks_log, st;
};
inline RowsSplit rows_split(int64_t K) {
    RowsSplit s{0, 10};
    while (s.ks_log < 3 && K > (int64_t)320 << s.ks_log) s.ks_log++;
    s.st = std::max(6, 2 * (int)cdiv(K, (int64_t)64 << s.ks_log));
    return s;
}
// Batches of weight rows that a projection of N rows has.
inline int rows_batches(int64_t N, const RowsSplit& sp) {
    return (int)cdiv(N, 16 * NR_BATCH * (NR_WAVES >> sp.ks_log));
}

// Where the rows kernel is the better one: K in whole scale groups a lane and at most 8 slices
// of 10 steps, and either slices and batches that K and N fill (five sixths at least) or tiles
// of so few rows that the stream counts and not the steps. Us a call of gate, up, SwiGLU, down
// and combine at 2560 / 640, exact, rows kernel and tiles: 512 experts top-10, 60 tokens 287
// and 601, 250 398 and 698, 500 451 and 722, 900 664 and 761, 1050 766 and 782, 1400 924 and
// 1224, 2048 1218 and 1472; 64 experts, 300 tokens 228 and 296, 1200 612 and 626. At 1600 / 448
// (slices 78 % and 88 % full) 128 experts top-4, 600 tokens 151 and 185, but 64 experts top-10,
// 1200 tokens (190 rows an expert) 398 and 327. The tiles also keep the steps of many experts
// whose 41 to 48 rows at most are one 48-row tile where the rows kernel decodes twice or more
// (512 experts, 1200 tokens: 815 and 786; with 128 experts 264 and 299).
inline bool rows_kernel_serves(int64_t N, int64_t K, int64_t w_off, int64_t s_off, int64_t n_experts, int64_t max_n,
                               bool exact) {
    if (K % 64 != 0 || K > NR_MAXK || w_off % 4 != 0 || s_off % 4 != 0) return false;
    const RowsSplit sp = rows_split(K);
    if (n_experts * cdiv(max_n, NR_M) * rows_batches(N, sp) > INT32_MAX) return false;
    if (exact && K % TW_BK == 0 && n_experts >= 384 && max_n > 40 && max_n <= TW_BM) return false;
    const int64_t rows = (int64_t)16 * NR_BATCH * (NR_WAVES >> sp.ks_log) * rows_batches(N, sp);
    return 6 * K * N >= 5 * ((int64_t)32 * sp.st << sp.ks_log) * rows || max_n <= 48;
}

enum class TiledRoute { rows, wide, narrow };

// The kernel of a projection of N rows of K inputs over n_experts experts of at most max_n
// assignments.
inline TiledRoute tiled_route(int64_t N, int64_t K, int64_t w_off, int64_t s_off, int64_t n_experts, int64_t max_n,
                              bool exact) {
    if (rows_kernel_serves(N, K, w_off, s_off, n_experts, max_n, exact)) return TiledRoute::rows;
    // weights straight into registers (records' parts are 16-byte aligned in the released layout)
    return K % TW_BK == 0 && w_off % 16 == 0 && s_off % 2 == 0 ? TiledRoute::wide : TiledRoute::narrow;
}

// ---- oom_moe_decode_nvfp4, several tokens (nvfp4.hip) -------------------------------------

constexpr int N4S_AMAX = 512;            // assignments of a step (and so routed experts)
constexpr int64_t N4S_XMAX = 144 * 1024; // of LDS for the tokens' x, beside the plan's 12 KiB

// Whether a step's gate/up runs as free-running waves over all its tokens' x, instead of staged
// per expert (the same bits). The plan and x fit LDS; at most three chunks of 1024 columns: with
// four the two rounds of loads in flight spill 79 registers (512 experts top-10, 4096 / 1536: 64
// us staged and 94 at 2 tokens, 243 and 325 at 8; 128 top-8, 4096 / 768: 104 and 142 at 8).
// And rows enough: every block stages all of x before its first sums, a wave's last round of
// items leaves others idle, and a row is decoded once an assignment where the staged launch
// decodes it once for two. So the rule is on the items a wave, of four rows of a routed expert,
// with the experts that evenly spread picks reach. Us a step, staged and this, by items a wave
// and assignments an expert:
//   three chunks (2560 / 640): 1.2, 2.1: 33.6, 36.7 (4 tokens, 16 experts top-8); 1.55, 1.0: 33.9,
//     35.1 (2, 512 top-10); 3.3, 1.5: 57.8, 58.8 (8, 64 top-8); 3.0, 1.0: 53.3, 48.9 (4, 512
//     top-10); 3.7, 1.7: 66.6, 65.7 (8, 64 top-10); 5.8, 1.1: 92.9, 82.6 (8, 512 top-10)
//   two (2048 / 1024): 1.7, 1.1: 27.5, 28.6; 2.7, 1.5: 35.9, 36.9; 3.9, 3.1: 67.4, 69.6; 4.4, 1.4:
//     47.8, 46.0; 6.3, 1.9: 84.2, 78.5; 10.3, 1.6: 118, 103
//   one (1024 / 512), where the decoding weighs most: 2.0, 6.0: 57.3, 61.5; 4.0, 4.1: 67.6, 72.2;
//     5.2, 1.6: 50.9, 50.9; 7.0, 2.3: 69.9, 74.0; 8.7, 1.2: 70.1, 66.6; 15, 1.3: 115, 108
constexpr int64_t N4S_MAX_H = 3072;
constexpr int N4S_WAVES = 8;    // waves a block, on one block a CU
constexpr int N4S_GRID = 256;
constexpr int N4S_ROWS = 4;     // gate (and up) rows an item
inline int64_t gate_up_step_lds(int T, int64_t hidden) {
    return (T + 1) / 2 * 2 * cdiv(hidden, 1024) * 4096;  // staged two rows at a time
}
inline bool gate_up_step_ok(int T, int E, int k, int64_t hidden, int64_t inter) {
    const int64_t A = (int64_t)T * k;
    if (A > N4S_AMAX || hidden > N4S_MAX_H || gate_up_step_lds(T, hidden) > N4S_XMAX) return false;
    const double experts = E * (1.0 - std::pow(1.0 - (double)k / E, T));
    const double items = experts * (double)cdiv(inter, N4S_ROWS) / (N4S_GRID * N4S_WAVES), per = A / experts;
    if (hidden <= 1024) return items >= (per <= 1.75 ? 5.0 : 8.0);
    return items >= (per <= 1.1 ? 2.9 : hidden <= 2048 ? 4.0 : 3.5);
}

// ---- oom_attn_decode_turbo (turbo.hip) ------------------------------------------------------

// How a KV head's keys are dealt: blocks of `waves` waves, `blocks` of them a KV head. A wave's
// groups follow each other (about 4 us each: 128 fp32 MFMAs and the decoding between them), so
// every wave takes one group as long as the grid then has a block a CU or fewer:
//   - blocks of 4 waves, one a SIMD, while ceil(groups / 4) blocks a KV head make at most
//     TT_FILL in all; past that two of them share a CU (9001 keys, 2 KV heads, us a call with
//     the combine: 27.7 as 282 blocks of 4 waves, 18.7 as 142 of 8);
//   - else blocks of 8 waves, at most TT_FILL in all, their waves taking more groups from there;
//   - fp32 rows (no decoding for a second wave's MFMAs to hide behind) keep 4 waves up to two
//     groups a wave: 17.0 us against 19.4 at 9001 keys, 2 KV heads.
// Before, every wave was sized for two groups on blocks of 8: us a call then and now, k8v6, all
// keys visible, 2 KV heads: 24.4 -> 15.5 at 700 keys, 24.5 -> 16.1 at 4500, 24.7 -> 18.7 at
// 9001, 24.8 -> 19.8 at 16384, 26.2 at 32768 (the same split).
constexpr int TT_FILL = 256;

struct TurboSplit {
    int waves, blocks;
};

inline TurboSplit turbo_split(int kv_len, int kv_heads, bool fp32) {
    const int groups = (kv_len + 15) / 16, most = std::max(1, TT_FILL / kv_heads);
    for (int per = 4; per <= (fp32 ? 8 : 4); per += 4)
        if ((groups + per - 1) / per <= most) return {4, (groups + per - 1) / per};
    return {8, std::min((groups + 7) / 8, most)};
}

// Two groups a wave on blocks of 8 waves: the fewest partials, for a workspace with room for
// no more.
inline TurboSplit turbo_split_least(int kv_len, int kv_heads) {
    const int groups = (kv_len + 15) / 16;
    return {8, std::max(1, std::min((groups + 15) / 16, std::max(1, TT_FILL / kv_heads)))};
}

}  // namespace oom
