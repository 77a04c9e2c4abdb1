// Which kernel or split a call takes: the host rules of the entry points that have more than
// one, as functions of sizes alone. No HIP here, so that a CPU test compiles them by themselves
// (tests/dispatch_rules.cpp).
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>

#ifdef __HIPCC__
#define OOM_HD __host__ __device__  // the device asks some of it too
#else
#define OOM_HD
#endif

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
    s.st = 2 * (int)cdiv(K, (int64_t)64 << s.ks_log);
    if (s.st < 6) s.st = 6;
    return s;
}
// Batches of weight rows that a projection of N rows has.
inline int rows_batches(int64_t N, const RowsSplit& sp) {
    return (int)cdiv(N, 16 * NR_BATCH * (NR_WAVES >> sp.ks_log));
}

// The tiles kernel of a shape: wide tiles where the weights can go straight into registers
// (records' parts are 16-byte aligned in the released layout).
inline bool tiled_wide(int64_t K, int64_t w_off, int64_t s_off) {
    return K % TW_BK == 0 && w_off % 16 == 0 && s_off % 2 == 0;
}

// What the few-row kernel can serve at all: K in whole scale groups a lane and at most 8 slices
// of 10 steps.
inline bool rows_kernel_serves(int64_t N, int64_t K, int64_t w_off, int64_t s_off, int64_t n_experts, int64_t max_n) {
    return K % 64 == 0 && K <= NR_MAXK && w_off % 4 == 0 && s_off % 4 == 0 &&
           n_experts * cdiv(max_n, NR_M) * rows_batches(N, rows_split(K)) <= INT32_MAX / 8;
}

// Blocks that each XCD gets: workgroup i of a launch runs on XCD i % 8.
struct XcdBlocks {
    int32_t on[8] = {};
    // `times` runs of n workgroups from workgroup `first` on
    OOM_HD void add(uint32_t first, int32_t n, int32_t times = 1) {
        for (uint32_t i = 0; i < 8; i++) on[i] += times * (n / 8 + (((i - first) & 7) < (uint32_t)n % 8 ? 1 : 0));
    }
};

// The tiles kernel's launch: workgroup x + nx (y + ny e) is N tile x, assignment tile y of expert e,
// and ends at once where expert e has no such tile.
struct TiledGrid {
    int32_t nx, ny, rows;  // rows: assignments a tile
};
inline TiledGrid tiled_grid(int64_t N, int64_t max_n, bool wide) {
    const int32_t bn = wide ? TW_BN : T4_BN, bm = wide ? TW_BM : T4_BM;
    return {(int32_t)cdiv(N, bn), (int32_t)cdiv(max_n, bm), bm};
}

// What a projection takes by either kernel, in ns, by what its experts' assignments make of it.
// The few-row kernel's blocks take equal runs of its batches, t16 tiles of 16 times the batches of N:
// a time a batch of the longest run, one a tile that the run touches (its activations load anew), one
// a batch that the chip has in hand on average. The tiles take one a round, of one block a CU on the
// busiest XCD (wide) or of blocks in flight together (narrow), one a block on average, and one a
// call. In whole numbers, so that every place that asks gets one answer. Fitted to 17000 calls (N 256
// to 4096, K 320 to 2560, 2 to 512 experts, 1 to 900 rows an expert, even and skewed): nine tenths of
// the few-row kernel's are within 11 % of what they took, of the wide tiles' within 18 %.
struct TiledCost {
    int32_t start, batch, tile, flow, batches;  // few-row kernel
    int32_t once, round, block;                 // tiles
    bool wide;
    OOM_HD int64_t rows_ns(int32_t t16) const {
        const int64_t all = (int64_t)t16 * batches;
        const int32_t run = all > 256 ? (int32_t)((all + 255) >> 8) : 1;
        return start + (int64_t)batch * run + (int64_t)tile * (1 + (run + batches - 2) / batches) + (flow * all >> 8);
    }
    OOM_HD int64_t tiles_ns(const XcdBlocks& blocks) const {
        int32_t most = 0;
        int64_t all = 0;
        for (int i = 0; i < 8; i++) {
            all += blocks.on[i];
            most = blocks.on[i] > most ? blocks.on[i] : most;
        }
        const int64_t rounds = wide ? (most + 31) / 32 * 32 : most > 32 ? most : 32;
        return once + (round * rounds >> 5) + (block * all >> 8);
    }
    // (a twentieth of difference goes to the few-row kernel: skewed picks are the worse to get wrong)
    OOM_HD bool rows_faster(int32_t t16, const XcdBlocks& blocks) const {
        return 20 * rows_ns(t16) <= 21 * tiles_ns(blocks);
    }
};
inline TiledCost tiled_cost(int64_t N, int64_t K, bool wide, bool exact) {
    const RowsSplit sp = rows_split(K);
    const int32_t rows[2][3][4] = {{{4099, 2176, 4154, 3143}, {4423, 2311, 5144, 4224}, {4820, 3100, 6205, 5329}},
                                   {{4213, 3205, 4274, 3379}, {4704, 3626, 5173, 4437}, {6674, 4960, 7362, 5524}}};
    const int32_t* const r = rows[exact][sp.st == 6 ? 0 : sp.st == 8 ? 1 : 2];
    const int32_t k = (int32_t)K;
    TiledCost c;
    c.start = r[0], c.batch = r[1], c.tile = r[2], c.flow = r[3];
    c.batches = rows_batches(N, sp);
    c.wide = wide;
    if (wide) {  // waves past N are idle: a part of a round goes with the rows there are
        const int32_t full = (int32_t)(k * N / (TW_BN * cdiv(N, TW_BN)));
        c.once = exact ? -228 * k / 100 : -126 * k / 100;
        c.round = exact ? 4825 + (2836 * k + 777 * full) / 100 : 3613 + (1348 * k + 1137 * full) / 100;
        c.block = exact ? 753 * k / 100 : 817 * k / 100;
    } else {
        c.once = exact ? 984 * k / 100 : 567 * k / 100;
        c.round = exact ? 557 + 1105 * k / 100 : std::max(0, 899 * k / 100 - 672);
        c.block = exact ? 452 * k / 100 : 592 * k / 100;
    }
    return c;
}

// The kernels that a call launches: the few-row kernel (rows), the tiles (wide or narrow), or both,
// which then count the assignments on the device: one of them works, the other returns at once.
struct TiledRoute {
    bool rows, tiles, wide;
};

// The host knows the largest expert only. Evenly spread picks reach it with most experts near it,
// and then the tiles are the faster ones, up to twice, once experts fill them (us a projection,
// exact, few-row kernel and tiles: 640 x 2560, 64 experts, 320 rows each, 295 and 251; 2560 x 640,
// 32 experts, 75 rows each, 60 and 36). Skewed picks reach it with most experts far below, and the
// few-row kernel is the faster one, up to three times: the tiles pad to 48 or 64, and the experts'
// first tiles alone can fall on half of the XCDs. So: the few-row kernel where it is the faster one
// of evenly spread picks, the tiles where they are with every expert but one in a single tile, both
// between the two. The second launch and the counting cost 3.3 us and 1 us a round of tiles, so a
// call whose tiles take less than TR_COUNT_NS takes them alone, as does one with more experts than a
// block counts in a few loads, or with sums past 2^24 (the device's are f32). On average over the
// calls above this takes 1.02 of the faster kernel's time for evenly spread picks and 1.03 to 1.05
// for skewed ones; the few-row kernel wherever N and K fill its slices took 1.06 and 1.06 to 1.09.
constexpr int64_t TR_COUNT_NS = 50000;
constexpr int TR_COUNT_E = 2048;
inline TiledRoute tiled_route(int64_t N, int64_t K, int64_t w_off, int64_t s_off, int64_t n_experts, int64_t max_n,
                              bool exact) {
    const bool wide = tiled_wide(K, w_off, s_off);
    if (!rows_kernel_serves(N, K, w_off, s_off, n_experts, max_n)) return {false, true, wide};
    const TiledGrid grid = tiled_grid(N, max_n, wide);
    const TiledCost cost = tiled_cost(N, K, wide, exact);
    // the blocks if each expert has `lo` tiles and `hi` of them one more, both spread evenly
    const auto blocks = [&](int64_t lo, int64_t hi) {
        XcdBlocks b;
        for (int j = 0; j < 8; j++) {  // the experts e with e % 8 == j start on one XCD
            const int64_t n = (n_experts + 7 - j) / 8, m = std::min(n, (hi + 7 - j) / 8);
            const uint32_t first = (uint32_t)grid.nx * grid.ny * j;
            b.add(first, (int32_t)(grid.nx * lo), (int32_t)n);
            b.add(first + (uint32_t)(grid.nx * lo), grid.nx, (int32_t)m);
        }
        return b;
    };
    // mean rows of evenly spread picks whose largest expert has max_n: sqrt(2 mean ln E) below it
    const double spread = 2.0 * std::log((double)std::max<int64_t>(n_experts, 2));
    const double root = (std::sqrt(spread + 4.0 * (double)max_n) - std::sqrt(spread)) / 2.0;
    const double mean = std::max(1.0, root * root);
    const auto tiles = [&](int64_t m) {
        return std::min(n_experts * cdiv(max_n, m), (int64_t)((double)n_experts * std::max(1.0, mean / (double)m + 0.5)));
    };
    const int64_t t16 = tiles(NR_M), tn = tiles(grid.rows);
    const XcdBlocks even = blocks(tn / n_experts, tn % n_experts);
    if (cost.rows_faster((int32_t)t16, even)) return {true, false, wide};
    XcdBlocks skewed = blocks(1, 0);
    skewed.add(0, grid.nx * (grid.ny - 1));
    const int64_t sums = n_experts * std::max(cdiv(max_n, NR_M), (int64_t)grid.nx * grid.ny);
    if (n_experts > TR_COUNT_E || sums >= 1 << 24 || cost.tiles_ns(even) < TR_COUNT_NS ||
        !cost.rows_faster((int32_t)(cdiv(max_n, NR_M) + n_experts - 1), skewed))
        return {false, true, wide};
    return {true, true, wide};
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
// Skewed picks reach fewer experts, so the lines lie above where even ones break even: over 420
// random steps (215 of even picks, 110 and 95 of popularity falling with rank to the 0.5 and 1.1) this
// takes 0.989, 0.997 and 1.000 of the staged time; lines at the break-even 0.990, 1.001 and 1.002, with
// 34 steps more than 2 % slower in place of 11.
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
    if (hidden <= 1024) return items >= (per <= 1.15 ? 7.0 : 10.0);
    return items >= (hidden <= 2048 ? 5.0 : per <= 1.1 ? 2.9 : 4.0);
}

// ---- oom_attn_decode_paged (attention.hip) --------------------------------------------------

constexpr int AKB = 1024;  // keys a block of the coarsest split
constexpr int AG = 8;      // query heads per KV head (at most)

// Splits of a KV head's keys: blocks of 4 waves with 32 NP keys a wave, NP = 1, 2, 4 or 8
// pairs of tiles. One wave's pairs follow each other (about 1.4 us each: one pair is in
// flight), so the finest split that still fits the chip is the fastest: at 64 / 8 heads, us a
// step, NP = 1, 2, 4, 8 by keys
//     1000:  8.0,  9.1, 12.1, 15.3      4096:  9.7, 10.0, 12.5, 18.7
//     8192: 13.3, 12.1, 13.2, 18.7     16384: 17.9, 17.4, 16.6, 19.4
//    32768: 49.1, 31.9, 30.5, 29.5     65536: 90.9, 70.9, 54.5, 54.2
// so NP is the smallest whose blocks number at most A_FILL over all KV heads (one a CU; the
// rows' best ends there: 4096 keys are 256 blocks at NP = 1, 8192 at NP = 2, 16384 at NP = 4)
// and whose partials a KV head the merge takes in one round (at 1 KV head and 32768 keys, 256
// partials: 25.3 us against 10.8 for 128 at NP = 2). Up to 256 keys one block holds the KV
// head and no merge is launched (200 keys: 5.9 us at NP = 2 against 7.9 at NP = 1 and 13.7 at
// NP = 8). The merge costs more the more query heads there are, one block a KV head does not, so
// many of them take one block up to 1024 keys as well: NP = 4 up to 512 keys (400 keys, 8 query
// heads a KV head, this against the finest split: 9.0 and 8.2 us at 256 query heads, 9.0 and 10.5
// at 384, 9.6 and 18.0 at 1024), NP = 8 past that in place of two blocks (1000 keys: 15.8 and 17.4
// at 640, 16.3 and 23.7 at 1024; with 4 a KV head 16.0 and 16.3 at 400, 16.4 and 19.5 at 512).
constexpr int A_FILL = 256;       // blocks over all KV heads
constexpr int A_ROUND = 128;      // partials a KV head the merge loads at once
constexpr int A_ONE_512 = 320;    // query heads that take one block up to 512 keys,
constexpr int A_ONE_1024 = 512;   // and in place of two up to 1024

struct AttnWs {
    size_t least, total;  // what the coarsest split needs, and what every split at up to kv_len keys fits in
};

inline size_t attn_part_bytes(int blocks, int kv_heads, int d) {
    return ((size_t)kv_heads * blocks * (2 * AG + AG * (size_t)d) * sizeof(float) + 255) & ~size_t(255);
}

// A sequence that grows within one workspace: the finer splits of shorter sequences take at
// most min(A_ROUND, A_FILL / kv_heads) blocks a KV head, so `total` never falls with kv_len.
inline AttnWs attn_ws(int kv_len, int kv_heads, int d) {
    AttnWs w;
    const int coarse = (int)cdiv(kv_len, AKB);
    const int fine = std::min((int)cdiv(kv_len, 128), std::min(A_ROUND, A_FILL / kv_heads));
    w.least = attn_part_bytes(coarse, kv_heads, d);
    w.total = attn_part_bytes(std::max(coarse, fine), kv_heads, d);
    return w;
}

// Pairs of tiles a wave (NP): the rule above, within the workspace at hand (one sized for the
// coarsest split alone still serves).
inline int attn_pairs(int kv_len, int heads, int kv_heads, int d, size_t ws_bytes) {
    if (kv_len > 256 && kv_len <= 512 && heads >= A_ONE_512) return 4;
    for (int np = kv_len <= 128 ? 1 : kv_len <= 256 ? 2 : 1; np < 8; np *= 2) {
        const int64_t blocks = cdiv(kv_len, 128 * np);
        if (np == 4 && blocks == 2 && heads >= A_ONE_1024) break;
        if (blocks == 1 || (blocks <= A_ROUND && blocks * kv_heads <= A_FILL &&
                            attn_part_bytes((int)blocks, kv_heads, d) <= ws_bytes))
            return np;
    }
    return 8;
}

// ---- oom_attn_decode_turbo (turbo.hip) ------------------------------------------------------

// How a KV head's keys are dealt: blocks of `waves` waves, `blocks` of them a KV head. A wave's
// groups follow each other (about 4 us each: 128 fp32 MFMAs and the decoding between them), so
// every wave takes one group as long as the grid then has a block a CU or fewer:
//   - blocks of 4 waves, one a SIMD, while ceil(groups / 4) blocks a KV head make at most
//     TT_FILL in all; past that some CUs have a second round of them (a wave's 340 registers leave
//     a SIMD no room for another; 9001 keys, 2 KV heads, us a call with the combine: 27.7 as 282
//     blocks of 4 waves, 18.7 as 142 of 8);
//   - else blocks of 8 waves, at most TT_FILL in all, their waves taking more groups from there;
//   - fp32 rows (no decoding for a second wave's MFMAs to hide behind) keep 4 waves up to two
//     groups a wave (17.0 us against 19.4 at 9001 keys, 2 KV heads), and two groups a wave on
//     blocks of 8 past that: half the blocks, and partials to combine, of one group a wave (2 KV
//     heads, 16500 keys: 31.1 us against 35.1; 28000: 34.4 and 35.9).
// Before, every wave was sized for two groups on blocks of 8: us a call then and now, k8v6, all
// keys visible, 2 KV heads: 24.4 -> 15.5 at 700 keys, 24.5 -> 16.1 at 4500, 24.7 -> 18.7 at
// 9001, 24.8 -> 19.8 at 16384, 26.2 at 32768 (the same split).
constexpr int TT_FILL = 256;

struct TurboSplit {
    int waves, blocks;
};

// Two groups a wave on blocks of 8 waves: the fewest partials, also for a workspace with room for
// no more.
inline TurboSplit turbo_split_least(int kv_len, int kv_heads) {
    const int groups = (kv_len + 15) / 16;
    return {8, std::max(1, std::min((groups + 15) / 16, std::max(1, TT_FILL / kv_heads)))};
}

inline TurboSplit turbo_split(int kv_len, int kv_heads, bool fp32) {
    const int groups = (kv_len + 15) / 16, most = std::max(1, TT_FILL / kv_heads);
    for (int per = 4; per <= (fp32 ? 8 : 4); per += 4)
        if ((groups + per - 1) / per <= most) return {4, (groups + per - 1) / per};
    if (fp32) return turbo_split_least(kv_len, kv_heads);
    return {8, std::min((groups + 7) / 8, most)};
}

}  // namespace oom
