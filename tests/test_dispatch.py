"""The host rules that pick a kernel or a split (homelab_amd/csrc/dispatch.hpp), on the CPU."""
import numpy as np
import pytest

import dispatch


@pytest.mark.parametrize("n,k,w_off,s_off,e,max_n,exact,want", [
    (640, 2560, 256, 819456, 512, 20, True, "rows"),   # the released record's gate, ten rows an expert
    (2560, 640, 256, 819456, 512, 20, False, "rows"),  # and its down
    (640, 4096, 256, 819456, 512, 20, True, "wide"),   # K past eight slices of ten steps
    (640, 2592, 256, 819456, 512, 20, True, "narrow"),  # K no whole K block
    (640, 2560, 258, 819456, 512, 20, True, "narrow"),  # codes at 2 bytes of alignment
    (640, 2560, 260, 819456, 512, 20, True, "rows"),
])
def test_tiled_route(n, k, w_off, s_off, e, max_n, exact, want):
    assert dispatch.tiled(n, k, w_off, s_off, e, max_n, exact) == want


# us a call of the few-row kernel and of the tiles it replaced, by the sizes that the host knows (n,
# k, experts, assignments of the largest) for evenly spread picks of T tokens
@pytest.mark.parametrize("n,k,e,max_n,exact,rows_us,tiles_us,want", [
    (640, 2560, 64, 24, True, 40, 92, "rows"),       # 100 tokens top-10
    (640, 2560, 128, 121, True, 185, 220, "rows"),   # 1200
    (640, 2560, 512, 62, True, 368, 475, "rows"),    # 2048: the experts' first tiles fall on four XCDs
    (704, 1152, 128, 13, False, 22, 30, "rows"),     # 68, one term: a round of tiles on every CU
    (2560, 640, 32, 33, True, 40, 28, "wide"),       # 100 top-8: one round of short tiles
    (2560, 640, 32, 86, True, 60, 36, "wide"),       # 300
    (2560, 640, 32, 168, False, 81, 44, "wide"),     # 600, one term
    (1024, 512, 64, 121, False, 46, 40, "wide"),     # 600
    (640, 2560, 64, 375, True, 295, 251, "rows+wide"),   # 2048 top-10
    (2560, 640, 64, 375, True, 311, 252, "rows+wide"),
    (2560, 640, 64, 682, False, 482, 328, "rows+wide"),  # 4096, one term
    (640, 2560, 512, 108, True, 679, 594, "rows+wide"),  # 4096
    (448, 1600, 64, 682, True, 380, 287, "rows+narrow"),
    (1600, 448, 128, 63, True, 73, 54, "rows+narrow"),
])
def test_tiled_route_of_even_picks(n, k, e, max_n, exact, rows_us, tiles_us, want):
    """The few-row kernel alone only where it is not the slower one; where both are launched the
    device's count takes the faster one of these calls too."""
    got = dispatch.tiled(n, k, 256, 1 << 20, e, max_n, exact)
    assert got == want
    assert got != "rows" or rows_us <= tiles_us
    if "+" in got:
        mean = int(max_n - (2 * max_n * np.log(e)) ** 0.5)
        assert dispatch.counted(n, k, k % 128 == 0, exact, [max_n] + [mean] * (e - 1)) == "tiles"


@pytest.mark.parametrize("n,k,exact,counts,want", [
    # the largest expert alone does not decide: the others' few rows stay with the few-row kernel
    (640, 2560, True, [375] + [20] * 63, "rows"),
    (2560, 640, True, [1200] + [12] * 511, "rows"),
    (640, 2560, False, [45] + [10] * 511, "rows"),
    (448, 1600, True, [2000] + [9] * 63, "rows"),
    (640, 2560, True, [320] * 64, "tiles"),
    (640, 2560, False, [80] * 512, "tiles"),
    (640, 2560, True, [900] * 16 + [3] * 16, "tiles"),
    (448, 1600, True, [640] * 64, "tiles"),
    # one tile an expert on even planes: all of them on four XCDs, two rounds where there is room for one
    (640, 2560, True, [40, 0] * 256, "rows"),
    (640, 2560, True, [40] * 256, "tiles"),
])
def test_tiled_counts(n, k, exact, counts, want):
    assert dispatch.counted(n, k, k % 128 == 0, exact, counts, max(counts)) == want


def test_tiled_counted_sums_are_exact():
    """Both kernels only where every sum of the device's count is a whole number below 2^24."""
    for e in (4, 300, 2048, 2049, 20000):
        for max_n in (100, 5000, 200000, 3000000):
            for n, k in ((640, 2560), (448, 1600), (20480, 2560), (65536, 320)):
                if "+" in dispatch.tiled(n, k, 256, 1 << 20, e, max_n, True):
                    wide = k % 128 == 0
                    planes = -(-n // (640 if wide else 128)) * -(-max_n // (48 if wide else 64))
                    assert e * max(-(-max_n // 16), planes) < 1 << 24 and e <= 2048


@pytest.mark.parametrize("T,E,k,hidden,inter,want", [
    (8, 512, 10, 2560, 640, "step"),
    (8, 512, 10, 3072, 1024, "step"),
    # past three chunks of 1024 the kernel's two rounds of loads spill
    (2, 512, 10, 4096, 1536, "staged"),
    (8, 128, 8, 4096, 768, "staged"),
    (4, 64, 8, 3088, 1536, "staged"),
    # few rounds of items a wave: a step's experts x rows / 4 over 2048 waves
    (2, 512, 10, 2560, 640, "staged"),
    (2, 128, 8, 2560, 640, "staged"),
    (4, 512, 10, 2560, 640, "step"),
    (4, 16, 8, 2560, 640, "staged"),
    # several assignments an expert, which the step decodes a row for each and the staged launch in pairs
    (8, 16, 8, 2560, 640, "staged"),
    (8, 64, 8, 2560, 640, "staged"),
    (24, 128, 8, 1024, 512, "staged"),
    (32, 64, 8, 1024, 512, "staged"),
    (32, 512, 10, 1024, 512, "step"),
    (16, 128, 8, 2048, 1536, "step"),
    (16, 64, 8, 2048, 1536, "step"),
    # near the break-even of even picks, where skewed ones lose
    (17, 256, 8, 1168, 336, "staged"),
    (18, 64, 8, 1184, 656, "staged"),
    (19, 256, 8, 880, 464, "staged"),
    (9, 128, 8, 2240, 544, "staged"),
    # past the plan's 512 slots; x past its LDS
    (33, 128, 16, 1008, 304, "staged"),
    (13, 512, 10, 2560, 640, "staged"),
    (12, 512, 10, 2560, 640, "step"),
])
def test_step_route(T, E, k, hidden, inter, want):
    assert dispatch.step(T, E, k, hidden, inter) == want


def test_turbo_split_covers_the_keys():
    """Every split deals every group of 16 keys, on at most 256 blocks over the KV heads, and one
    block a KV head past 256 of them."""
    shapes = [(n, h, f) for n in range(1, 70000, 487) for h in (1, 2, 3, 4, 7, 8, 64, 256, 300) for f in (0, 1)]
    for (n, h, f), ans in zip(shapes, dispatch.ask(*(f"turbo {n} {h} {f}" for n, h, f in shapes))):
        waves, blocks = map(int, ans.split())
        groups = -(-n // 16)
        assert waves in (4, 8) and 1 <= blocks and (blocks == 1 or blocks * h <= 256)
        assert (blocks - 1) * waves < groups, "an empty block"
        assert waves == 8 or blocks * waves * (2 if f else 1) >= groups


@pytest.mark.parametrize("kv_len,kv_heads,fp32,want", [
    (8192, 2, False, "4 128"), (8193, 2, False, "8 65"), (40000, 2, False, "8 128"),
    (8193, 2, True, "4 65"), (16384, 2, True, "4 128"),
    # fp32 rows past two groups a wave of 4: two groups a wave of 8, half the blocks of one group
    (16500, 2, True, "8 65"), (28000, 2, True, "8 110"), (36000, 1, True, "8 141"), (10000, 4, True, "8 40"),
    (65536, 2, True, "8 128"),
])
def test_turbo_split(kv_len, kv_heads, fp32, want):
    assert dispatch.ask(f"turbo {kv_len} {kv_heads} {int(fp32)}") == [want]


@pytest.mark.parametrize("kv_len,heads,kv_heads,want", [
    (100, 64, 8, 1), (200, 64, 8, 2), (700, 64, 8, 1), (4096, 64, 8, 1), (4097, 64, 8, 2), (16384, 64, 8, 4),
    (32768, 64, 8, 8), (16384, 8, 1, 1), (16385, 8, 1, 2), (700, 32, 8, 1), (1000, 128, 128, 4),
    # the merge of many query heads costs more than one block's longer waves
    (257, 1024, 128, 4), (512, 1024, 128, 4), (400, 384, 48, 4), (400, 256, 32, 1), (513, 1024, 128, 8),
    (1000, 1024, 128, 8), (1000, 640, 80, 8), (1000, 512, 128, 8), (1000, 400, 100, 4), (1000, 512, 64, 2),
    (1025, 1024, 128, 8),
])
def test_attn_pairs(kv_len, heads, kv_heads, want):
    assert dispatch.ask(f"attn {kv_len} {heads} {kv_heads} -1") == [str(want)]
