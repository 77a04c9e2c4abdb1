"""The host rules that pick a kernel or a split (homelab_amd/csrc/dispatch.hpp), on the CPU."""
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
