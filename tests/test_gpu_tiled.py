"""GPU parity of the tiled NVFP4 grouped GEMM (oom_moe_tiled_nvfp4) and the SwiGLU range
(oom_moe_swiglu_range) through the C ABI.

Bar, as the reference's own test (crates/oominf-cuda/tests/moe_tiled.rs:176-226): at its
three shapes (partial tiles both ways and an empty expert; gate 640 x 2560 and down
2560 x 640) and both precisions, worst |y - f64| / sum |x w| below 2e-6, where the f64
evaluation takes x exact (OOM_EXPERT_EXACT) or rounded to bf16 (OOM_EXPERT_BF16); and the
same bar against the oracle's restatement. SwiGLU against numpy in f64 within 2 ulp.
"""
import numpy as np
import pytest

import dispatch
import oracle
from tiled_cases import SHAPES, case, f64_eval

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import torch

    import homelab_amd

    homelab_amd.lib()  # raises if the library is missing: no fallback
    torch.cuda.init()
    return homelab_amd


def run_tiled(hip, recs, x, off, rows, precision):
    import torch

    buf = torch.from_numpy(np.stack(recs.recs)).cuda()
    addrs = torch.tensor([buf.data_ptr() + e * recs.stride for e in range(len(recs.recs))], dtype=torch.int64,
                         device="cuda")
    A = int(off[-1])
    y = torch.full((max(A, 1), recs.n), float("nan"), dtype=torch.float32, device="cuda")
    rd = None if rows is None else torch.from_numpy(rows).cuda()
    max_n = int(np.diff(off).max())
    hip.moe_tiled_nvfp4(addrs, torch.from_numpy(off).cuda(), rd, len(recs.recs), max_n, torch.from_numpy(x).cuda(), y,
                        recs.n, recs.k, recs.w_off, recs.s_off, 0, precision)
    torch.cuda.synchronize()
    return y.cpu().numpy()[:A]


@pytest.mark.parametrize("n,k,counts", SHAPES)
@pytest.mark.parametrize("exact", [True, False])
def test_tiled_matches_f64_and_oracle(hip, n, k, counts, exact):
    print(f"case: moe_tiled_nvfp4 n={n} k={k} counts={counts} exact={exact}", flush=True)
    recs, x, off, rows = case(n, k, counts, seed=n * 31 + k)
    prec = hip.EXPERT_EXACT if exact else hip.EXPERT_BF16
    got = run_tiled(hip, recs, x, off, rows, prec)
    ref, mag = f64_eval(recs, x, off, rows, exact)
    tiny = np.finfo(np.float64).tiny
    worst = (np.abs(got - ref) / np.maximum(mag, tiny)).max()
    assert worst < 2e-6, f"worst error / sum|x*w| = {worst:.3e}"
    want = oracle.moe_tiled_nvfp4(recs.recs, off, rows, x, n, k, recs.w_off, recs.s_off, 0, 3 if exact else 1)
    assert (np.abs(got - want) / np.maximum(mag, tiny)).max() < 2e-6
    # a second call gives the same bits
    np.testing.assert_array_equal(run_tiled(hip, recs, x, off, rows, prec), got)


def test_tiled_without_rows(hip):
    recs, x, off, _ = case(136, 64, [7, 0, 12], seed=3, tokens=19)
    got = run_tiled(hip, recs, x, off, None, hip.EXPERT_EXACT)
    ref, mag = f64_eval(recs, x, off, np.arange(19, dtype=np.int32), True)
    assert (np.abs(got - ref) / mag).max() < 2e-6


def test_tiled_rejects_bad_arguments(hip):
    import torch

    z = torch.zeros(64, dtype=torch.float32, device="cuda")
    i = torch.zeros(4, dtype=torch.int32, device="cuda")
    with pytest.raises(hip.OomError, match="multiple of 32"):
        hip.moe_tiled_nvfp4(i, i, None, 1, 4, z, z, 16, 48, 64, 0, 0)
    with pytest.raises(hip.OomError, match="precision"):
        hip.moe_tiled_nvfp4(i, i, None, 1, 4, z, z, 16, 64, 64, 0, 0, precision=7)


def test_swiglu_range(hip):
    import torch

    rng = np.random.default_rng(4)
    g = (rng.standard_normal(10007) * 6).astype(np.float32)
    u = rng.standard_normal(10007).astype(np.float32)
    h = torch.full((10007,), -9.0, dtype=torch.float32, device="cuda")
    hip.moe_swiglu_range(torch.from_numpy(g).cuda(), torch.from_numpy(u).cuda(), h, 13, 9001)
    torch.cuda.synchronize()
    got = h.cpu().numpy()
    want = (g.astype(np.float64) / (1.0 + np.exp(-g.astype(np.float64)))) * u
    assert np.all(got[:13] == -9.0) and np.all(got[9001:] == -9.0)
    np.testing.assert_allclose(got[13:9001], want[13:9001], rtol=4e-7, atol=1e-30)


@pytest.mark.parametrize("n,k,counts,route", [
    (1024, 128, [1, 0, 2] * 200, "rows"),    # one slice, fewer columns than its 6 steps; more experts than threads
    (1020, 192, [3, 0, 2] * 100, "rows"),    # one slice filled; rows past a row group's last subtile
    (1030, 256, [2, 17, 0, 1] * 75, "rows"),  # one slice of 8 steps
    (1024, 320, [5, 0, 1] * 100, "rows"),    # one slice of 10 steps
    (300, 384, [3, 0, 16] * 100, "rows"),    # two slices of 6 steps
    (650, 448, [5, 17, 0] * 40, "rows"),     # two slices of 8 steps, the last one part filled
    (520, 1088, [7, 31], "rows"),            # four slices of 10, the last one part filled
    (520, 1024, [16, 31], "rows"),           # four slices of 8, filled
    (520, 1024, [200], "rows"),              # one expert, many tiles
    (96, 1536, [16] * 20, "rows"),           # eight slices of 6 steps, more tiles than experts' share of a block
    (100, 1984, [3, 18, 40], "rows"),        # eight slices of 8, the last one part filled
    (1100, 2496, [3, 18], "rows"),           # eight slices of 10, the last one part filled
    (640, 2560, [600], "rows"),              # one expert, many tiles and batches
    (200, 2688, [3, 50], "wide"),            # past 8 slices of 10 steps
    (64, 256, [120], "wide"),                # tiles filled by one expert
    (40, 64, [1, 16, 17], "narrow"),         # short rows
    (64, 96, [5, 60], "narrow"),             # K no whole scale words a lane
])
@pytest.mark.parametrize("precision", [0, 1])
def test_tiled_rows_kernel(hip, n, k, counts, route, precision):
    """The few-row kernel's slices, row groups, tiles and shares at their edges (the file's f64
    bar), with the rows in any order and without a row list."""
    import torch

    print(f"case: tiled rows n={n} k={k} experts={len(counts)} precision={precision}", flush=True)
    recs, x, off, rows = case(n, k, counts, 5 + n + k)
    assert dispatch.tiled(n, k, recs.w_off, recs.s_off, len(counts), max(counts), precision == 0) == route
    A = int(off[-1])
    buf = torch.from_numpy(np.stack(recs.recs)).cuda()
    addrs = torch.tensor([buf.data_ptr() + e * recs.stride for e in range(len(counts))], dtype=torch.int64,
                         device="cuda")
    for row_list in (True, False):
        xs = x if row_list else x[rows]
        y = torch.full((A + 3, n), float("nan"), dtype=torch.float32, device="cuda")
        hip.moe_tiled_nvfp4(addrs, torch.from_numpy(off).cuda(), torch.from_numpy(rows).cuda() if row_list else None,
                            len(counts), max(counts), torch.from_numpy(np.ascontiguousarray(xs)).cuda(), y, n, k,
                            recs.w_off, recs.s_off, 0, precision)
        got = y.cpu().numpy()
        want, mag = f64_eval(recs, x, off, rows, precision == 0)
        assert np.isnan(got[A:]).all(), "rows past the assignments were written"
        assert (np.abs(got[:A] - want) / mag).max() < 2e-6


@pytest.mark.parametrize("n,k,counts,bound,precision,works", [
    (640, 2560, [1700] * 4, 1700, 0, "tiles"),          # wide tiles
    (640, 2560, [1800] * 8, 2000, 1, "tiles"),          # a bound above the largest expert
    (640, 2560, [1800] + [20, 0, 49] * 3, 1800, 0, "rows"),
    (650, 2560, [17] * 40, 900, 1, "rows"),
    (448, 1600, [1100] * 20, 1100, 0, "tiles"),         # narrow tiles
    (448, 1600, [1100] + [7, 0, 65] * 13, 1100, 0, "rows"),
])
def test_tiled_counted(hip, n, k, counts, bound, precision, works):
    """Calls that launch both kernels: whichever the count leaves working writes every row, and
    nothing past them (the file's f64 bar)."""
    import torch

    print(f"case: tiled counted n={n} k={k} experts={len(counts)} precision={precision} {works}", flush=True)
    recs, x, off, rows = case(n, k, counts, 11 + n + len(counts))
    wide = k % 128 == 0
    both = dispatch.tiled(n, k, recs.w_off, recs.s_off, len(counts), bound, precision == 0)
    assert both == ("rows+wide" if wide else "rows+narrow")
    assert dispatch.counted(n, k, wide, precision == 0, counts, bound) == works
    A = int(off[-1])
    buf = torch.from_numpy(np.stack(recs.recs)).cuda()
    addrs = torch.tensor([buf.data_ptr() + e * recs.stride for e in range(len(counts))], dtype=torch.int64,
                         device="cuda")
    y = torch.full((A + 3, n), float("nan"), dtype=torch.float32, device="cuda")
    hip.moe_tiled_nvfp4(addrs, torch.from_numpy(off).cuda(), torch.from_numpy(rows).cuda(), len(counts), bound,
                        torch.from_numpy(x).cuda(), y, n, k, recs.w_off, recs.s_off, 0, precision)
    got = y.cpu().numpy()
    want, mag = f64_eval(recs, x, off, rows, precision == 0)
    assert np.isnan(got[A:]).all(), "rows past the assignments were written"
    assert (np.abs(got[:A] - want) / mag).max() < 2e-6
