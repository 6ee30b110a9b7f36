"""Fused slice products at the sizes where their C tile and split change
(tiles as chosen at level 4 on 256 CUs): 128 x 128 with ragged edges, whole
and cut over K; 192 x 128 and 128 x 192 whole with ragged edges (planes are
padded to 128 rows); 128 x 192 with the last 74 of 330 tiles cut, and with all
of 96 cut; C dense, through a view, accumulated twice.  INT8 digits against the one-GEMM-per-
product path (the same exact integers, recombined in FP64 in another order:
1e-13 of the largest result, as test_gpu_mixed); BF16 and FP16 against FP64
(5e-6, the bound stated for their FP32 sums)."""
import numpy as np
import pytest
import torch

from dtcf_amd import mixed, ops

pytestmark = pytest.mark.gpu

SIZES = ((2304, 2304, 1000), (3000, 2400, 700), (2400, 3000, 300), (193, 5000, 260), (5000, 193, 260),
         (130, 190, 6000), (1537, 129, 2100), (64, 64, 64), (2900, 2000, 1000), (2000, 2900, 1000),
         (2700, 2700, 8000), (1500, 1400, 9000))
MODES = ((mixed.I8, 3, 4), (mixed.I8, 4, 4), (mixed.I8, 4, 6), (mixed.I8, 5, 6), (mixed.BF16X3, 3, 4),
         (mixed.F16X3, 3, 4))


@pytest.mark.parametrize("prec,ns,lev", MODES)
@pytest.mark.parametrize("m,n,k", SIZES)
def test_fused_tiles(dev, prec, ns, lev, m, n, k):
    A, B = mixed.fill_normal(m * k, 1, 1.0), mixed.fill_normal(n * k, 2, 1.0)
    sa = mixed.Split(prec, A, mixed.dense_view(m, k), ns)
    sb = mixed.Split(prec, B, mixed.dense_view(n, k), ns)
    C0 = mixed.fill_normal(m * n, 3, 1.0)
    print("slices", prec, ns, lev, m, n, k, flush=True)
    got = C0.clone()
    for _ in range(2):
        mixed.gemm_split(sa, sb, got, alpha=0.5, ldc=n, max_level=lev)
    if prec == mixed.I8:
        mixed.set_fused(False)
        try:
            ref = C0.clone()
            for _ in range(2):
                mixed.gemm_split(sa, sb, ref, alpha=0.5, ldc=n, max_level=lev)
        finally:
            mixed.set_fused(True)
        tol = 1e-13
    else:
        ref = C0 + (A.view(m, k) @ B.view(n, k).t().contiguous()).reshape(-1)
        tol = 5e-6
    scale = ref.abs().max()
    assert ((got - ref).abs().max() / scale).item() <= tol
    # C through a view of its transpose: the same values, element for element
    view = ops.View(m, n, np.arange(m), np.arange(n) * m)
    gv = C0.view(m, n).t().contiguous().reshape(-1)
    for _ in range(2):
        mixed.gemm_split(sa, sb, gv, alpha=0.5, cview=view, max_level=lev)
    assert torch.equal(gv.view(n, m).t().contiguous().reshape(-1), got)



@pytest.mark.parametrize("prec", [mixed.BF16X3, mixed.F16X3])
def test_fp32_sums_stay_short(dev, prec):
    """The FP32 level sums run over half of K at most where 128 x 128 tiles
    would leave a short last round, whatever tile the plan takes.  One product
    of 2^30 at the start and 1310 of 1 in the second half (K padded to 2688, 84
    steps of 32): added to 2^30 in FP32 a step's 32 is below half a unit in the
    last place and is lost, in a sum of its own every one counts."""
    m, n, k = 5954, 928, 2654
    row = torch.zeros(k, dtype=torch.float64, device=dev)
    row[0], row[1344:] = 2.0 ** 15, 1.0
    sa = mixed.Split(prec, row.repeat(m), mixed.dense_view(m, k), 3)
    sb = mixed.Split(prec, row.repeat(n), mixed.dense_view(n, k), 3)
    C = torch.zeros(m * n, dtype=torch.float64, device=dev)
    print("fp32 sums", prec, flush=True)
    mixed.gemm_split(sa, sb, C, ldc=n, max_level=4)
    assert (C == 2.0 ** 30 + (k - 1344)).all()


@pytest.mark.parametrize("ns", [3, 4])
def test_flush_inside_wide_tiles(dev, ns):
    """Level 4 in one piece (216 tiles of 128 x 192 on 256 CUs) over K = 70,000,
    past the interval at which the INT32 level sums are flushed (65,027), with
    every digit product near its bound: x = -(63 * 256^(ns-1) + 128 * (256^(ns-1)
    - 1) / 255) / 2^(8 ns - 2).  Exact up to the dropped levels."""
    m, n, k = 2304, 2304, 70000
    x = -(63 * 256 ** (ns - 1) + 128 * (256 ** (ns - 1) - 1) // 255) / 2.0 ** (8 * ns - 2)
    A = torch.full((m * k,), x, dtype=torch.float64, device=dev)
    sa = mixed.Split(mixed.I8, A, mixed.dense_view(m, k), nslice=ns)
    sb = mixed.Split(mixed.I8, A, mixed.dense_view(n, k), nslice=ns)
    C = torch.zeros(m * n, dtype=torch.float64, device=dev)
    print("flush", ns, flush=True)
    mixed.gemm_split(sa, sb, C, alpha=0.5, ldc=n, max_level=4)
    ref = 0.5 * k * x * x
    assert (C == C[0]).all()
    assert abs(C[0].item() - ref) <= 0.5 * k * 16 * ns * 128 * 128 * 2.0 ** -40 + 1e-14 * ref
