"""View products whose operands keep a block table (tiles in an order that is
no sum of a row and a column part): pairs adjacent and aligned, adjacent off
alignment, broken at odd block extents, along the columns or the rows, one
operand or both, whole and partial last K steps, odd row counts.  Against
torch's float64 product of the gathered operands, 1e-12 of the largest result
as in test_gpu_core."""
import numpy as np
import pytest
import torch

from dtcf_amd import ops

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _rand(n, seed, dev):
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    return torch.randn(n, dtype=torch.float64, generator=g).to(dev)


def _tiles(rows, cols, rpb, cpb, rowwise, rng, off=0):
    """rows x cols in rpb x cpb tiles stored one after another in a random
    order, each row-major (or column-major): the view and its offsets."""
    nr, nc = rows // rpb, cols // cpb
    blk = rng.permutation(nr * nc).astype(np.int64) * (rpb * cpb) + off
    r, c = np.arange(rows), np.arange(cols)
    ro, co = (r % rpb, (c % cpb) * rpb) if rowwise else ((r % rpb) * cpb, c % cpb)
    at = ro[:, None] + co[None, :] + blk.reshape(nr, nc)[(r // rpb)[:, None], (c // cpb)[None, :]]
    return ops.View(rows, cols, ro, co, blk, rpb, cpb), at


# tile (rows, columns) of A, of B, both along K or the rows, an odd first offset
FORMS = (((6, 8), (10, 8), False, False, 0), ((6, 8), (10, 8), True, True, 0), ((6, 8), (10, 8), False, True, 1),
         ((7, 5), (3, 5), False, False, 0), ((7, 5), (3, 5), True, True, 0), ((1, 40), (1, 20), False, False, 0),
         ((21, 1), (15, 1), True, True, 0), ((3, 10), (5, 2), True, False, 0))


@pytest.mark.parametrize("cfg", [-1, 0, 3, 4])
@pytest.mark.parametrize("form", FORMS)
def test_block_tables(dev, form, cfg):
    (ra, ca), (rb, cb), wa, wb, off = form
    rng = np.random.default_rng(2)
    ops.set_gemm_config(cfg)
    try:
        for m, n, k in ((42, 30, 40), (63, 75, 80), (147, 135, 120), (168, 330, 200)):
            m, n = m // ra * ra, n // rb * rb
            av, ia = _tiles(m, k, ra, ca, wa, rng, off)
            bv, ib = _tiles(n, k, rb, cb, wb, rng, off)
            A, B, C = _rand(m * k + off, 1, dev), _rand(n * k + off, 2, dev), _rand(m * n, 3, dev)
            Ad, Bd = A[torch.from_numpy(ia).to(dev)], B[torch.from_numpy(ib).to(dev)]
            ref = C.view(m, n) + 0.5 * (Ad @ Bd.t().contiguous())
            dense = [ops.View(r, k, np.arange(r) * k, np.arange(k)) for r in (m, n)]
            cv = ops.View(m, n, np.arange(m) * n, np.arange(n)) if m % 2 else None
            Ac, Bc = Ad.contiguous().reshape(-1), Bd.contiguous().reshape(-1)
            for x, xv, y, yv in ((A, av, B, bv), (A, av, Bc, dense[1]), (Ac, dense[0], B, bv)):
                print("tables", form, cfg, m, n, k, flush=True)
                X = C.clone()
                ops.gemm_view(m, n, k, 0.5, x, xv, y, yv, X, cv, ldc=n)
                assert ((X.view(m, n) - ref).abs().max() / ref.abs().max()).item() <= TOL
    finally:
        ops.set_gemm_config(-1)


def test_scrambled_tiles_cost_no_checked_loads(dev):
    """The same 2304^3 product with its tiles in a scrambled order and in
    order (a table that folds, read straight into LDS).  Scrambled it takes
    1.3 times as long; with every K step loaded element by element under
    bounds checks it took 3.2 times."""
    n, t = 2304, 144
    rng = np.random.default_rng(1)
    A, B = _rand(n * n, 1, dev), _rand(n * n, 2, dev)
    C = torch.zeros(n * n, dtype=torch.float64, device=dev)
    scr = [_tiles(n, n, t, t, False, rng)[0] for _ in range(2)]
    r = np.arange(n)
    order = [ops.View(n, n, (r % t) * t, r % t, np.arange((n // t) ** 2) * t * t, t, t) for _ in range(2)]

    def us(av, bv):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        out = []
        for _ in range(7):
            ev[0].record()
            ops.gemm_view(n, n, n, 1.0, A, av, B, bv, C, None, ldc=n)
            ev[1].record()
            torch.cuda.synchronize()
            out.append(ev[0].elapsed_time(ev[1]) * 1e3)
        return sorted(out)[3]

    a, b = us(*scr), us(*order)
    print("scrambled", a, "in order", b, flush=True)
    assert a <= 2.0 * b, (a, b)


@pytest.mark.parametrize("dims,oa,ob", [((23, 34, 20, 35, 30, 15), (2, 0, 3, 1), (1, 2, 3, 0)),
                                        ((11, 16, 18, 35, 26, 35), (2, 0, 3, 1), (0, 3, 1, 2))])
def test_gathered_operands_fill_the_chip(dev, dims, oa, ob):
    """(a, b) x (c, d) summed over (e, f) with B's (or A's) last memory index
    no neighbour along rows or columns, so B is read element by element,
    against the same product with both stored rows first: 1.06 and 1.15 times
    its time; cut over K as if it were read in pairs it took 1.55 times."""
    a, b, c, d, e, f = dims
    m, n, k = a * b, c * d, e * f

    def view(x, order):
        st, s = [0] * 4, 1
        for q in reversed(order):
            st[q], s = s, s * x[q]
        i = [np.arange(v) * t for v, t in zip(x, st)]
        return ops.View(x[0] * x[1], x[2] * x[3], (i[0][:, None] + i[1]).ravel(), (i[2][:, None] + i[3]).ravel())

    A, B, C = _rand(m * k, 1, dev), _rand(n * k, 2, dev), torch.zeros(m * n, dtype=torch.float64, device=dev)

    def us(av, bv):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        out = []
        for _ in range(7):
            ev[0].record()
            for _ in range(30):
                ops.gemm_view(m, n, k, 1.0, A, av, B, bv, C, None, ldc=n)
            ev[1].record()
            torch.cuda.synchronize()
            out.append(ev[0].elapsed_time(ev[1]) / 30 * 1e3)
        return sorted(out)[3]

    x, y = (a, b, e, f), (c, d, e, f)
    p, q = us(view(x, oa), view(y, ob)), us(view(x, (0, 1, 2, 3)), view(y, (0, 1, 2, 3)))
    print("gathered", p, "rows first", q, flush=True)
    assert p <= 1.3 * q, (p, q)


# Rectangles of a view keep its pair flags only where they start and end on
# pairs: odd and even first rows and columns, odd counts, of views whose pairs
# run along K or the rows, aligned or not.
@pytest.mark.parametrize("kind", ["k", "k odd", "r", "r odd"])
@pytest.mark.parametrize("r0,c0,m,k", [(0, 0, 66, 48), (1, 0, 65, 47), (2, 1, 64, 48), (3, 3, 61, 33), (4, 2, 63, 34)])
def test_sub_views(dev, kind, r0, c0, m, k):
    import ctypes as C

    from dtcf_amd import _lib

    rows, cols, n = 70, 52, 40
    ro, co = {"k": (np.arange(rows) * cols, np.arange(cols)), "k odd": (np.arange(rows) * (cols + 1), np.arange(cols)),
              "r": (np.arange(rows), np.arange(cols) * rows), "r odd": (np.arange(rows), np.arange(cols) * (rows + 1))}[kind]
    A, B, X = _rand(int(ro.max() + co.max()) + 1, 1, dev), _rand(n * k, 2, dev), _rand(m * n, 3, dev)
    parent = ops.View(rows, cols, ro, co)
    sub = ops.View.__new__(ops.View)
    h = C.c_void_p()
    L = _lib.lib()
    _lib.check(L.dtcf_view_sub(parent.h, C.c_int64(r0), C.c_int64(m), C.c_int64(c0), C.c_int64(k), C.byref(h)))
    sub.h, sub.rows, sub.cols = h, m, k
    bv = ops.View(n, k, np.arange(n) * k, np.arange(k))
    at = torch.from_numpy(ro[r0:r0 + m, None] + co[None, c0:c0 + k]).to(dev)
    ref = X.view(m, n) + A[at] @ B.view(n, k).t().contiguous()
    print("sub", kind, r0, c0, m, k, flush=True)
    ops.gemm_view(m, n, k, 1.0, A, sub, B, bv, X, None, ldc=n)
    assert ((X.view(m, n) - ref).abs().max() / ref.abs().max()).item() <= TOL
