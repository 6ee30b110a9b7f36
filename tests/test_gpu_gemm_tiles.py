"""FP64 GEMM tiles at the sizes where their loads change form: whole and
partial K steps of 16, odd extents and pitches, buffers off 16-byte
alignment, and views whose pairs are adjacent, adjacent off alignment, or
not adjacent.  Against torch's float64 product; every C element sums K
products of N(0, 1) numbers, so the bound is 1e-12 of the largest result,
as in test_gpu_core."""
import numpy as np
import pytest
import torch

from dtcf_amd import _lib, ops

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _rand(n, seed, dev):
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    return torch.randn(n, dtype=torch.float64, generator=g).to(dev)


def _close(got, ref, what):
    err = ((got - ref).abs().max() / ref.abs().max().clamp_min(1e-300)).item()
    assert err <= TOL, (what, err)


@pytest.fixture
def cfg_reset():
    yield
    ops.set_gemm_config(-1)


SIZES = ((1, 1, 1), (1, 3, 17), (2, 64, 15), (63, 65, 16), (64, 64, 31), (65, 63, 32), (127, 129, 33),
         (129, 255, 48), (131, 97, 113), (257, 191, 160))


@pytest.mark.parametrize("cfg", [-1, 0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_dense_odd_sizes_and_pitches(dev, cfg_reset, cfg, ta, tb):
    ops.set_gemm_config(cfg)
    for m, n, k in SIZES:
        for pad, off in ((0, 0), (1, 0), (2, 1), (3, 0)):
            ra, ca = (k, m) if ta else (m, k)
            rb, cb = (n, k) if tb else (k, n)
            lda, ldb, ldc = ca + pad, cb + pad, n + pad
            # buffers end with the operand's last element: no slack behind it
            A = _rand(off + (ra - 1) * lda + ca, 1, dev)
            B = _rand(off + (rb - 1) * ldb + cb, 2, dev)
            C = _rand((m - 1) * ldc + n, 3, dev)
            a = torch.as_strided(A, (ra, ca), (lda, 1), off)
            b = torch.as_strided(B, (rb, cb), (ldb, 1), off)
            ref = C.clone()
            torch.as_strided(ref, (m, n), (ldc, 1)).add_(
                0.5 * ((a.t() if ta else a).contiguous() @ (b.t() if tb else b).contiguous()))
            print("dense", cfg, ta, tb, m, n, k, pad, off, flush=True)
            ops.gemm(ta, tb, m, n, k, 0.5, A[off:], lda, B[off:], ldb, C, ldc)
            _close(C, ref, (m, n, k, pad, off))


def _offsets(rows, cols, kind, rng):
    """rows x cols offset tables over a dense array: the columns (k...) or the
    rows (r...) contiguous, in runs of an odd length, or off alignment."""
    if kind == "k":
        return np.arange(rows) * (cols + cols % 2), np.arange(cols)
    if kind == "k odd":  # pairs adjacent, rows at odd offsets
        return np.arange(rows) * (cols | 1), np.arange(cols)
    if kind == "k runs":  # runs of 7 columns
        return np.arange(rows) * 7, (np.arange(cols) // 7) * (7 * rows) + np.arange(cols) % 7
    if kind == "r":
        return np.arange(rows), np.arange(cols) * (rows + rows % 2)
    if kind == "r odd":
        return np.arange(rows), np.arange(cols) * (rows | 1)
    if kind == "r runs":
        return (np.arange(rows) // 5) * (5 * cols) + np.arange(rows) % 5, np.arange(cols) * 5
    return rng.permutation(rows) * cols, rng.permutation(cols)  # neither


@pytest.mark.parametrize("cfg", [-1, 0, 3, 4])
@pytest.mark.parametrize("ka", ["k", "k odd", "k runs", "r", "r odd", "r runs", "none"])
@pytest.mark.parametrize("kb", ["k", "k odd", "r odd", "r runs", "none"])
def test_views_off_alignment(dev, cfg_reset, cfg, ka, kb):
    ops.set_gemm_config(cfg)
    rng = np.random.default_rng(5)
    for m, n, k in ((66, 70, 34), (65, 129, 47), (140, 67, 16), (3, 5, 9)):
        ra, ca = _offsets(m, k, ka, rng)
        rb, cb = _offsets(n, k, kb, rng)
        A, B = _rand(int(ra.max() + ca.max()) + 1, 4, dev), _rand(int(rb.max() + cb.max()) + 1, 5, dev)
        C = _rand(m * n, 6, dev)
        ia = torch.from_numpy(ra[:, None] + ca[None, :]).to(dev)
        ib = torch.from_numpy(rb[:, None] + cb[None, :]).to(dev)
        ref = C + (A[ia] @ B[ib].t().contiguous()).reshape(-1)
        cv = ops.View(m, n, np.arange(m) * n, np.arange(n)) if m % 2 else None
        print("view", cfg, ka, kb, m, n, k, flush=True)
        ops.gemm_view(m, n, k, 1.0, A, ops.View(m, k, ra, ca), B, ops.View(n, k, rb, cb), C, cv, ldc=n)
        _close(C, ref, (ka, kb, m, n, k))


# Grids where the last tiles' K steps are dealt in runs: fewer tiles than
# workgroup slots, a little and a lot over whole rounds of slots, runs that
# cover several pieces of tiles, and K with a checked last step.
@pytest.mark.parametrize("cfg,m,n,k", [(3, 64, 64, 4096), (3, 500, 500, 500), (3, 130, 70, 3001),
                                       (3, 2112, 2112, 80), (3, 2200, 2050, 333), (0, 128, 128, 9000),
                                       (0, 1300, 1200, 700), (0, 2400, 2400, 171), (0, 2944, 2944, 100),
                                       (4, 192, 48, 20001), (5, 48, 192, 20001), (1, 1000, 900, 800)])
@pytest.mark.parametrize("cview", [False, True])
def test_split_runs(dev, cfg_reset, cfg, m, n, k, cview):
    ops.set_gemm_config(cfg)
    A, B, C = _rand(m * k, 7, dev), _rand(n * k, 8, dev), _rand(m * n, 9, dev)
    ref = C.view(m, n) - 2.0 * (A.view(m, k) @ B.view(n, k).t().contiguous())
    print("split", cfg, m, n, k, cview, flush=True)
    outs = []
    for _ in range(2):
        X = C.clone()
        if cview:  # C through a view of its transpose
            X = X.view(m, n).t().contiguous().reshape(-1)
            v = ops.View(m, n, np.arange(m), np.arange(n) * m)
            ops.gemm_view(m, n, k, -2.0, A, ops.View(m, k, np.arange(m) * k, np.arange(k)), B,
                          ops.View(n, k, np.arange(n) * k, np.arange(k)), X, v)
            outs.append(X.view(n, m).t().contiguous())
        else:
            ops.gemm(0, 1, m, n, k, -2.0, A, k, B, k, X, n)
            outs.append(X.view(m, n))
    _close(outs[0], ref, (cfg, m, n, k))
    assert torch.equal(outs[0], outs[1])  # the order of the additions is fixed


@pytest.mark.parametrize("sizes", [{"Oa": 5, "Ob": 4, "Va": 23, "Vb": 22}, {"Oa": 4, "Ob": 7, "Va": 21, "Vb": 19}])
def test_served_odd_extents_read_in_place(dev, sizes):
    # operands with odd extents are read in place in runs, not copied; small
    # enough for the einsum oracle, large enough (rows * K >= 65536) that the
    # rule applies
    import oracle
    from dtcf_amd import serve, termlist

    tl = termlist.load("t2")
    with serve.Server(1 << 30, 4) as srv:
        system = serve.System(srv, 0, 0, [tl], seed=3, sizes=sizes)
        prog = serve.Program(srv, tl, system)
        print("served", sizes, flush=True)
        got = prog.run()
        prog.destroy()
        stms = [(s.lhs.name, s.kind, s.lhs.idx, [(t.name, t.idx) + ((t.coef,) if s.kind == "sum" else ())
                                                 for t in s.terms]) for s in tl.statements]
        ref = oracle.termlist_run(stms, {n: system.host(n) for n in tl.inputs()})
    for n, x in got.items():
        err = np.abs(x - ref[n]).max() / np.abs(ref[n]).max()
        assert err <= TOL, (n, err)


def _group(ms, k, dev):
    """Grouped problems m x m x k over shared operands: the ctypes list and C."""
    import ctypes as C

    from dtcf_amd import blocksparse

    A, B = _rand(max(ms) * k, 1, dev), _rand(max(ms) * k, 2, dev)
    Cs = [torch.full((m * m,), float("nan"), dtype=torch.float64, device=dev) for m in ms]
    probs = (blocksparse.GemmProblem * len(ms))(*[
        blocksparse.GemmProblem(m, m, k, A.data_ptr(), k, B.data_ptr(), k, c.data_ptr(), m) for m, c in zip(ms, Cs)])

    def run(cfg):
        _lib.check(_lib.lib().dtcf_gemm_group_ex_f64(C.cast(probs, C.c_void_p), len(ms), 0, 1, 1.0, 1, cfg,
                                                     C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return run, A.view(-1, k), B.view(-1, k), Cs


# tiles of 64 x 64 and 128 x 128 in all: one problem of one tile, problems
# split whole, in part and not at all, sixteen problems and a second launch,
# past one and two rounds of workgroups
@pytest.mark.parametrize("cfg", [0, 3])
@pytest.mark.parametrize("ms,k", [([5], 40), ([300, 65, 129], 700), ([640, 600, 650, 610, 630], 333),
                                  ([130] * 20, 250), ([1100, 1200, 64, 900], 100), ([2300, 100, 2400], 170)])
def test_group_overwrite(dev, cfg, ms, k):
    run, A, B, Cs = _group(ms, k, dev)
    print("group", cfg, ms, k, flush=True)
    run(cfg)
    for m, c in zip(ms, Cs):
        _close(c.view(m, m), A[:m] @ B[:m].t().contiguous(), (cfg, ms, k, m))


def test_group_fills_the_chip_like_a_lone_launch(dev):
    """222 tiles of 128 x 128 x 640 in eight problems, and 225 in one: 108 us
    each; 167 us with every problem padded to whole rounds of XCDs by
    workgroups that exit at once."""
    run = _group([652, 620, 627, 630, 633, 631, 647, 610], 640, dev)[0]
    lone = _group([1900], 640, dev)[0]

    def us(f):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        out = []
        for _ in range(9):
            ev[0].record()
            for _ in range(5):
                f(0)
            ev[1].record()
            torch.cuda.synchronize()
            out.append(ev[0].elapsed_time(ev[1]) * 200)
        return sorted(out)[4]

    a, b = us(run), us(lone)
    print("group", a, "lone", b, flush=True)
    assert a <= 1.25 * b, (a, b)


# One served product with a fresh result: every element stored, none read or
# cleared before, by whole tiles, by runs that cover a tile and by the sums of
# cut ones.  The request block is first left full of another program's values.
@pytest.mark.parametrize("cfg", [-1, 0, 3])
@pytest.mark.parametrize("m,n,k", [(500, 500, 500), (130, 70, 3001), (2200, 2050, 333), (1300, 1200, 700)])
def test_served_overwrite(dev, cfg_reset, cfg, m, n, k):
    from dtcf_amd import serve, termlist

    text = ("range M = 1.0;\nrange N = 1.0;\nrange K = 1.0;\nindex i = M;\nindex j = N;\nindex l = K;\n"
            "array a([M][K]), b([K][N]), c([M][N]);\nc[i,j] = (a[i,l] * b[l,j])\n")
    tl = termlist.parse(text)
    ops.set_gemm_config(cfg)
    with serve.Server(1 << 29, 1) as srv:
        system = serve.System(srv, 0, 0, [tl], sizes={"M": m, "N": n, "K": k})
        prog = serve.Program(srv, tl, system)
        print("served overwrite", cfg, m, n, k, flush=True)
        out = [torch.full((m * n,), float("nan"), dtype=torch.float64, device=dev)]
        for _ in range(2):
            rid = prog.submit(out)[0]
            _lib.check(srv.wait(rid, 60000.0))
            srv.release(rid)
        prog.destroy()
        ref = system.host("a") @ system.host("b")
    got = out[0].view(m, n).cpu().numpy()
    assert np.abs(got - ref).max() / np.abs(ref).max() <= TOL
