"""Products recorded on a capturing stream whose split workspace was never
reserved: those that whole tiles serve nearly as well run without the split,
those that would leave most of the device idle are refused, and after a
reservation both are recorded with it.  Replays against the eager result
(another order of the same K sums: 1e-12 of the largest) and bit for bit
against each other."""
import ctypes as C

import pytest
import torch

from dtcf_amd import _lib, blocksparse, mixed, ops

pytestmark = pytest.mark.gpu


def _cases(dev):
    def dense(m, n, k):
        A, B = mixed.fill_normal(m * k, 1, 1.0), mixed.fill_normal(n * k, 2, 1.0)
        out = torch.zeros(m * n, dtype=torch.float64, device=dev)
        return out, lambda: ops.gemm(0, 1, m, n, k, 1.0, A, k, B, k, out, n), (A, B)

    def slices(m, n, k):
        A, B = mixed.fill_normal(m * k, 1, 1.0), mixed.fill_normal(n * k, 2, 1.0)
        sa = mixed.Split(mixed.I8, A, mixed.dense_view(m, k), 3)
        sb = mixed.Split(mixed.I8, B, mixed.dense_view(n, k), 3)
        out = torch.zeros(m * n, dtype=torch.float64, device=dev)
        return out, lambda: mixed.gemm_split(sa, sb, out, ldc=n, max_level=4), (sa, sb)

    def group(m, count, k):
        A, B = mixed.fill_normal(m * k, 1, 1.0), mixed.fill_normal(m * k, 2, 1.0)
        out = torch.zeros(count * m * m, dtype=torch.float64, device=dev)
        probs = (blocksparse.GemmProblem * count)(*[
            blocksparse.GemmProblem(m, m, k, A.data_ptr(), k, B.data_ptr(), k, out.data_ptr() + 8 * i * m * m, m)
            for i in range(count)])

        def run():
            _lib.check(_lib.lib().dtcf_gemm_group_ex_f64(
                C.cast(probs, C.c_void_p), count, 0, 1, 1.0, 0, 0, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        return out, run, (A, B, probs)

    # (maker, runs uncut): 361 tiles of 128 x 128, 144 of 128 x 128 or 96 of 128
    # x 192, 360 tiles in ten problems; and grids of a few tiles with long K
    return [(lambda: dense(2400, 2400, 2400), True), (lambda: dense(300, 300, 3000), False),
            (lambda: slices(1500, 1500, 9000), True), (lambda: slices(300, 300, 9000), False),
            (lambda: group(768, 10, 1600), True), (lambda: group(256, 2, 4000), False)]


@pytest.mark.parametrize("case", range(6))
def test_capture_without_workspace(dev, case):
    make, uncut = _cases(dev)[case]
    out, run, keep = make()
    run()
    torch.cuda.synchronize()
    want = out.clone()
    scale = want.abs().max().item()
    s = torch.cuda.Stream()

    def capture():
        g = torch.cuda.CUDAGraph()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            g.capture_begin()
            try:
                run()
                err = None
            except _lib.DtcfError as e:
                err = e
                out.mul_(1.0)  # the graph is not empty
            g.capture_end()
        torch.cuda.current_stream().wait_stream(s)
        return g, err

    def replays(g):
        got = []
        for rep in range(3):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            got.append(out.clone())
            run()  # the program's own eager work between the replays
            torch.cuda.synchronize()
        assert all(torch.equal(x, got[0]) for x in got)
        assert ((got[0] - want).abs().max().item()) <= 1e-12 * scale

    print("capture", case, uncut, flush=True)
    g, err = capture()
    if uncut:
        assert err is None
        replays(g)
    else:
        assert err is not None and "reserve" in str(err)
    _lib.check(_lib.lib().dtcf_gemm_reserve_workspace(C.c_void_p(s.cuda_stream)))
    g2, err = capture()
    assert err is None
    replays(g2)
