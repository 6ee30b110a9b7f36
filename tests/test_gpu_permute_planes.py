"""Permute copies where the flat form's tiles and plane groups change: extents
of one or two, exactly 63 / 64 / 65 and one past several tiles, planes that
fill a work item and that leave the last one short, rows longer than an item,
extents at which the 16-byte form starts and stops; offsets from steps and
from tables, with and without accumulation.  Copies are exact; 0.5 * x + y
rounds once, so both are bit for bit against torch's permute on the CPU."""
import itertools

import pytest
import torch

from dtcf_amd import ops

pytestmark = pytest.mark.gpu

SHAPES = ([1, 3, 1, 2], [63, 2, 64, 1], [64, 3, 63, 2], [65, 2, 129, 3], [2, 2, 2, 9], [13, 11, 3, 7],
          [127, 5, 2, 61], [2, 4099, 1, 3], [28, 2, 32, 2], [26, 2, 30, 4], [3, 8192])


@pytest.mark.parametrize("tables", (False, True))
@pytest.mark.parametrize("w", SHAPES)
def test_permute_planes(dev, w, tables):
    nt, n = 3, int(torch.tensor(w).prod())
    g = torch.Generator().manual_seed(n)
    step_in, step_out = n + 5, n + 2  # gaps that must stay as they are
    x = torch.randn(nt * step_in, dtype=torch.float64, generator=g)
    y = torch.randn(nt * step_out, dtype=torch.float64, generator=g)
    order = [2, 0, 1] if tables else [0, 1, 2]
    off = dict(src_off=torch.tensor([o * step_in for o in order], device=dev),
               dst_off=torch.tensor([(2 - o) * step_out for o in order], device=dev)) if tables else \
        dict(src_step=step_in, dst_step=step_out)
    xd = x.to(dev)
    istr_in = [int(torch.tensor(w[i + 1:]).prod()) if i + 1 < len(w) else 1 for i in range(len(w))]
    for pm in itertools.permutations(range(len(w))):
        ext = [w[c] for c in pm]
        ostr = [int(torch.tensor(ext[i + 1:]).prod()) if i + 1 < len(w) else 1 for i in range(len(w))]
        for alpha, beta in ((1.0, 0.0), (0.5, 1.0)):
            print("planes", w, tables, pm, alpha, beta, flush=True)
            got = y.to(dev)
            ops.permute_copy(xd, got, ext, [istr_in[c] for c in pm], ostr, ntiles=nt, alpha=alpha, beta=beta,
                             **off)
            want = y.clone()
            for o in range(nt):
                d = (2 - o if tables else o) * step_out
                p = x[o * step_in:o * step_in + n].view(w).permute(pm).reshape(-1)
                want[d:d + n] = alpha * p + (want[d:d + n] if beta else 0.0)
            assert torch.equal(got.cpu(), want), (pm, alpha, beta)


# The fixed 32 x 32 tiles next to the flat form, on either side of the rule:
# fill 0.4 (32 x 13, 31 x 13), second tiles nearly empty from 40 MB on
# (33 x 75 in 1000 and 1100 planes), more than 275 MB (257 x 63).
@pytest.mark.parametrize("w,nt", [([32, 13], 700), ([31, 13], 700), ([33, 75], 1000), ([33, 75], 1100),
                                  ([257, 63], 1050), ([257, 63], 1080), ([19, 5, 31], 40)])
def test_permute_tiles_either_side(dev, w, nt):
    n = nt * int(torch.tensor(w).prod())
    x = torch.randn(n, dtype=torch.float64, device=dev)
    y = torch.randn(n, dtype=torch.float64, device=dev)
    order = list(range(len(w)))[::-1]
    want = x.view(nt, *w).permute(0, *[1 + c for c in order]).reshape(-1)
    print("sides", w, nt, flush=True)
    got = torch.full_like(x, float("nan"))
    assert torch.equal(ops.permute_tiles(x, w, order, nt, got), want)
    ext = [w[c] for c in order]
    istr = [int(torch.tensor(w[c + 1:]).prod()) if c + 1 < len(w) else 1 for c in order]
    ostr = [int(torch.tensor(ext[i + 1:]).prod()) if i + 1 < len(w) else 1 for i in range(len(w))]
    step = n // nt
    got = y.clone()
    ops.permute_copy(x, got, ext, istr, ostr, ntiles=nt, src_step=step, dst_step=step, alpha=0.5, beta=1.0)
    assert torch.equal(got, 0.5 * want + y)


def test_filled_odd_tiles_keep_their_rate(dev):
    """75 x 2028 in 49 planes (119 MB read and written) by 8-byte accesses
    against 64 x 2016 in 57 by 16-byte ones: 21 us and about 20.  In flat
    tiles of up to 64 x 63 it took 31."""
    def us(w, nt):
        n = nt * w[0] * w[1]
        x = torch.randn(n, dtype=torch.float64, device=dev)
        y = torch.empty_like(x)
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        out = []
        for _ in range(9):
            ev[0].record()
            for _ in range(20):
                ops.permute_tiles(x, w, [1, 0], nt, y)
            ev[1].record()
            torch.cuda.synchronize()
            out.append(ev[0].elapsed_time(ev[1]) * 50)
        return sorted(out)[4]

    a, b = us([2028, 75], 49), us([2016, 64], 57)
    print("odd", a, "even", b, flush=True)
    assert a <= 1.3 * b, (a, b)
