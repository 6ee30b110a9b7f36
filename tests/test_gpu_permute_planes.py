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
