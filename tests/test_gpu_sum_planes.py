"""Sum statements whose output planes (the last two indices) fall on either
side of each kernel instance: planes below and above 512, 1024 and 2048
elements, even and odd extents, close to the 3072 limit and past it, as many
planes as fit one round of workgroups and more.  Every statement against the
einsum oracle, with the bound of the serving parity tests."""
import numpy as np
import pytest

import oracle
from dtcf_amd import serve, termlist

pytestmark = pytest.mark.gpu


SIZES = (("t2", 22, 23), ("t2", 32, 31), ("t1", 32, 33), ("t1", 38, 40), ("t1", 45, 46), ("t1", 54, 53),
         ("t1", 54, 56))


def _instances(which, oa, ob):
    """(pairs, elements per thread of 512) of the sum statements' planes."""
    tl, ext, out = termlist.load(which), {"Oa": oa, "Ob": ob, "Va": 3, "Vb": 2}, set()
    for s in tl.statements:
        shape = [1] * 4 + [ext[r] for r in tl.arrays[s.lhs.name].ranges]
        d2, d3 = shape[-2:]
        if s.kind == "sum" and (d2 + 1) * d3 <= 3072:
            pairs = d2 % 2 == 0 and d3 % 2 == 0
            out.add((pairs, min(x for x in ((2, 4, 6) if pairs else (1, 2, 4, 6)) if 512 * x >= d2 * d3)))
    return out


def test_sizes_reach_every_instance(dev):
    assert set().union(*[_instances(*x) for x in SIZES]) == {(True, x) for x in (2, 4, 6)} | {
        (False, x) for x in (1, 2, 4, 6)}


@pytest.mark.parametrize("which,oa,ob", SIZES)
def test_sum_planes(dev, which, oa, ob):
    tl = termlist.load(which)
    print("sum planes", which, oa, ob, flush=True)
    with serve.Server(4 << 30, 4) as srv:
        system = serve.System(srv, 0, 0, [tl], seed=5, sizes={"Oa": oa, "Ob": ob, "Va": 3, "Vb": 2})
        prog = serve.Program(srv, tl, system, expose=True)
        got = prog.run()
        prog.destroy()
        stms = [(s.lhs.name, s.kind, s.lhs.idx, [(t.name, t.idx) + ((t.coef,) if s.kind == "sum" else ())
                                                 for t in s.terms]) for s in tl.statements]
        ref = oracle.termlist_run(stms, {n: system.host(n) for n in tl.inputs()})
    for s in tl.statements:
        n = s.lhs.name
        err = np.abs(got[n] - ref[n]).max() / max(np.abs(ref[n]).max(), 1e-300)
        assert err <= 1e-12, (n, s.kind, err)
