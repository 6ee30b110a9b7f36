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


@pytest.mark.parametrize("which,oa,ob", [("t2", 22, 23), ("t2", 32, 31), ("t1", 32, 33), ("t1", 45, 46),
                                         ("t1", 54, 53), ("t1", 54, 56)])
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
