"""The framework's workloads as timed cases, through its public entry points.

Each case is a dict of plain values: a ``kind`` (one public path) and its
sizes.  ``listed()`` names the fixed ones, ``draw(rng)`` gives others of the
same kinds and ranges, ``prepare`` makes a case's inputs and the plan or
handle a program would keep, ``run`` does one pass, ``work`` states the bytes
and operations the path cannot do without, and ``exact`` gives what ``run``
returns, computed in 64 bits by plain torch.

Orbital counts are o occupied and v virtual; inputs are N(0, 0.05^2) as
everywhere in this repository unless a case says otherwise.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from dtcf_amd import _lib, blocksparse, ccsd, dltc, mixed, ops, rrr, serve, termlist

SIGMA = 0.05
DEV = "cuda"


def listed():
    return [
        # The CCD ladder of a small molecule as one DLTC term: the latency of
        # a single small contraction (two launches' worth of work).
        {"name": "ladder_term_o8_v32", "kind": "term", "o": 8, "v": 32},
        # local_contraction at odd extents and pitches: what a caller with
        # odd orbital counts (11^3 rows, 11*107 columns, 5*181 summed) passes.
        {"name": "gemm_odd_1331x1177x905", "kind": "gemm", "m": 1331, "n": 1177, "k": 905,
         "ta": 0, "tb": 1},
        # One rank's ring step of a SUMMA round, operands read in place: the
        # largest dense FP64 contraction, the headline of bench.py.
        {"name": "ring_step_o48_v192", "kind": "step", "o": 48, "v": 192, "vo": 4, "vv": 4,
         "sym": False, "mode": rrr.FUSED},
        # A mid-size ring step whose first operand is symmetric (stored and
        # bounced tiles), packed by one pass per class.
        {"name": "symmetric_step_o24_v100", "kind": "step", "o": 24, "v": 100, "vo": 4, "vv": 5,
         "sym": True, "mode": rrr.FUSED},
        # A T1-type product of the UHF iteration: one side 48 wide, short K.
        {"name": "thin_1769472x48x192", "kind": "gemm", "m": 1769472, "n": 48, "k": 192,
         "ta": 0, "tb": 0},
        # A block-sparse T2 ring term under D2h, one dense GEMM per irrep.
        {"name": "d2h_ring_o64_v256", "kind": "d2h", "o": 64, "v": 256, "orbitals": 5},
        # Mixed precision at 1e-9 accuracy: the ladder with four INT8 digits to
        # level 6, the integral's digits kept, the amplitudes split each time.
        {"name": "ladder_int8x4_o32_v128", "kind": "mixed", "m": 16384, "n": 1024, "k": 16384,
         "prec": mixed.I8, "ns": 4, "lev": 6, "keep_a": True, "rows": True},
        # The fast mixed form of a CCSD iteration: a ring with three digits to
        # level 4, both operands split in the call.
        {"name": "ring_int8x3_o48_v192", "kind": "mixed", "m": 9216, "n": 9216, "k": 9216,
         "prec": mixed.I8, "ns": 3, "lev": 4, "keep_a": False, "rows": False},
        # The tile transposes of a rank's tensor at odd tile extents.
        {"name": "transpose_tiles_11x13x45x47", "kind": "permute", "ntiles": 256, "w0": 11,
         "w1": 13, "w2": 45, "w3": 47, "perm": "2031"},
        # Amplitude update, energy and residual norm of one CCD iteration.
        {"name": "amplitudes_o64_v256", "kind": "amplitudes", "o": 64, "v": 256},
        # The T1 and T2 residual programs of a small open-shell molecule (the
        # term lists' own O = 10, V = 100 for the alpha spin), served in FP64:
        # 378 statements, most of them of a few microseconds.
        {"name": "served_fp64_o19_v199", "kind": "served", "oa": 10, "ob": 9, "va": 100, "vb": 99,
         "slots": 8},
        # A whole UHF CCSD iteration with mixed-precision residuals, integral
        # digits resident: residuals, amplitude update, energy and norms.
        {"name": "ccsd_int8x3_o64_v256", "kind": "ccsd", "o": 64, "v": 256, "ns": 3, "lev": 4},
    ]


# ------------------------------------------------------------------- draws
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["term", "gemm", "gemm", "thin", "step", "step", "d2h", "mixed", "mixed",
                       "permute", "permute", "amplitudes", "served", "ccsd"])
    if kind == "term":
        return {"kind": "term", "o": rng.randint(3, 24), "v": rng.randint(12, 72)}
    if kind == "gemm":
        while True:
            m, n, k = _log(rng, 33, 12000), _log(rng, 33, 12000), _log(rng, 17, 12000)
            if 1e6 <= 2.0 * m * n * k <= 4e11:
                return {"kind": "gemm", "m": m, "n": n, "k": k, "ta": rng.randint(0, 1),
                        "tb": rng.randint(0, 1)}
    if kind == "thin":
        w, k = rng.choice([16, 24, 40, 48]), 8 * rng.randint(3, 24)
        rows, tall = _log(rng, 2e5, 3e6), rng.random() < 0.5
        return {"kind": "gemm", "m": rows if tall else w, "n": w if tall else rows, "k": k, "ta": 0,
                "tb": rng.randint(0, 1)}
    if kind == "step":
        vo, vv = rng.randint(2, 4), rng.randint(2, 5)
        sym = rng.random() < 0.4
        return {"kind": "step", "o": vo * rng.randint(3, 12), "v": vv * rng.randint(5, 36), "vo": vo,
                "vv": vv, "sym": sym,
                "mode": rng.choice([rrr.FUSED, rrr.FUSED, rrr.PACKED, rrr.LITERAL])}
    if kind == "d2h":
        return {"kind": "d2h", "o": rng.randint(24, 64), "v": rng.randint(64, 240),
                "orbitals": rng.randint(1, 99)}
    if kind == "mixed":
        prec, ns, lev = rng.choice([(mixed.I8, 3, 4), (mixed.I8, 4, 4), (mixed.I8, 4, 5),
                                    (mixed.I8, 4, 6), (mixed.I8, 5, 6), (mixed.BF16X3, 3, 4),
                                    (mixed.F16X3, 3, 4)])
        while True:
            m, n, k = _log(rng, 500, 16000), _log(rng, 500, 16000), _log(rng, 500, 16000)
            if 2.0 * m * n * k <= 8e11:
                return {"kind": "mixed", "m": m, "n": n, "k": k, "prec": prec, "ns": ns, "lev": lev,
                        "keep_a": rng.random() < 0.5, "rows": rng.random() < 0.5}
    if kind == "permute":
        return {"kind": "permute", "ntiles": _log(rng, 16, 300), "w0": rng.randint(5, 14),
                "w1": rng.randint(5, 14), "w2": rng.randint(8, 48), "w3": rng.randint(8, 48),
                "perm": rng.choice(["2031", "0213", "1032", "2301", "3120", "0132", "2103"])}
    if kind == "amplitudes":
        return {"kind": "amplitudes", "o": rng.randint(9, 60), "v": rng.randint(40, 240)}
    if kind == "served":
        return {"kind": "served", "oa": rng.randint(5, 16), "ob": rng.randint(5, 16),
                "va": rng.randint(24, 96), "vb": rng.randint(24, 96), "slots": rng.choice([1, 4, 8])}
    o = 2 * rng.randint(12, 30)
    return {"kind": "ccsd", "o": o, "v": 2 * rng.randint(40, 110), **rng.choice(
        [{"ns": 3, "lev": 4}, {"ns": 4, "lev": 4}, {"ns": 4, "lev": 5}])}


# ------------------------------------------------------------------ inputs
def _normal(shape, seed, sigma=SIGMA):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    n = int(np.prod(shape))
    return torch.randn(n, dtype=torch.float64, device=DEV, generator=g).mul_(sigma)


def _energies(n, seed, lo, hi):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.rand(n, dtype=torch.float64, device=DEV, generator=g).mul_(hi - lo).add_(lo)


class _Served:
    """A server with its system and programs, given back with the state."""

    def __init__(self, budget, slots):
        self.server = serve.Server(budget, slots)
        self.programs = []

    def __del__(self):
        torch.cuda.synchronize()
        for p in self.programs:
            p.destroy()
        self.server.close()


def _step_tensors(c, seed):
    o, v, vo, vv = c["o"], c["v"], c["vo"], c["vv"]
    vg = [vo, vo, vv, vv]
    out = []
    addrs = rrr.tile_addresses("cccc", vg)
    for i in range(3):
        x = _normal((o * o * v * v,), 4 * seed + i)
        sym = c["sym"] and i == 0
        if sym:
            # a tile with address 0 below address 1 arrives as the copy of its
            # stored partner, the dims exchanged
            own = np.arange(len(addrs)).reshape(vg)
            src = np.where(addrs[:, 0] < addrs[:, 1],
                           own[addrs[:, 1], addrs[:, 0], addrs[:, 2], addrs[:, 3]], own.ravel())
            x = x.view(len(addrs), -1)[torch.from_numpy(src).to(DEV)].reshape(-1)
        out.append(rrr.TileTensor("aacc" if sym else "cccc", [o, o, v, v], vg, DEV, data=x,
                                  addrs=addrs))
    return out


def _mixed_inputs(c, seed):
    return _normal((c["m"], c["k"]), 4 * seed), _normal((c["n"], c["k"]), 4 * seed + 1)


def _widths(c):
    return [c["w0"], c["w1"], c["w2"], c["w3"]]


def prepare(case, seed):
    c = dict(case)
    _lib.check(_lib.lib().dtcf_init(0))
    kind = c["kind"]
    if kind == "term":
        o, v = c["o"], c["v"]
        sp = dltc.make_space(o, v, o, v)
        A, B = _normal((v ** 4,), 4 * seed), _normal((v * v * o * o,), 4 * seed + 1)
        C = _normal((v * v * o * o,), 4 * seed + 2)
        t = dltc.Term(sp, ["p1", "p2", "h1", "h2"], C, ["p1", "p2", "p3", "p4"], A,
                      ["p3", "p4", "h1", "h2"], B, 0.5)
        return {"c": c, "term": t, "C": C}
    if kind == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"c": c, "A": _normal((m, k), 4 * seed), "B": _normal((k, n), 4 * seed + 1),
                "C": _normal((m, n), 4 * seed + 2)}
    if kind == "step":
        A, B, C = _step_tensors(c, seed)
        st = rrr.LocalStep(A, "i,k,a,c", B, "k,j,c,b", C, "i,j,a,b", mode=c["mode"])
        return {"c": c, "step": st, "C": C.tiles}
    if kind == "d2h":
        sp = blocksparse.Space.seeded(c["o"], c["v"], c["orbitals"])
        ts = [blocksparse.BSTensor(sp, "oovv", DEV) for _ in range(3)]
        for i, t in enumerate(ts):
            t.data = _normal((t.size,), 4 * seed + i)
        term = blocksparse.BlockTerm(ts[2], "ijab", ts[0], "ikac", ts[1], "kjcb", cfg=4)
        return {"c": c, "term": term, "C": ts[2].data}
    if kind == "mixed":
        A, B = _mixed_inputs(c, seed)
        m, n, k = c["m"], c["n"], c["k"]
        # rows: B is stored k x n (its rows contiguous), as amplitudes c,d,i,j are
        bv = mixed.dense_view(n, k, trans=c["rows"])
        st = {"c": c, "A": A, "B": B, "av": mixed.dense_view(m, k), "bv": bv,
              "C": torch.zeros(m * n, dtype=torch.float64, device=DEV)}
        if c["keep_a"]:
            st["sa"] = mixed.Split(c["prec"], A, st["av"], c["ns"])
        return st
    if kind == "permute":
        n = c["ntiles"] * int(np.prod(_widths(c)))
        return {"c": c, "x": _normal((n,), seed), "y": torch.empty(n, dtype=torch.float64, device=DEV),
                "perm": [int(d) for d in c["perm"]]}
    if kind == "amplitudes":
        o, v = c["o"], c["v"]
        n = o * o * v * v
        return {"c": c, "R": _normal((n,), 4 * seed), "V": _normal((n,), 4 * seed + 1),
                "T": torch.empty(n, dtype=torch.float64, device=DEV),
                "eo": _energies(o, 4 * seed + 2, -2.0, -0.5), "ev": _energies(v, 4 * seed + 3, 0.2, 3.0),
                "E": torch.zeros(1, dtype=torch.float64, device=DEV),
                "N": torch.zeros(1, dtype=torch.float64, device=DEV)}
    sizes = _sizes(c)
    lists = [termlist.load("t1"), termlist.load("t2")]
    # the inputs (once more for digits kept of them) and every temporary
    names = {n for tl in lists for n in tl.inputs()}
    every = sum(tl.array_elements(n, sizes) * (0.8 if n in names else 1.3)
                for tl in lists for n in tl.arrays)
    budget = int(8 * every * 1.1) + (1 << 28)
    if kind == "served":
        s = _Served(budget, c["slots"])
        system = serve.System(s.server, 0, 0, lists, seed=seed, sizes=sizes)
        s.programs = [serve.Program(s.server, tl, system) for tl in lists]
        return {"c": c, "served": s, "system": system,
                "outs": [p.new_outputs() for p in s.programs]}
    # an iteration from the first-order amplitudes, at a spread of the
    # integrals for which the iteration converges
    s = _Served(budget, 1)
    system = ccsd.CCSystem(s.server, c["o"], c["v"], seed=seed, sigma=0.5 / c["v"], lists=lists)
    drv = ccsd.UHFCCSD(s.server, system, prec=mixed.I8, nslice=c["ns"], max_level=c["lev"])
    s.programs = drv.progs
    drv.iterate()
    amps = {n: torch.empty(int(np.prod(system.shape[n])), dtype=torch.float64, device=DEV)
            for n in ccsd.AMPS}
    return {"c": c, "served": s, "system": system, "drv": drv, "amps": amps}


def _sizes(c):
    if c["kind"] == "served":
        return {"Oa": c["oa"], "Ob": c["ob"], "Va": c["va"], "Vb": c["vb"]}
    return serve.system_sizes(c["o"], c["v"])


# ---------------------------------------------------------------- one pass
def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "term":
        s["term"].run()
        return s["C"]
    if kind == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return ops.gemm(c["ta"], c["tb"], m, n, k, 1.0, s["A"], m if c["ta"] else k, s["B"],
                        k if c["tb"] else n, s["C"], n)
    if kind == "step":
        s["step"].run(1.0)
        return s["C"]
    if kind == "d2h":
        s["term"].run(1.0)
        return s["C"]
    if kind == "mixed":
        sa = s["sa"] if c["keep_a"] else mixed.Split(c["prec"], s["A"], s["av"], c["ns"])
        sb = mixed.Split(c["prec"], s["B"], s["bv"], c["ns"])
        return mixed.gemm_split(sa, sb, s["C"], ldc=c["n"], max_level=c["lev"])
    if kind == "permute":
        return ops.permute_tiles(s["x"], _widths(c), s["perm"], c["ntiles"], s["y"])
    if kind == "amplitudes":
        T = ops.denom_update(s["R"], s["eo"], s["ev"], s["T"])
        return {"T": T, "energy": ops.energy(s["V"], T, c["o"], c["v"], s["E"]),
                "norm": ops.norm2(s["R"], s["N"])}
    if kind == "served":
        srv = s["served"].server
        rids = [p.submit(o)[0] for p, o in zip(s["served"].programs, s["outs"])]
        for r in rids:
            _lib.check(srv.wait(r, 600000.0))
            srv.release(r)
        return s["outs"]
    rec = s["drv"].iterate()
    for name, t in s["amps"].items():
        serve.copy_device(t.data_ptr(), s["system"].ptr[name], t.numel())
    return {"residuals": s["drv"].res, "amplitudes": s["amps"],
            "energies": {n: rec[n] for n in ccsd.OUT_NAMES}}


# ------------------------------------------------------------------- work
def work(case):
    c = case
    kind = c["kind"]
    if kind in ("gemm", "term", "mixed"):
        m, n, k = ((c["v"] ** 2, c["o"] ** 2, c["v"] ** 2) if kind == "term"
                   else (c["m"], c["n"], c["k"]))
        f, b = 2.0 * m * n * k, 8.0 * (m * k + n * k + 2 * m * n)
        if kind == "mixed":
            f *= mixed.n_products(c["prec"], c["ns"], c["lev"])
            if c["keep_a"]:  # the kept digits in place of the operand
                b -= m * k * (8.0 - (c["ns"] if c["prec"] == mixed.I8 else 6))
        return {"bytes": b, "flops": f}
    if kind == "step":
        n = float(c["o"] * c["v"])
        return {"bytes": 8 * 4 * n ** 2, "flops": 2 * n ** 3}
    if kind == "d2h":
        sp = blocksparse.Space.seeded(c["o"], c["v"], c["orbitals"])
        n = sum(float(_class(sp, h)) ** 2 for h in range(8))
        f = sum(2.0 * float(_class(sp, h)) ** 3 for h in range(8))
        return {"bytes": 8 * 4.0 * n, "flops": f}
    if kind == "permute":
        n = float(c["ntiles"]) * float(np.prod(_widths(c)))
        return {"bytes": 16 * n, "flops": 0.0}
    if kind == "amplitudes":
        n = float(c["o"] * c["v"]) ** 2
        return {"bytes": 8 * 3 * n, "flops": 10 * n}
    sizes = _sizes(c)
    f = b = 0.0
    seen = set()
    for tl in (termlist.load("t1"), termlist.load("t2")):
        f += sum(st.dense_flops(sizes) for st in tl.statements)
        for n in tl.inputs() + tl.outputs():
            if n not in seen:
                seen.add(n)
                b += 8.0 * tl.array_elements(n, sizes)
    return {"bytes": b, "flops": f}


def _class(sp, h):
    """Pairs (occupied, virtual) whose irreps multiply to h."""
    return sum(sp.counts["o"][g] * sp.counts["v"][g ^ h] for g in range(8))


# ------------------------------------------------------------------ exact
def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "term":
        o, v = c["o"], c["v"]
        A = _normal((v ** 4,), 4 * seed).view(v * v, v * v)
        B = _normal((v * v * o * o,), 4 * seed + 1).view(v * v, o * o)
        return (_normal((v * v * o * o,), 4 * seed + 2).view(v * v, o * o) + 0.5 * (A @ B)).reshape(-1)
    if kind == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        A, B = _normal((m, k), 4 * seed), _normal((k, n), 4 * seed + 1)
        A = A.view(k, m).t().contiguous() if c["ta"] else A.view(m, k)
        B = B.view(n, k).t().contiguous() if c["tb"] else B.view(k, n)
        return (_normal((m, n), 4 * seed + 2).view(m, n) + A @ B).reshape(-1)
    if kind == "step":
        return _exact_step(c, seed)
    if kind == "d2h":
        return _exact_d2h(c, seed)
    if kind == "mixed":
        A, B = _mixed_inputs(c, seed)
        m, n, k = c["m"], c["n"], c["k"]
        B = B.view(k, n) if c["rows"] else B.view(n, k).t().contiguous()
        return (A.view(m, k) @ B).reshape(-1)
    if kind == "permute":
        n = c["ntiles"] * int(np.prod(_widths(c)))
        x = _normal((n,), seed).view(c["ntiles"], *_widths(c))
        return x.permute(0, *[1 + int(d) for d in c["perm"]]).contiguous().reshape(-1)
    if kind == "amplitudes":
        o, v = c["o"], c["v"]
        R, V = _normal((v, v, o, o), 4 * seed), _normal((o, o, v, v), 4 * seed + 1)
        eo, ev = _energies(o, 4 * seed + 2, -2.0, -0.5), _energies(v, 4 * seed + 3, 0.2, 3.0)
        T = R.view(v, v, o, o) / (eo[:, None] + eo[None, :] - ev[:, None, None, None]
                                  - ev[None, :, None, None])
        E = 0.25 * (V.view(o * o, v * v).t() * T.view(v * v, o * o)).sum()
        return {"T": T.reshape(-1), "energy": E.reshape(1), "norm": R.square().sum().sqrt().reshape(1)}
    return None


def _exact_step(c, seed):
    o, v, vo, vv = c["o"], c["v"], c["vo"], c["vv"]
    vg, br = (vo, vo, vv, vv), (o // vo, o // vo, v // vv, v // vv)

    def dense(i, sym):
        x = _normal((o * o * v * v,), 4 * seed + i).view(*vg, *br)
        if sym:  # tiles below the diagonal of the first two addresses, exchanged, no sign
            for a in range(vo):
                for b in range(a):
                    x[b, a] = x[a, b].transpose(2, 3)
        return x.permute(0, 4, 1, 5, 2, 6, 3, 7).reshape(o, o, v, v)

    n = o * v
    A = dense(0, c["sym"]).permute(0, 2, 1, 3).reshape(n, n)  # i,a x k,c
    B = dense(1, False).permute(0, 2, 1, 3).reshape(n, n)     # k,c x j,b
    C = dense(2, False).contiguous()
    C += (A @ B).view(o, v, o, v).permute(0, 2, 1, 3)
    return C.view(vo, br[0], vo, br[1], vv, br[2], vv, br[3]).permute(
        0, 2, 4, 6, 1, 3, 5, 7).reshape(-1)


def _exact_d2h(c, seed):
    sp = blocksparse.Space.seeded(c["o"], c["v"], c["orbitals"])
    co, cv = sp.counts["o"], sp.counts["v"]
    keys = [(p, q, r, p ^ q ^ r) for p in range(8) for q in range(8) for r in range(8)]
    shape = {g: (co[g[0]], co[g[1]], cv[g[2]], cv[g[3]]) for g in keys}

    def blocks(i):
        x = _normal((sum(int(np.prod(shape[g])) for g in keys),), 4 * seed + i)
        out, at = {}, 0
        for g in keys:
            n = int(np.prod(shape[g]))
            out[g] = x[at:at + n].view(shape[g])
            at += n
        return out, x

    A, B, (C, flat) = blocks(0)[0], blocks(1)[0], blocks(2)
    for h in range(8):
        ov = [(p, p ^ h) for p in range(8)]  # pairs (occupied, virtual) of class h
        Ah = torch.cat([torch.cat([A[i, k, a, d].permute(0, 2, 1, 3).reshape(co[i] * cv[a], -1)
                                   for k, d in ov], 1) for i, a in ov], 0)
        Bh = torch.cat([torch.cat([B[k, j, d, b].permute(0, 2, 1, 3).reshape(co[k] * cv[d], -1)
                                   for j, b in ov], 1) for k, d in ov], 0)
        Ch = Ah @ Bh
        r = 0
        for i, a in ov:
            q = 0
            for j, b in ov:
                blk = Ch[r:r + co[i] * cv[a], q:q + co[j] * cv[b]]
                C[i, j, a, b] += blk.reshape(co[i], cv[a], co[j], cv[b]).permute(0, 2, 1, 3)
                q += co[j] * cv[b]
            r += co[i] * cv[a]
    return flat
