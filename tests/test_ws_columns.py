"""Wave-subtree plans whose top rows outnumber the free places of the waves:
the kernels' waves move 64 * ws_cols columns each, and a plan is given only
where these cover the whole solution.

Two arms of 62 sections on a core of small resistors fill two waves of 64
rows, with five top rows of which two have a place there: the last two of the
130 columns had no lane (their results were left as they were)."""
import numpy as np
import pytest

import plan_emulator as pe
from test_ws_plan import WsPlan


def two_arms(a0, a1, r=3e-4):
    """A capacitor at four of five nodes: one element per lane, so that one row per lane is what is launched."""
    t = [f"RT x0 x1 {r}", f"RV x0 x2 {r}", "LT x0 x3 1u", "RL x3 0 1k", "V0 x2 0 PULSE(0 1 0 0 0 1 1) AC 1"]
    for a, (p, n) in enumerate((("x0", a0), ("x1", a1))):
        for k in range(n):
            t.append(f"R{a}_{k} {p} c{a}_{k} {50 + k}")
            if k % 5:
                t.append(f"C{a}_{k} c{a}_{k} 0 {(1 + 0.01 * k) * 1e-12!r}")
            p = f"c{a}_{k}"
    return "\n".join(t) + "\n"


def columns(nw, rows):
    rows = 4 if rows == 3 else rows
    return 64 * rows if nw == 1 else 64 * ((rows * nw + nw - 2) // (nw - 1)) * (nw - 1)


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("nw", [1, 2, 4, 8])
def test_every_column_has_a_lane(nw, adjoint):
    import krets_amd as kg
    plans = 0
    for a0 in range(58, 66):
        for a1 in range(58, 66):
            c = kg.Circuit(two_arms(a0, a1))
            P = WsPlan(c, 2e9, nw, adjoint)
            if P.status == 0:
                plans += 1
                assert c.n <= columns(nw, P.h["rows"]), (a0, a1, c.n, P.h)
    assert plans or nw != 2


@pytest.mark.gpu
@pytest.mark.parametrize("tps", [0, 3064, 3128, 3256, 3512])
def test_gpu_every_column_is_written(oracle, tps):
    """Transient and adjoint of the two arms of 62. The step's matrix has a condition number of 1.8e4 with its rows
    scaled (6.7e6 without): 40 steps of rounding are 2e-10 of the solution, gradients take both passes."""
    import torch
    import krets_amd as kg
    print(f"[gpu case] two arms of 62 sections, tps={tps}", flush=True)
    text, h, N = two_arms(62, 62), 1e-9, 40
    c = kg.Circuit(text)
    ctx = kg.Context()
    ctx.load(c.elements, np.repeat(c.params[None], 2, axis=0), c.n)
    cfg = kg.SolverConfig(threads_per_system=tps)
    out = torch.full((2 * (N + 1) * c.n,), float("nan"), dtype=torch.float64, device="cuda:0")
    r, st, _ = ctx.transient(h, N, method=kg.TRAP, config=cfg, out=out)
    assert r == 0 and (st == 0).all()
    x = out.cpu().numpy().reshape(2, N + 1, c.n)
    assert not np.isnan(x).any(), np.flatnonzero(np.isnan(x[0, 1]))
    xr, _ = oracle.Circuit(text).tran(h, N * h, method=kg.TRAP)
    assert max(np.linalg.norm(x[i, k] - xr[k]) / max(np.linalg.norm(xr[k]), 1e-300)
               for i in range(2) for k in range(N + 1)) < 1e-9
    if tps:
        return
    cvec = np.linspace(0.5, 1.0, c.n)
    J, g, st = ctx.adjoint(h, N, cvec, method=kg.TRAP)
    Jr, gr = oracle.Circuit(text).adjoint(h, N, cvec, method=kg.TRAP)
    assert (st == 0).all() and abs(J[0] - Jr) <= 1e-9 * abs(Jr)
    assert np.max(np.abs(g[0] - gr)) < 1e-7 * np.max(np.abs(gr))
