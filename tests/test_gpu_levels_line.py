"""GPU: systems on both sides of the size from which 64 threads and more factor
by pivot levels (9 unknowns), against the row-by-row mapping of 16 threads and
the oracle. Both subtract in the same order; tolerance 1e-12 normwise, as for
FP64 solves of these sizes elsewhere (Newton iterations 1e-9)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def chain(n, diodes):
    """n unknowns: a source, its branch and n - 2 RC sections, a diode at every fourth node."""
    t = ["V1 x0 0 0.7 SIN(0.7 1 1k 0 0 0) AC 1"]
    for k in range(n - 2):
        t += [f"R{k} x{k} x{k + 1} {100 + k}", f"C{k} x{k + 1} 0 1u"]
        if diodes and k % 4 == 3:
            t.append(f"D{k} x{k + 1} 0 DM")
    return "\n".join(t + [".model DM D (is=1e-14 n=1)"] * diodes) + "\n"


def near(a, b, tol):
    a, b = np.asarray(a), np.asarray(b)
    assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b), np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n", [8, 9, 10, 33, 64, 65])
@pytest.mark.parametrize("tps", [64, 256])
def test_levels_and_rows(oracle, n, tps):
    import krets_amd as kg
    print(f"[gpu case] factorisation by levels, {n} unknowns, tps={tps}", flush=True)
    f, tol = np.geomspace(10.0, 1e5, 7), dict(voltage_absolute_tolerance=1e-9, current_absolute_tolerance=1e-12)
    for diodes in (0, 1):
        text = chain(n, diodes)
        c, o = kg.Circuit(text), oracle.Circuit(text)
        ocfg = oracle.config(vabstol=1e-9, iabstol=1e-12)
        ctx = kg.Context()
        ctx.load(c.elements, np.repeat(c.params[None], 3, axis=0), c.n)
        got = []
        for t in (tps, 16):
            cfg = kg.SolverConfig(threads_per_system=t, **tol)
            lte = kg.SolverConfig(threads_per_system=t, compat=False, **tol)
            xo, so, _ = ctx.op(cfg)
            xa, sa, _ = ctx.ac_sweep(f, config=cfg)
            xt, st, _ = ctx.transient(1e-5, 20, method=kg.BE_COMPAT, config=cfg)
            xl = ctx.transient_lte(2e-4, 1e-6, 1e-14, 5e-5, 1e-3, 1e-6, 400, lte)
            assert not (so.any() or sa.any() or st.any())
            got.append((xo[2], xa[2], xt[2], xl[1][2][:xl[2][2]]))
        for a, b in zip(*got):
            near(a, b, 1e-12)
        near(got[0][0], o.op(ocfg)[0], 1e-9 if diodes else 1e-12)
        near(got[0][2], o.tran(1e-5, 2e-4, method=kg.BE_COMPAT, cfg=ocfg)[0], 1e-9 if diodes else 1e-12)
        near(got[0][1], o.ac(f, cfg=ocfg), 1e-9 if diodes else 1e-12)
