"""GPU: systems that fill a CU's 160 KB of LDS to the last 256 bytes, which the
Newton and transient kernels hold themselves: they go to the global workspace
like larger ones. Ladder lengths whose system and reduction buffer take between
163584 and 163840 bytes, one shorter and one longer, against the oracle with
the bound of the other systems around this size (1e-9)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def batch(sections):
    import krets_amd as kg
    from krets_amd import workloads as W
    b = W.c5_rc_ladder(1, sections=sections, seed=31)
    b.load(ctx := kg.Context())
    return kg, b, ctx


def near(x, r):
    assert np.linalg.norm(np.asarray(x) - r) <= 1e-9 * max(np.linalg.norm(r), 1e-300)


@pytest.mark.parametrize("sections,tps", [(2494, 0), (2495, 0), (2498, 0), (2499, 0), (2527, 256), (2530, 256),
                                          (2551, 64), (2554, 64)])
def test_operating_point_at_the_limit(oracle, sections, tps):
    print(f"[gpu case] operating point, {sections} sections, tps={tps}", flush=True)
    kg, b, ctx = batch(sections)
    text = b.netlists[0].replace("V1 in 0 ", "V1 in 0 2 ")
    c = kg.Circuit(text)
    ctx.load(c.elements, c.params[None], c.n)
    x, st, _ = ctx.op(kg.SolverConfig(threads_per_system=tps))
    assert (st == 0).all()
    near(x[0], oracle.Circuit(text).op()[0])


@pytest.mark.parametrize("sections,tps", [(1188, 256), (1189, 256), (1190, 256), (1191, 256), (1200, 64), (1201, 64)])
def test_transient_at_the_limit(oracle, sections, tps):
    print(f"[gpu case] transient, {sections} sections, tps={tps}", flush=True)
    kg, b, ctx = batch(sections)
    x, st, _ = ctx.transient(1e-9, 12, method=kg.TRAP, config=kg.SolverConfig(threads_per_system=tps))
    xr, _ = oracle.Circuit(b.netlists[0]).tran(1e-9, 12e-9, method=kg.TRAP)
    assert (st == 0).all()
    near(x[0][1:], xr[1:])


@pytest.mark.parametrize("sections,tps", [(1123, 256), (1124, 256), (1133, 64), (1134, 64)])
def test_step_control_at_the_limit(oracle, sections, tps):
    print(f"[gpu case] step control, {sections} sections, tps={tps}", flush=True)
    kg, b, ctx = batch(sections)
    lte = (2e-8, 5e-10, 1e-14, 1e-8, 1e-3, 1e-6, 200)
    t, x, npts, _, _ = ctx.transient_lte(*lte, kg.SolverConfig(compat=False, threads_per_system=tps))
    tr, xr, _, _ = oracle.Circuit(b.netlists[0]).tran_lte(*lte[:-1])
    assert npts[0] == len(tr)
    near(x[0][1:npts[0]], xr[1:])
