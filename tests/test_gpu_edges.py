"""GPU: the edges of the kernels' splits, against the oracle.

Sizes one below, at and one above what a wave, a quad of lanes or a block of
rows holds. Tolerances are those of the same comparisons at the sizes of
tests/test_gpu_parity.py and tests/test_gpu_adjoint.py: FP64 solves of these
ladders 1e-12 (1e-11 over many transient steps of long ladders), mixed
precision its promised 1e-9, Newton waveforms 1e-9.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu case] {msg}", flush=True)
    sys.stdout.flush()


def nerr(x, r):
    d = np.linalg.norm(r)
    return np.linalg.norm(x - r) / (d if d > 0 else 1.0)


@pytest.fixture(scope="module")
def kg():
    import krets_amd
    return krets_amd


# unknowns = sections + 2: every remainder of a group of four; systems: one,
# a wave but for one lane, a wave, one more, and a second instance block
@pytest.mark.parametrize("sections", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("precision,tps", [(0, 2001), (0, 2011), (1, 2001), (1, 2002), (1, 2012)])
def test_ac_lane_quads(kg, oracle, sections, precision, tps):
    from krets_amd import workloads as W
    tol = 1e-12 if precision == 0 else 1e-9
    for ni, nf in [(1, 1), (9, 7), (1, 64), (13, 5), (65, 3)]:
        say(f"AC lanes sections={sections} precision={precision} tps={tps} {ni} x {nf}")
        b = W.c2_rc_ladder_mc(ni, sections=sections, seed=41)
        f = np.geomspace(10.0, 1e5, nf)
        ctx = kg.Context()
        b.load(ctx)
        xs, st, _ = ctx.ac_sweep(f, precision=precision, config=kg.SolverConfig(threads_per_system=tps))
        assert (st == 0).all()
        for i in {0, ni // 2, ni - 1}:
            xr = oracle.Circuit(b.netlists[i]).ac(f)
            e = max(nerr(xs[i][j], xr[j]) for j in range(nf))
            assert e < tol, (ni, nf, i, e)


# the looped form: remainders of its four rows a turn, and long chains; more systems than one round of its grid holds
@pytest.mark.parametrize("sections,ni,nf", [(24, 3, 5), (25, 1, 64), (26, 65, 3), (27, 13, 5), (120, 2, 70), (300, 2, 3),
                                            (24, 1400, 100)])
@pytest.mark.parametrize("precision,tps", [(0, 2021), (0, 2031), (1, 2021)])
def test_ac_looped_lanes(kg, oracle, sections, ni, nf, precision, tps):
    from krets_amd import workloads as W
    say(f"looped AC lanes sections={sections} precision={precision} tps={tps} {ni} x {nf}")
    b = W.c2_rc_ladder_mc(ni, sections=sections, seed=43)
    f = np.geomspace(10.0, 1e5, nf)
    ctx = kg.Context()
    b.load(ctx)
    xs, st, _ = ctx.ac_sweep(f, precision=precision, config=kg.SolverConfig(threads_per_system=tps))
    assert (st == 0).all()
    for i in {0, ni // 2, ni - 1}:
        xr = oracle.Circuit(b.netlists[i]).ac(f)
        assert max(nerr(xs[i][j], xr[j]) for j in range(nf)) < 1e-12, i


# unknowns = sections + 2 around multiples of a wave's 64 rows and around the
# 256 rows that one wave can hold
@pytest.mark.parametrize("sections", [1, 2, 61, 62, 63, 126, 127, 190, 253, 254, 255, 300])
@pytest.mark.parametrize("tps", [3064, 3128, 3256, 3512])
def test_wave_subtree_transient_rows(kg, oracle, sections, tps):
    from krets_amd import workloads as W
    say(f"wave subtrees, RC ladder of {sections}, tps={tps}")
    b = W.c5_rc_ladder(2, sections=sections, seed=23)
    ctx = kg.Context()
    b.load(ctx)
    h, n = 1e-9, 130  # two source buffers of 64 steps and a remainder
    if sections + 2 > 4 * (tps - 3000):
        with pytest.raises(kg.KretsGpuError, match="4 rows per thread"):
            ctx.transient(h, n, config=kg.SolverConfig(threads_per_system=tps))
        return
    for method in (kg.TRAP, kg.BE_COMPAT):
        xs, st, _ = ctx.transient(h, n, method=method, config=kg.SolverConfig(threads_per_system=tps))
        assert (st == 0).all()
        for i in range(2):
            xr, _ = oracle.Circuit(b.netlists[i]).tran(h, n * h, method=method)
            e = max(nerr(xs[i][k], xr[k]) for k in range(n + 1))
            assert e < 1e-11, (i, method, e)


@pytest.mark.parametrize("sections", [1, 2, 20, 21, 62, 84, 85])  # 3 s + 2 unknowns
@pytest.mark.parametrize("tps", [3064, 3128, 3256, 3512])
def test_wave_subtree_adjoint_rows(kg, oracle, sections, tps):
    from krets_amd import workloads as W
    say(f"wave subtree adjoint, RLC ladder of {sections}, tps={tps}")
    b = W.c3_rlc_uneven(2, smin=sections, smax=sections, seed=29)
    c0 = kg.Circuit(b.netlists[0])
    el, n = c0.elements, c0.n
    pr = np.stack([kg.Circuit(t).params for t in b.netlists])
    ctx = kg.Context()
    ctx.load(el, pr, n)
    c = np.zeros(n)
    c[c0.names.index(f"V(n{sections})")] = 1.0
    h, N = 1e-11, 200
    if n > 4 * (tps - 3000):
        with pytest.raises(kg.KretsGpuError, match="a fitting system"):
            ctx.adjoint(h, N, c, method=kg.TRAP, config=kg.SolverConfig(compat=False, threads_per_system=tps))
        return
    J, g, st = ctx.adjoint(h, N, c, method=kg.TRAP, checkpoint_every=64,
                           config=kg.SolverConfig(compat=False, threads_per_system=tps))
    assert (st == 0).all()
    for i in range(2):
        Jr, gr = oracle.Circuit(b.netlists[i]).adjoint(h, N, c, method=kg.TRAP)
        assert abs(J[i] - Jr) <= 1e-11 * abs(Jr)
        assert np.max(np.abs(g[i] - gr)) < 1e-9 * np.max(np.abs(gr)), i


# instances around one, two and four a wave (one wave per CU: 256 waves)
@pytest.mark.parametrize("ni", [1, 2, 63, 255, 256, 257, 511, 513, 1025])
def test_lane_transients_spread(kg, oracle, ni):
    from krets_amd import workloads as W
    say(f"lane transients, {ni} rectifiers")
    b = W.c4_rectifier(ni, seed=4)
    ctx = kg.Context()
    b.load(ctx)
    tol = dict(voltage_absolute_tolerance=1e-9, current_absolute_tolerance=1e-12, threads_per_system=2001)
    ocfg = oracle.config(vabstol=1e-9, iabstol=1e-12)
    h, n = 1e-6, 130
    xs, st, (it, _) = ctx.transient(h, n, method=kg.BE_COMPAT, config=kg.SolverConfig(**tol))
    assert (st == 0).all()
    args = (2e-4, 1e-6, 1e-14, 5e-5, 1e-3, 1e-6)
    t, xl, npts, nt, rej = ctx.transient_lte(*args, 1000, kg.SolverConfig(compat=False, **tol))
    for i in {0, ni // 2, ni - 1}:
        oc = oracle.Circuit(b.netlists[i])
        xr, itr = oc.tran(h, n * h, method=kg.BE_COMPAT, cfg=ocfg)
        assert np.array_equal(it[i][1:], itr[1:]), i
        # the state at zero bias is a rounding residue (1e-31 V): no relative figure there
        assert np.max(np.abs(xs[i][0])) < 1e-12 and np.max(np.abs(xr[0])) < 1e-12
        assert max(nerr(xs[i][k], xr[k]) for k in range(1, n + 1)) < 1e-9, i
        tr, xr, ntr, rejr = oc.tran_lte(*args, cfg=ocfg)
        assert npts[i] == len(tr) and nt[i] == ntr and rej[i] == rejr, i
        assert np.max(np.abs(t[i][:npts[i]] - tr)) <= 1e-9 * args[0]


# host results below, at and above the sizes that go through the copying threads, and with a ragged last chunk
@pytest.mark.parametrize("ni,steps", [(1, 50), (175, 1000), (300, 1001), (513, 1999)])
def test_large_host_results_match_device(kg, ni, steps):
    import torch
    from krets_amd import workloads as W
    say(f"host results of {ni} rectifiers, {steps} steps")
    b = W.c4_rectifier(ni, seed=4)
    ctx = kg.Context()
    b.load(ctx)
    cfg = kg.SolverConfig(voltage_absolute_tolerance=1e-9, current_absolute_tolerance=1e-12, threads_per_system=2001)
    xs, st, _ = ctx.transient(1e-6, steps, method=kg.BE_COMPAT, config=cfg)
    dev = torch.zeros(ni * (steps + 1) * 3, dtype=torch.float64, device="cuda:0")
    ctx.transient(1e-6, steps, method=kg.BE_COMPAT, config=cfg, out=dev)
    assert (st == 0).all()
    assert np.array_equal(np.asarray(xs).reshape(-1), dev.cpu().numpy())
