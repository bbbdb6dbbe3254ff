"""GPU: linear transients and adjoints of meshes, against the oracle.

Meshes couple rows to more than two rows of one elimination level: they do not
take the wave-subtree form and stay with the LDS-resident kernels (k_tran_lin,
k_adj_lin_*), which each case shows by the kernels' names. Sizes around one,
two and four rows per thread. Tolerances: those of the same comparisons on
ladders (tests/test_gpu_edges.py).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu case] {msg}", flush=True)


@pytest.fixture(scope="module")
def kg():
    import krets_amd
    return krets_amd


def mesh(seed, instance, k, stubs, loads=0):
    """k x k nodes, capacitors to ground, resistors between neighbours, a driven corner; `stubs` inductors from nodes of
    the mesh to loaded nodes of their own (two unknowns each), `loads` resistors to such nodes (one). Instances differ
    by up to 1 %: they share one static pivot order."""
    rng, rel = np.random.default_rng(seed), np.random.default_rng((seed, instance))
    u = lambda a, b: repr(rng.uniform(a, b) * rel.uniform(0.99, 1.01))
    t = ["* mesh", "V1 in 0 PULSE(0 1 0 1n 1n 20n 1)", f"RS in a0_0 {u(20, 60)}"]
    for i in range(k):
        for j in range(k):
            t.append(f"C{i}_{j} a{i}_{j} 0 {u(1e-12, 3e-12)}")
            if i + 1 < k:
                t.append(f"RV{i}_{j} a{i}_{j} a{i + 1}_{j} {u(50, 100)}")
            if j + 1 < k:
                t.append(f"RH{i}_{j} a{i}_{j} a{i}_{j + 1} {u(50, 100)}")
    for s in range(stubs + loads):
        a = f"a{s * 5 % k}_{s * 3 % k}"
        t.append(f"LT{s} {a} b{s} {u(1e-9, 5e-9)}" if s < stubs else f"RT{s} {a} b{s} {u(50, 100)}")
        t += [f"CT{s} b{s} 0 {u(1e-12, 3e-12)}", f"RL{s} b{s} 0 {u(200, 400)}"]
    return "\n".join(t) + "\n"


def batch(kg, ni, n, seed):
    """ni meshes of exactly n unknowns, at least four inductors. The seed: the first whose operating points the
    static-pivot guard (1e-9) lets pass by a factor of two (inductors are shorts there)."""
    import plan_emulator as pe
    from test_plan import values

    def bound(text):
        c = kg.Circuit(text)
        return pe.static_pivot_bound(pe.Plan(c.elements, c.n, pe.DC, pe.NESTED, c.params, 0.0), values(c, pe.DC)[0])
    k = 2
    while (k + 1) ** 2 + 2 + 8 <= n:
        k += 1
    rest = n - k * k - 2
    make = lambda i: mesh(seed, i, k, rest // 2, rest % 2)
    while max(bound(make(i)) for i in range(2)) > 5e-10:
        seed += 1
    nets = [make(i) for i in range(ni)]
    cs = [kg.Circuit(t) for t in nets]
    assert cs[0].n == n and rest // 2 >= 4 and not any((c.elements != cs[0].elements).any() for c in cs)
    ctx = kg.Context()
    ctx.load(cs[0].elements, np.stack([c.params for c in cs]), n)
    return ctx, nets, cs[0]


def names(ctx, f):
    ctx.profile(True)
    r = f()
    k = set(ctx.profile_summary())
    ctx.profile(False)
    return r, k


@pytest.mark.parametrize("tps,n", [(3064, 30), (3064, 63), (3064, 64), (3064, 65), (3064, 128), (3064, 129), (3064, 256),
                                   (3128, 127), (3128, 128), (3128, 129), (3128, 257), (3256, 60), (3256, 256),
                                   (3256, 257), (3512, 200), (3512, 257), (4024, 257)])
def test_mesh_transient(kg, oracle, tps, n):
    say(f"mesh transient, {n} unknowns, tps={tps}")
    ctx, nets, _ = batch(kg, 2, n, seed=n)
    h, N = 1e-10, 130
    for method in (kg.TRAP, kg.BE, kg.BE_COMPAT):
        cfg = kg.SolverConfig(compat=method == kg.BE_COMPAT, threads_per_system=tps)
        (xs, st, _), k = names(ctx, lambda: ctx.transient(h, N, method=method, config=cfg))
        assert (st == 0).all() and "k_tran_lin" in k and "k_tran_ws" not in k, k
        for i in range(2):
            xr, _ = oracle.Circuit(nets[i]).tran(h, N * h, method=method)
            e = max(np.linalg.norm(xs[i][s] - xr[s]) / max(np.linalg.norm(xr[s]), 1e-300) for s in range(1, N + 1))
            assert e < 1e-11, (i, method, e)


def test_mesh_too_large_for_its_block(kg):
    ctx, _, _ = batch(kg, 1, 257, seed=1)
    with pytest.raises(kg.KretsGpuError, match="4 rows per thread"):
        ctx.transient(1e-10, 10, config=kg.SolverConfig(threads_per_system=3064))


def check_adjoint(kg, oracle, ctx, nets, c, N, tps, every, h=1e-10):
    cvec = np.random.default_rng(7).uniform(0.5, 1.0, c.n)
    cfg = kg.SolverConfig(compat=False, threads_per_system=tps)
    for method in (kg.TRAP, kg.BE):
        (J, g, st), k = names(ctx, lambda: ctx.adjoint(h, N, cvec, method=method, checkpoint_every=every, config=cfg))
        assert (st == 0).all() and {"k_adj_lin_fwd", "k_adj_lin_bwd"} <= k and "k_tran_ws" not in k, k
        for i in range(len(nets)):
            Jr, gr = oracle.Circuit(nets[i]).adjoint(h, N, cvec, method=method)
            assert abs(J[i] - Jr) <= 1e-11 * abs(Jr), i
            assert np.max(np.abs(g[i] - gr)) < 1e-9 * np.max(np.abs(gr)), i
    return k


@pytest.mark.parametrize("tps,n", [(3064, 64), (3064, 65), (3064, 128), (3064, 129), (3064, 200), (3256, 64), (3256, 200),
                                   (3512, 65), (3512, 200)])
@pytest.mark.parametrize("every", [1, 7, 64])
def test_mesh_adjoint(kg, oracle, tps, n, every):
    say(f"mesh adjoint, {n} unknowns, tps={tps} checkpoint every {every}")
    ctx, nets, c = batch(kg, 2, n, seed=n)
    k = check_adjoint(kg, oracle, ctx, nets, c, 100, tps, every)
    assert ("k_adj_lin_rec" in k) == (every > 1)


def test_mesh_adjoint_recomputes_segments(kg, oracle):
    """A trajectory of more than a quarter of the free memory: the backward pass recomputes each segment itself."""
    from test_gpu_memory import MB, left
    say("mesh adjoint, segments recomputed in the backward pass")
    ctx, _, c = batch(kg, 64, 64, seed=3)
    N, cvec = 20000, np.zeros(c.n)
    cvec[c.names.index("V(a1_1)")] = 1.0
    cfg = kg.SolverConfig(compat=False, threads_per_system=3256)
    run = lambda n: ctx.adjoint(1e-10, n, cvec, checkpoint_every=1000, config=cfg)
    run(40)  # modules and small buffers
    with left(2000 * MB):  # the trajectory: 64 x 20001 x 64 x 8 bytes = 655 MB
        (J, g, st), k = names(ctx, lambda: run(N))
    assert (st == 0).all() and "k_adj_lin_rec" not in k and "k_adj_lin_bwd" in k, k
    (J2, g2, _), k2 = names(ctx, lambda: run(N))
    assert "k_adj_lin_rec" in k2, k2
    assert np.array_equal(J, J2) and np.max(np.abs(g - g2)) <= 1e-12 * np.max(np.abs(g2))
