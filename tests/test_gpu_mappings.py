"""GPU: a remembered work mapping that a batch does not take.

Mappings are remembered under the batch's sizes, within a context and in the
tune file, so that a batch of equal sizes and another topology finds the
first one's. Where it does not take it, the call tunes again. Each test lets
one topology write the tune file, puts the mapping of the other into it and
runs the second from that file, against the oracle, with the tolerances of
the same comparisons elsewhere.
"""
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu case] {msg}", flush=True)


@pytest.fixture(scope="module")
def kg():
    import krets_amd
    return krets_amd


def rel(x, r):
    return np.linalg.norm(x - r) / max(np.linalg.norm(r), 1e-300)


def ladder(sections=200, shuffled=False, extra=""):
    """RC ladder; shuffled: its capacitors listed in another order; extra: three more conductances ("G", controlled by
    their own voltage) or resistors ("R") per section. Sizes and factor patterns are the same for equal lengths."""
    t, caps, prev = ["V1 in 0 PULSE(0 1 0 0 0 1 1) AC 1"], [], "in"
    for k in range(1, sections + 1):
        t.append(f"R{k} {prev} n{k} {1000 + k}")
        caps.append(f"C{k} n{k} 0 {1e-9 * (1 + 0.01 * k)!r}")
        if not shuffled:
            t.append(caps[-1])
        for j in range(3 if extra else 0):
            t.append(f"{extra}X{k}_{j} n{k} 0 " + (f"n{k} 0 1u" if extra == "G" else "1e6"))
        prev = f"n{k}"
    if shuffled:
        t += [caps[i] for i in np.random.default_rng(1).permutation(sections)]
    return "\n".join(t) + "\n"


def mesh(nx, ny):
    t = ["* grid", "V1 a0_0 0 PULSE(0 1 0 0 0 1 1) AC 1"]
    for i in range(nx):
        for j in range(ny):
            t.append(f"C{i}_{j} a{i}_{j} 0 {1e-9 * (1 + 0.01 * (i + 2 * j))!r}")
            if i + 1 < nx:
                t.append(f"RV{i}_{j} a{i}_{j} a{i + 1}_{j} {900 + 10 * i + j}")
            if j + 1 < ny:
                t.append(f"RH{i}_{j} a{i}_{j} a{i}_{j + 1} {800 + i + 10 * j}")
    return "\n".join(t) + "\n"


def load(kg, ctx, text, ni=2):
    c = kg.Circuit(text)
    ctx.load(c.elements, np.repeat(c.params[None], ni, axis=0), c.n)
    return c


def rewrite(path, subs):
    """Replaces the file's entries whose key begins with a pattern's first item: (key begin, new begin, mapping)."""
    s = path.read_text()
    for old, new, tps in subs:
        s, k = re.subn(rf'"{old}\|([^"#]*)": \d+', rf'"{new}|\1": {tps}', s)
        assert k, (old, s)
    path.write_text(s)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("tps", [2021, 2031])
def test_ac_looped_mapping_of_another_ladder(kg, oracle, tmp_path, monkeypatch, precision, tps):
    say(f"AC mapping {tps} remembered for another ladder, precision={precision}")
    file = tmp_path / "tune"
    monkeypatch.setenv("KRETS_GPU_TUNE_FILE", str(file))
    f = np.geomspace(1e2, 1e5, 40)
    load(kg, (ctx := kg.Context()), ladder())
    ctx.ac_sweep(f, precision=precision)
    rewrite(file, [("ac", "ac", tps)])
    text = ladder(shuffled=True)
    load(kg, (ctx := kg.Context()), text)
    xr = oracle.Circuit(text).ac(f)
    for _ in range(3):  # tuned again, then from the captured graph
        x, st, _ = ctx.ac_sweep(f, precision=precision)
        assert (st == 0).all()
        assert max(rel(x[i][j], xr[j]) for i in range(2) for j in range(len(f))) < (1e-9 if precision else 1e-12)
    assert str(tps) not in re.findall(r'"ac\|[^"]*": (\d+)', file.read_text())


def test_adjoint_waves_of_another_ladder(kg, oracle, tmp_path, monkeypatch):
    say("adjoint waves remembered for another ladder")
    file = tmp_path / "tune"
    monkeypatch.setenv("KRETS_GPU_TUNE_FILE", str(file))
    h, N = 1e-9, 60

    def run(extra):
        c = load(kg, (ctx := kg.Context()), ladder(extra=extra))
        cvec = np.zeros(c.n)
        cvec[c.names.index("V(n3)")] = 1.0
        return ctx, cvec, ctx.adjoint(h, N, cvec, method=kg.TRAP)
    run("G")
    for backward, forward in [(3064, 3256), (3128, 3512), (3256, 3064)]:
        rewrite(file, [("adjb", "adjb", backward), ("adjw", "adjw", forward)])
        ctx, cvec, (J, g, st) = run("R")
        assert (st == 0).all()
        Jr, gr = oracle.Circuit(ladder(extra="R")).adjoint(h, N, cvec, method=kg.TRAP)
        for i in range(2):
            assert abs(J[i] - Jr) <= 1e-9 * abs(Jr)
            assert np.max(np.abs(g[i] - gr)) < 1e-9 * np.max(np.abs(gr))
        ctx.profile(True)  # the wave-subtree passes, not the checkpoints
        ctx.adjoint(h, N, cvec, method=kg.TRAP)
        names = set(ctx.profile_summary())
        ctx.profile(False)
        assert {"k_tran_ws", "k_adj_ws_bwd"} <= names, names
        assert {int(v) for v in re.findall(r'"adj[bw]\|[^"]*": (\d+)', file.read_text())} <= {3256, 3512}


@pytest.mark.parametrize("begin", ["tranw", "tran"])
def test_transient_mapping_of_another_topology(kg, oracle, tmp_path, monkeypatch, begin):
    """One wave holds 256 rows: a mesh of more, which does not take the subtree form, has no kernel of 64 threads."""
    say(f"transient mapping remembered for another topology ({begin})")
    file = tmp_path / "tune"
    monkeypatch.setenv("KRETS_GPU_TUNE_FILE", str(file))
    text, h, N = mesh(5, 54), 1e-9, 20
    load(kg, (ctx := kg.Context()), text)
    ctx.transient(h, N, method=kg.TRAP)
    rewrite(file, [("tran", begin, 3064)])
    load(kg, (ctx := kg.Context()), text)
    xr, _ = oracle.Circuit(text).tran(h, N * h, method=kg.TRAP)
    for _ in range(2):
        x, st, _ = ctx.transient(h, N, method=kg.TRAP)
        assert (st == 0).all()
        assert max(rel(x[i][k], xr[k]) for i in range(2) for k in range(N + 1)) < 1e-11


def test_uneven_transient_mapping_of_other_topologies(kg, oracle, tmp_path, monkeypatch):
    say("uneven transient mapping remembered for other topologies")
    from krets_amd import workloads as W
    file = tmp_path / "tune"
    monkeypatch.setenv("KRETS_GPU_TUNE_FILE", str(file))
    b = W.c3_rlc_uneven(64, smin=90, smax=100, seed=7)  # 272 to 302 unknowns; some lengths take no subtree form
    h, N = 1e-11, 30
    b.load(ctx := kg.Context())
    ctx.transient(h, N, method=kg.TRAP)
    rewrite(file, [("tranw", "tranw", 3064)])
    b.load(ctx := kg.Context())
    x, st, _ = ctx.transient(h, N, method=kg.TRAP)
    assert (st == 0).all()
    for i in (0, 31, 63):
        xr, _ = oracle.Circuit(b.netlists[i]).tran(h, N * h, method=kg.TRAP)
        assert max(rel(x[i][k], xr[k]) for k in range(N + 1)) < 1e-11


def test_checkpointed_adjoint_mapping_of_another_topology(kg, oracle, tmp_path, monkeypatch):
    """A mesh, which the subtree form does not take, with more rows than the remembered block size holds."""
    say("checkpointed adjoint mapping remembered for another topology")
    file = tmp_path / "tune"
    monkeypatch.setenv("KRETS_GPU_TUNE_FILE", str(file))
    text, h, N = mesh(5, 54), 1e-9, 20
    for again in (False, True):
        c = load(kg, (ctx := kg.Context()), text)
        cvec = np.zeros(c.n)
        cvec[c.names.index("V(a2_3)")] = 1.0
        J, g, st = ctx.adjoint(h, N, cvec)
        if not again:
            rewrite(file, [("adjf", "adjf", 3064)])
    Jr, gr = oracle.Circuit(text).adjoint(h, N, cvec, method=kg.TRAP)
    assert (st == 0).all() and abs(J[0] - Jr) <= 1e-9 * abs(Jr)
    assert np.max(np.abs(g[0] - gr)) < 1e-9 * np.max(np.abs(gr))


def test_step_control_mapping_of_another_topology(kg, oracle, tmp_path, monkeypatch):
    """The lane kernel (2001), remembered for a mesh whose state exceeds its registers."""
    say("step-controlled mapping remembered for another topology")
    file = tmp_path / "tune"
    monkeypatch.setenv("KRETS_GPU_TUNE_FILE", str(file))
    text, lte = mesh(5, 54), (1e-7, 1e-9, 1e-14, 1e-8, 1e-3, 1e-6, 400)
    for again in (False, True):
        load(kg, (ctx := kg.Context()), text)
        t, x, npts, _, _ = ctx.transient_lte(*lte, config=kg.SolverConfig(compat=False))
        if not again:
            rewrite(file, [("lte", "lte", 2001)])
    tr, _, _, _ = oracle.Circuit(text).tran_lte(*lte[:-1])
    assert npts[0] == len(tr) and np.max(np.abs(t[0][:npts[0]] - tr)) <= 1e-9 * lte[0]


@pytest.mark.parametrize("ni,want,other", [(1, 2031, 2021), (162, 2031, 2021), (163, 2021, 2031)])
def test_one_looped_kernel_is_tried(kg, ni, want, other):
    """Each form costs a compilation: up to 256 waves of systems (162 x 101) the balanced order, above the other."""
    say(f"looped AC kernels tried for {ni} x 101 systems")
    load(kg, (ctx := kg.Context()), ladder(), ni)
    ctx.ac_sweep(np.geomspace(1e2, 1e5, 101))
    tried = {t for t, _ in ctx.last_autotune()}
    assert want in tried and other not in tried
