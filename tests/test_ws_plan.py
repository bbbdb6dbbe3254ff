"""CPU: the wave-subtree plan of the linear transient kernels (kg_ws.h).

The plan's step loop is run in numpy with the kernel's order of events: the
waves' lower levels, the top rows, the waves' upper levels. Every index is
checked against the array it indexes, and a row may only be read by its own
wave after the level that finishes it, or by the top / below the top."""
import ctypes

import numpy as np
import pytest

import plan_emulator as pe
from test_plan import active_netlist, ladder, read_circuit, values

HDR = ("n nnz ndyn nsrc nw rows elems ntop npart o_wave o_slot o_top o_elem o_src o_pair o_rhs o_cpos nrhs more "
       "top_nl ntel words adjoint pad").split()
SLOT, WAVE, ELEM, TOP_LEVELS = 13, 7, 6, 4
ROW, LEV, PAIR, UC0, UC1, US0, US1, DIAG, RHS, NRHS, PART, NPART, COL = range(SLOT)
AELEM = 9
A_KIND, A_E, A_A, A_B, A_P, A_M, A_H1, A_H2, A_GRAD = range(AELEM)


def levels_kept(q):
    return {0: 9, 1: 3}.get(q // 64, 1)


class WsPlan:
    def __init__(self, c, s_rep, nw, adjoint=False):
        from krets_amd import _lib
        el = np.ascontiguousarray(c.elements, _lib.ELEMENT_DTYPE)
        pr = np.ascontiguousarray(c.params, np.float64)
        f = lambda b, k: _lib.lib().kg_ws_plan_export(el.ctypes.data, len(el), c.n, pr.ctypes.data, s_rep, nw,
                                                      int(adjoint), b, k)
        size = f(None, 0)
        self.status = -size if size < 0 else 0
        if size < 0:
            return
        w = np.zeros(size, np.uint16)
        f(ctypes.c_void_p(w.ctypes.data), size)
        h = self.h = {k: int(v) for k, v in zip(HDR, w[:2 * len(HDR)].view(np.int32))}
        assert h["words"] == size and size % 8 == 0 and h["nw"] == nw
        w = w.astype(np.int64)

        def a(name, k):
            o = h["o_" + name]
            assert 2 * len(HDR) <= o and o + k <= size and o % 4 == 0, name
            return w[o:o + k]
        n, nnz, nh = h["n"], h["nnz"], h["ndyn"] + h["nsrc"]
        self.wave = a("wave", WAVE * nw).reshape(nw, WAVE)
        ns, ne, nv = (int(self.wave[-1, k]) for k in (1, 3, 5))
        ne += h["ntel"]
        assert nv == h["nsrc"] and h["ntel"] <= 64 and h["ntop"] <= 64 and h["adjoint"] == int(adjoint)
        assert adjoint or ne == h["ndyn"]
        self.slot, self.top = a("slot", SLOT * ns).reshape(ns, SLOT), a("top", SLOT * h["ntop"]).reshape(-1, SLOT)
        esz = AELEM if adjoint else ELEM
        self.elem, self.src = a("elem", esz * ne).reshape(ne, esz), a("src", 2 * nv).reshape(nv, 2)
        both = np.concatenate([self.slot, self.top])
        npair = int((both[:, PAIR] + both[:, LEV]).max(initial=0))
        self.pair = a("pair", 4 * npair).reshape(-1, 4)
        self.rhs, cpos = a("rhs", h["nrhs"]), a("cpos", n)
        # indices
        assert np.all(self.pair[:, ::2] <= n) and np.all(self.pair[:, 1::2] <= nnz)
        assert np.all(both[:, RHS] + both[:, NRHS] <= h["nrhs"]) and np.all(self.rhs >> 1 < nh)
        assert h["more"] == int(both[:, NRHS].max(initial=0) > 2)
        assert np.all(both[:, UC0:UC1 + 1] <= n) and np.all(both[:, US0:DIAG + 1] <= nnz)
        rows = np.concatenate([self.slot[self.slot[:, ROW] < n, ROW], self.top[:, ROW]])
        assert np.array_equal(np.sort(rows), np.arange(n)) and np.all(self.top[:, ROW] < n)
        pseudo = self.slot[self.slot[:, ROW] >= n, ROW] - n - 1
        assert np.array_equal(np.sort(pseudo), np.arange(h["npart"]))
        assert np.all(self.top[:, PART] + self.top[:, NPART] <= h["npart"]) and self.top[:, NPART].sum() == h["npart"]
        assert np.all(self.top[:, LEV] <= min(h["top_nl"], TOP_LEVELS)) and h["top_nl"] <= TOP_LEVELS
        if adjoint:
            hs = self.elem[:, [A_H1, A_H2]].ravel()
            assert np.array_equal(np.sort(hs[hs < nh]), np.arange(nh)) and np.all(hs[hs >= nh] == nh + 1)
            assert np.all(self.elem[:, A_A:A_M + 1] <= n) and np.all(self.elem[:, A_KIND] <= 2)
            lead = self.elem[self.elem[:, A_GRAD] == 1, A_E]
            assert len(set(lead.tolist())) == len(lead) and set(lead.tolist()) == set(self.elem[:, A_E].tolist())
        else:
            assert np.array_equal(np.sort(np.concatenate([self.elem[:, 0], self.src[:, 0]])), np.arange(nh))
            assert np.all(self.elem[:, 2:5] <= n) and np.all((self.elem[:, 1] == 1) | (self.elem[:, 1] == 2))
        assert np.array_equal(np.sort(self.src[:, 1]), np.arange(h["nsrc"])) and nh < 1 << 14
        # krets column -> row: the top's from its records, the others' from cpos
        assert np.array_equal(np.flatnonzero(cpos == n), np.sort(self.top[:, COL]))
        self.cpos = cpos.copy()
        self.cpos[self.top[:, COL]] = self.top[:, ROW]
        assert np.array_equal(np.sort(self.cpos), np.arange(n))
        at = [0, 0, 0]
        for r in self.wave:
            assert [r[0], r[2], r[4]] == at and r[5] - r[4] <= 64
            assert r[1] - r[0] <= 64 * h["rows"] and r[3] - r[2] <= 64 * h["elems"]
            at = [int(r[1]), int(r[3]), int(r[5])]
            sl, ev = self.slot[r[0]:r[1]], self.elem[r[2]:r[3]]
            # a wave's elements touch its own unknowns and the top, and its rows read no other wave's histories
            own = set(sl[:, ROW].tolist()) | set(self.top[:, ROW].tolist()) | {n}
            assert own.issuperset(ev[:, [A_A, A_B] if adjoint else [2, 3, 4]].ravel().tolist())
            seen = {int(c) >> 1 for q in sl for c in self.rhs[q[RHS]:q[RHS] + q[NRHS]]}
            mine = ev[:, A_H1:A_H2 + 1].ravel() if adjoint else np.concatenate([ev[:, 0], self.src[r[4]:r[5], 0]])
            assert seen <= set(mine.tolist())
            assert np.all(np.diff(sl[:, LEV]) <= 0) and r[6] == sl[:, LEV].max(initial=0)
            assert np.all(sl[:, LEV] <= [levels_kept(q) for q in range(len(sl))])


def step(P, v, hist, n, load=None):
    """One solve on the plan (transposed for an adjoint plan); v[nnz] = 0, hist[nh] = 0; load: what each row's
    right-hand side has besides its histories. Unknowns not final yet are NaN."""
    h, tr = P.h, P.h["adjoint"]

    def rhs(r):
        base = load[r[ROW]] if load is not None and r[ROW] < n else 0.0
        return base + sum((-1.0 if c & 1 else 1.0) * hist[c >> 1] for c in P.rhs[r[RHS]:r[RHS] + r[NRHS]])

    def lower(recs, levels, y, extra):
        acc = [rhs(r) + e for r, e in zip(recs, extra)]
        for lv in range(levels + 1):
            for k, r in enumerate(recs):
                if r[LEV] == lv:
                    assert not np.isnan(acc[k]), "an entry was read before its row was finished"
            for k, r in enumerate(recs):
                if r[LEV] == lv:
                    if tr and r[ROW] < n:
                        acc[k] *= v[r[DIAG]]
                    y[r[ROW]] = acc[k]
            for k, r in enumerate(recs):
                if lv < r[LEV]:
                    c0, s0, c1, s1 = P.pair[r[PAIR] + lv]
                    acc[k] = acc[k] - v[s0] * y[c0] - v[s1] * y[c1]
        return acc

    def upper(recs, acc, levels, x):
        for lv in range(levels, -1, -1):
            for k, r in enumerate(recs):
                if r[LEV] != lv or r[ROW] >= n:
                    continue
                t = acc[k] - v[r[US0]] * x[r[UC0]] - v[r[US1]] * x[r[UC1]]
                assert not np.isnan(t)
                x[r[ROW]] = t if tr else t * v[r[DIAG]]
    accs, part = [], np.full(h["npart"], np.nan)
    for r in P.wave:  # each wave sees only its own rows
        y = np.full(n + 1 + h["npart"], np.nan)
        y[n] = 0.0
        sl = P.slot[r[0]:r[1]]
        accs.append(lower(sl, r[6], y, [0.0] * len(sl)))
        part = np.where(np.isnan(y[n + 1:]), part, y[n + 1:])
    y = np.full(n + 1, np.nan)
    x = y.copy()
    y[n] = x[n] = 0.0
    acc = lower(P.top, h["top_nl"], y, [part[r[PART]:r[PART] + r[NPART]].sum() for r in P.top])
    upper(P.top, acc, h["top_nl"], x)
    done = x.copy()
    for r, a in zip(P.wave, accs):
        xw = x.copy()
        upper(P.slot[r[0]:r[1]], a, r[6], xw)
        done = np.where(np.isnan(done), xw, done)
    assert not np.isnan(done).any()
    return done


def transient(P, v, params, x0, h, N, alpha, src):
    n, nh = P.h["n"], P.h["ndyn"] + P.h["nsrc"]
    trap = alpha == 2.0
    hist, ed, vo = np.zeros(nh + 1), np.zeros(nh), np.zeros(nh)
    x = np.zeros(n + 1)
    x[P.cpos] = x0

    def update(x, s, first):
        for d, kind, p, m, c, e in P.elem:
            vn = x[p] - x[m]
            if kind == 1:
                cf = alpha * (params[e, 0] / h)
                if trap and not first:
                    ed[d] = cf * (vn - vo[d]) - ed[d]
                vo[d] = vn
                hist[d] = -cf * vn - (ed[d] if trap else 0.0)
            else:
                hist[d] = -alpha * (params[e, 0] / h) * x[c] - (vn if trap else 0.0)
        for d, k in P.src:
            hist[d] = src(k, s)
    update(x, 1, True)
    out = [np.array(x0)]
    for s in range(1, N + 1):
        x = step(P, v, hist, n)
        out.append(x[P.cpos])
        update(x, s + 1, False)
    return np.array(out)


def backward(P, v, params, xs, h, N, alpha, cvec):
    """The kernel's backward pass: gradient per element and dJ/dx_0 (krets numbering)."""
    n, nh, trap = P.h["n"], P.h["ndyn"], alpha == 2.0
    hist, load = np.zeros(nh + 2), np.zeros(n)
    K = len(P.elem)
    sb, gr = np.zeros(K), np.zeros(len(params))
    X = np.concatenate([xs, np.zeros((N + 1, 1))], axis=1)
    d1 = X[N, P.elem[:, A_P]] - X[N, P.elem[:, A_M]]
    for s in range(N - 1, -1, -1):
        load[P.cpos] = (0.5 * h if s + 1 == N else h) * cvec
        hist[nh] = 0.0
        lam = step(P, v, hist, n, load)
        for k, (kind, e, a, b, p, m, h1, h2, lead) in enumerate(P.elem):
            val = params[e, 0]
            cf, z, d0 = alpha * val / h, lam[a] - lam[b] - sb[k], X[s, p] - X[s, m]
            if kind == 0:
                gr[e] += lead * z * d1[k] / val ** 2
            elif kind == 1:
                gr[e] += lead * z * alpha / h * (d0 - d1[k])
                hist[h1] = z * cf * (2.0 if trap and s > 0 else 1.0)
                sb[k] = z if trap else 0.0
            else:
                gr[e] += lead * z * alpha / h * (d1[k] - d0)
                hist[h1], hist[h2] = (-z if trap else 0.0), -cf * z
            d1[k] = d0
    xbar = 0.5 * h * np.asarray(cvec)
    recs = np.concatenate([P.slot[P.slot[:, ROW] < n], P.top])
    for r in recs:
        xbar[r[COL]] += sum((-1.0 if c & 1 else 1.0) * hist[c >> 1] for c in P.rhs[r[RHS]:r[RHS] + r[NRHS]])
    return gr, xbar


def circuit(case):
    import krets_amd as k
    from krets_amd import workloads as W
    if case.startswith("rlc"):
        return ladder(int(case[3:])), 1e-11, 12
    if case.startswith("rc"):
        return W.c5_rc_ladder(1, sections=int(case[2:]), seed=5).netlists[0], 1e-9, 12
    if case == "active":
        return active_netlist(), 2e-6, 30
    return read_circuit(case), 50e-6, 20


@pytest.mark.parametrize("method", [0, 2])
@pytest.mark.parametrize("nw", [1, 2, 4, 8])
@pytest.mark.parametrize("case", ["rc1", "rc9", "rc40", "rc200", "rlc4", "rlc23", "rlc171", "active",
                                  "dual_rc_ladder/dual_rc_ladder.cir", "high_pass_filter/transient.cir"])
def test_ws_plan_step_loop_vs_oracle(oracle, case, nw, method):
    import krets_amd as k
    text, h, N = circuit(case)
    c = k.Circuit(text)
    alpha = 2.0 if method == 2 else 1.0
    plan = pe.Plan(c.elements, c.n, pe.TRAN, pe.NESTED, c.params, alpha / h)
    P = WsPlan(c, alpha / h, nw)
    if P.status:  # more than 4 rows per lane, or a source that two waves of a tiny system would share
        assert P.status == 6 and (c.n > 250 * nw or (nw > 1 and c.n < 64))
        return
    contrib, _ = values(c, pe.TRAN, h=h, alpha=alpha)
    vf = np.append(plan.factor(plan.gather(contrib)[0]).real, 0.0)
    lp = pe.LinPlan(c.elements, c.n, c.params, alpha / h)
    xr, _ = oracle.Circuit(text).tran(h, N * h, method=method)

    def src(i, s):
        kind, e = lp.src[i]
        t = (s - 1 if method == 0 else s) * h
        return pe.wave_value(c.params[e], t) if kind == pe.KG_V else c.params[e, 0]
    x = transient(P, vf, c.params, xr[0], h, N, alpha, src)
    for s in range(N + 1):
        assert np.linalg.norm(x[s] - xr[s]) <= 1e-12 * max(np.linalg.norm(xr[s]), 1e-300) + 1e-300, s


@pytest.mark.parametrize("method", [1, 2])
@pytest.mark.parametrize("nw", [1, 2, 4, 8])
@pytest.mark.parametrize("case", ["rc1", "rc9", "rc40", "rlc4", "rlc23", "active"])
def test_ws_adjoint_vs_oracle(oracle, case, nw, method):
    """The transposed plan's backward pass plus the operating-point term, against the oracle's discrete adjoint."""
    import krets_amd as k
    from krets_amd import workloads as W
    text, h, N = circuit(case)
    if case.startswith("rlc"):  # a pulse, so that the capacitors' gradients are not those of a steady state
        s = int(case[3:])
        text = W.c3_netlist(np.linspace(20, 90, s), np.linspace(2e-9, 9e-9, s), np.linspace(0.2e-12, 0.9e-12, s))
    c = k.Circuit(text)
    alpha = 2.0 if method == 2 else 1.0
    plan = pe.Plan(c.elements, c.n, pe.TRAN, pe.NESTED, c.params, alpha / h)
    P = WsPlan(c, alpha / h, nw, adjoint=True)
    if P.status:  # (the active filter's transposed factors couple three rows of one level)
        assert P.status == 6 and (c.n > 250 * nw or (nw > 1 and c.n < 64) or case == "active")
        return
    contrib, _ = values(c, pe.TRAN, h=h, alpha=alpha)
    vf = np.append(plan.factor(plan.gather(contrib)[0]).real, 0.0)
    oc = oracle.Circuit(text)
    cvec = np.random.default_rng(1).uniform(0.5, 1.0, c.n)
    xr, _ = oc.tran(h, N * h, method=method)
    g, xbar0 = backward(P, vf, c.params, xr, h, N, alpha, cvec)
    A, _ = oc.assemble_dc()
    lam0 = np.linalg.solve(A.T, xbar0)
    at = lambda v, i: v[i] if i >= 0 else 0.0
    for e, el in enumerate(c.elements):
        if el["type"] == 0:
            g[e] += ((at(lam0, el["plus"]) - at(lam0, el["minus"])) * (at(xr[0], el["plus"]) - at(xr[0], el["minus"]))
                     / c.params[e, 0] ** 2)
    _, gr = oc.adjoint(h, N, cvec, method=method)
    assert np.max(np.abs(g - gr)) <= 1e-9 * np.max(np.abs(gr)), np.max(np.abs(g - gr)) / np.max(np.abs(gr))


def test_ws_plan_largest_ladder():
    """The 512-section RLC ladder at eight waves: 7 top rows, at most 4 rows
    per lane, half a CU's LDS."""
    import krets_amd as k
    c = k.Circuit(ladder(512))
    P = WsPlan(c, 2e11, 8)
    h = P.h
    assert P.status == 0 and h["rows"] <= 4 and h["ntop"] == 7
    fac = h["nnz"] + h["n"] + 2
    step = 2 * h["n"] + h["npart"] + 5 + h["ndyn"] + 65 * h["nsrc"] + 2 + 16 * h["ntop"]
    assert 64 + 2 * h["nrhs"] + 16 + 8 * max(fac, step) <= 80 * 1024


def test_ws_plan_declines_meshes():
    """A grid of resistors and capacitors couples rows to more than two rows
    of one level: the plan says so instead of dropping couplings."""
    import krets_amd as k
    lines = ["* grid", "V1 a0_0 0 1"]
    for i in range(6):
        for j in range(6):
            lines.append(f"C{i}_{j} a{i}_{j} 0 1n")
            if i < 5:
                lines.append(f"RV{i}_{j} a{i}_{j} a{i + 1}_{j} 1k")
            if j < 5:
                lines.append(f"RH{i}_{j} a{i}_{j} a{i}_{j + 1} 1k")
    assert WsPlan(k.Circuit("\n".join(lines) + "\n"), 1e6, 1).status == 6
