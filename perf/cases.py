"""Timed workloads of the MNA backend: operating points, DC sweeps, AC sweeps, transients and adjoint gradients.

A case is a dict of plain values. prepare() draws the element values of its instances and loads them into a Context,
run() makes one pass through the package's public entry points, work() counts the bytes and operations a pass cannot do
without, and exact() computes the same outputs in 64 bits with torch or numpy alone (None where the outputs depend on
the Newton or step-size tolerances and so have no tolerance-free value). The per-instance error figures are not among
the outputs: which bound they hold depends on the work mapping that the autotuner picked.

Kinds and their ranges (draw() spreads over them, by logarithm):

  op          series + shunt resistor ladders, 1-8 instances of 1-1500 sections: operating point, host arrays
  dc          resistor + diode, 1-1024 instances, 11-201 points: DC sweep of the source (krets' I-V curve), host arrays
  ac          RC ladders of 1-200 sections, 1-4096 instances, 10-200 frequencies, FP64 or mixed precision
  tran        RC ladders of 1-200 sections, 1-256 instances, 50-2000 steps, backward Euler as in krets or trapezoidal
  tran_uneven RLC ladders of uneven length (up to 512 sections), 8-512 instances, 50-500 trapezoidal steps
  tran_diode  half-wave rectifiers, 1-1024 instances, 100-2000 backward Euler steps (krets' Newton)
  lte         half-wave rectifiers, 1-1024 instances, 1-5 ms of LTE-controlled backward Euler
  adjoint     RC ladders of 5-200 sections, 4-256 instances, 50-2000 steps: objective and gradient through autograd
"""
import math

import numpy as np
import torch

import krets_amd as kg
from krets_amd import workloads as W
from krets_amd.autograd import TransientObjective

DEV = "cuda:0"


def listed():
    return [
        # a voltage divider's operating point: the smallest call there is, all latency
        dict(name="op_divider", kind="op", sections=1, instances=1),
        # krets' long resistor ladders: one large system
        dict(name="op_ladder_1000", kind="op", sections=1000, instances=1),
        # a diode I-V curve over process variation
        dict(name="dc_diode_curve", kind="dc", instances=256, points=101),
        # krets' AC benchmark: one low-pass filter, 100 frequencies, results on the host
        dict(name="ac_low_pass", kind="ac", sections=1, instances=1, points=100, precision="fp64", outputs="host"),
        # Monte Carlo AC sweep, the headline batch
        dict(name="ac_monte_carlo_mixed", kind="ac", sections=50, instances=4096, points=200, precision="mixed",
             outputs="device"),
        # the same in FP64, at sizes that are no multiple of a wave or a cache line
        dict(name="ac_monte_carlo_fp64", kind="ac", sections=37, instances=1001, points=151, precision="fp64",
             outputs="device"),
        # ladders too long for registers: AC sweep of the 200-section line
        dict(name="ac_long_ladder", kind="ac", sections=200, instances=64, points=101, precision="fp64",
             outputs="device"),
        # krets' transient benchmark: one dual RC ladder, 1000 steps, results on the host
        dict(name="tran_dual_rc", kind="tran", sections=2, instances=1, steps=1000, method="be_compat",
             outputs="host"),
        # uneven RLC ladders, trapezoidal
        dict(name="tran_uneven_rlc", kind="tran_uneven", smin=8, smax=512, instances=512, steps=500),
        # rectifiers, one period of krets' fixed-step Newton
        dict(name="tran_rectifier", kind="tran_diode", instances=1024, steps=1000),
        # rectifiers under step-size control
        dict(name="lte_rectifier", kind="lte", instances=1024, tstop=5e-3),
        # one step of fitting ladder values: objective and gradient, values changing from step to step
        dict(name="adjoint_rc_200", kind="adjoint", sections=200, instances=256, steps=2000, checkpoint_every=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["op", "dc", "ac", "ac", "tran", "tran", "tran_uneven", "tran_diode", "lte", "adjoint"])
    if kind == "op":
        return dict(kind=kind, sections=_log(rng, 1, 1500), instances=_log(rng, 1, 8))
    if kind == "dc":
        return dict(kind=kind, instances=_log(rng, 1, 1024), points=_log(rng, 11, 201))
    if kind == "ac":
        s = _log(rng, 1, 200)
        # long ladders leave the register-resident kernels: fewer of them in a batch
        most = 4096 if s <= 50 else 64
        ni = _log(rng, 1, most)
        return dict(kind=kind, sections=s, instances=ni, points=_log(rng, 10, 200),
                    precision=rng.choice(["fp64", "mixed"]), outputs="host" if ni <= 16 else "device")
    if kind == "tran":
        return dict(kind=kind, sections=_log(rng, 1, 200), instances=_log(rng, 1, 256), steps=_log(rng, 50, 2000),
                    method=rng.choice(["be_compat", "trap"]), outputs=rng.choice(["host", "device"]))
    if kind == "tran_uneven":
        smin = _log(rng, 4, 64)
        return dict(kind=kind, smin=smin, smax=_log(rng, smin + 4, 512), instances=_log(rng, 8, 512),
                    steps=_log(rng, 50, 500))
    if kind == "tran_diode":
        return dict(kind=kind, instances=_log(rng, 1, 1024), steps=_log(rng, 100, 2000))
    if kind == "lte":
        return dict(kind=kind, instances=_log(rng, 1, 1024), tstop=round(rng.uniform(1e-3, 5e-3), 5))
    return dict(kind=kind, sections=_log(rng, 5, 200), instances=_log(rng, 4, 256), steps=_log(rng, 50, 2000),
                checkpoint_every=rng.choice([16, 33, 64]))


# ------------------------------------------------------------------ inputs
def _op_values(c, seed):
    """Series resistors [ni, S] and shunts [ni, S + 1]."""
    rng = np.random.default_rng(seed)
    s, ni = c["sections"], c["instances"]
    return (1e3 * np.exp(0.05 * rng.standard_normal((ni, s))),
            1e3 * np.exp(0.05 * rng.standard_normal((ni, s + 1))))


def _dc_values(c, seed):
    rng = np.random.default_rng(seed)
    ni = c["instances"]
    return 1e3 * np.exp(0.1 * rng.standard_normal(ni)), 1e-12 * np.exp(0.3 * rng.standard_normal(ni))


def _rc_values(c, seed):
    rng = np.random.default_rng(seed)
    s, ni = c["sections"], c["instances"]
    return (1e3 * np.exp(0.05 * rng.standard_normal((ni, s))),
            1e-9 * np.exp(0.10 * rng.standard_normal((ni, s))))


def _rlc_batch(c, seed):
    """The uneven RLC ladder batch; its lengths are the case's, its element values the seed's."""
    b = W.c3_rlc_uneven(c["instances"], c["smin"], c["smax"], seed=3)
    rng = np.random.default_rng(seed)
    for e, lo, hi in ((kg._lib.R, 10, 100), (kg._lib.L, 1e-9, 10e-9), (kg._lib.C, 0.1e-12, 1e-12)):
        of = b.elements["type"] == e
        b.params[of, 0] = rng.uniform(lo, hi, int(of.sum()))
    return b


def _frequencies(c):
    """Log-spaced from 1 Hz to 1 MHz."""
    p = c["points"]
    return 10.0 ** (6.0 * np.arange(p) / (p - 1))


def _rc_params(tmpl, r, cv):
    params = np.repeat(tmpl.params[None], r.shape[0], axis=0)  # element order: V1, R1, C1, R2, C2, ...
    params[:, 1::2, 0] = r
    params[:, 2::2, 0] = cv
    return params


# C4's tolerances: 1 nV and 1 pA
_DIODE_TOL = dict(voltage_absolute_tolerance=1e-9, current_absolute_tolerance=1e-12)
_LTE = (1e-6, 1e-14, 5e-5, 1e-3, 1e-6)  # h0, hmin, hmax, reltol, abstol
_LTE_POINTS = 1000  # accepted points per millisecond that a row has room for


def prepare(case, seed):
    k, st = case["kind"], {"case": dict(case)}
    ctx = st["ctx"] = kg.Context()
    if k == "op":
        r, g = _op_values(case, seed)
        t = kg.Circuit(W.c1_ladder(case["sections"]))  # V1, R1..RS, RS1..RS(S+1)
        p = np.repeat(t.params[None], case["instances"], axis=0)
        p[:, 1:1 + case["sections"], 0] = r
        p[:, 1 + case["sections"]:, 0] = g
        ctx.load(t.elements, p, t.n)
    elif k == "dc":
        r, i_s = _dc_values(case, seed)
        t = kg.Circuit("* diode curve\nV1 in 0 1\nR1 in out 1000\nD1 out 0 DMOD\n.model DMOD D (is=1e-12)\n")
        p = np.repeat(t.params[None], case["instances"], axis=0)
        p[:, 1, 0] = r
        p[:, 2, 0] = i_s
        ctx.load(t.elements, p, t.n)
        st["element"] = t.element_index("V1")
    elif k == "ac":
        r, cv = _rc_values(case, seed)
        t = kg.Circuit(W.c2_netlist(r[0], cv[0]))
        ctx.load(t.elements, _rc_params(t, r, cv), t.n)
        st["freqs"] = _frequencies(case)
        if case["outputs"] == "device":
            st["out"] = torch.empty(case["instances"] * case["points"] * t.n * 2, dtype=torch.float64, device=DEV)
    elif k == "tran":
        r, cv = _rc_values(case, seed)
        t = kg.Circuit(W.c5_netlist(r[0], cv[0]))
        ctx.load(t.elements, _rc_params(t, r, cv), t.n)
        if case["outputs"] == "device":
            st["out"] = torch.empty(case["instances"] * (case["steps"] + 1) * t.n, dtype=torch.float64, device=DEV)
    elif k == "tran_uneven":
        b = _rlc_batch(case, seed)
        b.load(ctx)
        st["out"] = torch.empty(int(b.n_unknowns.sum()) * (case["steps"] + 1), dtype=torch.float64, device=DEV)
    elif k in ("tran_diode", "lte"):
        W.c4_rectifier(case["instances"], seed=seed).load(ctx)
    else:
        r, cv = _rc_values(case, seed)
        t = kg.Circuit(W.c5_netlist(r[0], cv[0]))
        p = _rc_params(t, r, cv)
        c = np.zeros(t.n)
        c[2:] = 1.0 / case["sections"]  # mean node voltage
        st.update(elements=t.elements, params=p, n=t.n, c=c,
                  values=torch.tensor(p[:, :, 0], device=DEV, requires_grad=True))
    return st


_TRAN_H, _ADJ_H, _RLC_H = 5e-8, 1e-9, 10e-12


def run(st):
    c, ctx = st["case"], st["ctx"]
    k = c["kind"]
    if k == "op":
        x, status, it = ctx.op()
        return {"x": x, "status": status, "iterations": it}
    if k == "dc":
        x, status, it = ctx.dc_sweep(st["element"], 0.0, 1.0, 1.0 / (c["points"] - 0.5))
        return {"x": x, "status": status, "iterations": it}
    if k == "ac":
        prec = kg.MIXED if c["precision"] == "mixed" else kg.FP64
        if "out" in st:
            _, status, _ = ctx.ac_sweep(st["freqs"], precision=prec, out=st["out"])
            return {"x": st["out"], "status": status}
        x, status, _ = ctx.ac_sweep(st["freqs"], precision=prec)
        return {"x": x, "status": status}
    if k == "tran":
        m = kg.TRAP if c["method"] == "trap" else kg.BE_COMPAT
        if "out" in st:
            _, status, _ = ctx.transient(_TRAN_H, c["steps"], method=m, out=st["out"])
            return {"x": st["out"], "status": status}
        x, status, (it, _) = ctx.transient(_TRAN_H, c["steps"], method=m)
        return {"x": x, "status": status, "iterations": it}
    if k == "tran_uneven":
        _, status, _ = ctx.transient(_RLC_H, c["steps"], method=kg.TRAP, out=st["out"])
        return {"x": st["out"], "status": status}
    if k == "tran_diode":
        x, status, (it, _) = ctx.transient(1e-6, c["steps"], method=kg.BE_COMPAT,
                                             config=kg.SolverConfig(**_DIODE_TOL))
        return {"x": x, "status": status, "iterations": it}
    if k == "lte":
        room = int(math.ceil(_LTE_POINTS * c["tstop"] * 1e3))
        t, x, npts, newton, rejected, status = ctx.transient_lte(
            c["tstop"], *_LTE, room, kg.SolverConfig(compat=False, **_DIODE_TOL), device=True, with_status=True)
        x.masked_fill_((torch.arange(room, device=t.device) >= npts[:, None])[:, :, None], 0.0)  # rows past the end
        return {"t": t, "x": x, "points": npts, "newton": newton, "rejected": rejected, "status": status}
    st["values"].grad = None
    J = TransientObjective.apply(st["values"], ctx, st["elements"], st["params"], st["n"], _ADJ_H, c["steps"], st["c"],
                                 kg.TRAP, kg.FP64, c["checkpoint_every"])
    J.sum().backward()
    return {"J": J.detach(), "gradient": st["values"].grad}


# ------------------------------------------------------------------ work
def work(case):
    """Each result written once and each element value read once; the operations of a tridiagonal elimination."""
    k, ni = case["kind"], case.get("instances", 1)
    if k == "op":
        n, ne = case["sections"] + 2, 2 * case["sections"] + 2
        return {"bytes": 8.0 * ni * (n + ne), "flops": 8.0 * n * ni}
    if k == "dc":
        return {"bytes": 8.0 * ni * (3 * case["points"] + 4), "flops": 4 * 60.0 * ni * case["points"]}
    if k == "ac":
        n, ne = case["sections"] + 2, 2 * case["sections"] + 1
        return {"bytes": 16.0 * ni * case["points"] * n + 8.0 * ni * ne, "flops": 40.0 * n * ni * case["points"]}
    if k == "tran":
        n, ne = case["sections"] + 2, 2 * case["sections"] + 1
        return {"bytes": 8.0 * ni * (case["steps"] + 1) * n + 8.0 * ni * ne, "flops": 10.0 * n * ni * case["steps"]}
    if k == "tran_uneven":
        n = 3.0 * (case["smin"] + case["smax"]) / 2 + 2
        return {"bytes": 8.0 * ni * ((case["steps"] + 1) * n + n), "flops": 10.0 * n * ni * case["steps"]}
    if k == "tran_diode":
        return {"bytes": 8.0 * ni * (3 * (case["steps"] + 1) + 4), "flops": 2.5 * 80.0 * ni * case["steps"]}
    if k == "lte":
        pts = 66e3 * case["tstop"]  # accepted points, about 1000 Newton solves in 5 ms
        return {"bytes": 8.0 * ni * (4 * pts + 4), "flops": 3.4 * 80.0 * ni * pts}
    n, ne = case["sections"] + 2, 2 * case["sections"] + 1
    # forward and transposed solve, states written and read once
    return {"bytes": 8.0 * ni * (2 * (case["steps"] + 1) * n + 2 * ne), "flops": 2 * 10.0 * n * ni * case["steps"]}


# ------------------------------------------------------------------ 64-bit values
def _dev():
    return torch.device(DEV if torch.cuda.is_available() else "cpu")


def _ladder_inverse(g, cap):
    """Inverses [ni, S, S] of a ladder's node matrices: conductances g [ni, S] in series, cap [ni, S] to ground.
    Elimination of the tridiagonal matrix with the identity's columns as right-hand sides."""
    ni, S = g.shape
    diag = g + torch.cat([g[:, 1:], torch.zeros_like(g[:, :1])], 1) + cap
    eye = torch.eye(S, dtype=g.dtype, device=g.device)
    d, y = [diag[:, :1]], [eye[0].expand(ni, S)]
    for k in range(1, S):
        m = g[:, k:k + 1] / d[-1]
        d.append(diag[:, k:k + 1] - m * g[:, k:k + 1])
        y.append(eye[k] + m * y[-1])
    x = [y[-1] / d[-1]]
    for k in range(S - 2, -1, -1):
        x.append((y[k] + g[:, k + 1:k + 2] * x[-1]) / d[k])
    x.reverse()
    return torch.stack(x, 1)


def _exact_op(case, seed):
    r, s = (torch.from_numpy(a) for a in _op_values(case, seed))
    S, ni = case["sections"], case["instances"]
    y = 1.0 / s[:, S]  # admittance to the right of node S + 1, its shunt included
    ys = [y]
    for k in range(S - 1, -1, -1):
        y = 1.0 / s[:, k] + 1.0 / (r[:, k] + 1.0 / y)
        ys.append(y)
    ys.reverse()
    v = torch.ones(ni, dtype=torch.float64)
    out = [-ys[0], v]
    for k in range(S):
        v = v / (1.0 + r[:, k] * ys[k + 1])
        out.append(v)
    return {"x": torch.stack(out, 1).numpy(), "status": None, "iterations": None}


def _exact_ac(case, seed):
    r, cv = (torch.from_numpy(a).to(_dev()) for a in _rc_values(case, seed))
    w = 2.0 * math.pi * torch.from_numpy(_frequencies(case)).to(_dev())
    S, ni, nf = case["sections"], case["instances"], case["points"]
    ys, y = [None] * S, None
    for k in range(S - 1, -1, -1):
        own = 1j * w[None] * cv[:, k, None]
        y = own if y is None else own + 1.0 / (r[:, k + 1, None] + 1.0 / y)
        ys[k] = y
    x = torch.empty(ni, nf, S + 2, dtype=torch.complex128, device=_dev())
    x[:, :, 0] = -1.0 / (r[:, 0, None] + 1.0 / ys[0])
    x[:, :, 1] = v = torch.ones(ni, nf, dtype=torch.complex128, device=_dev())
    for k in range(S):
        v = v / (1.0 + r[:, k, None] * ys[k])
        x[:, :, 2 + k] = v
    if case["outputs"] == "device":
        return {"x": torch.view_as_real(x).reshape(-1), "status": None}
    return {"x": x.cpu().numpy(), "status": None}


def _exact_tran(case, seed):
    r, cv = (torch.from_numpy(a).to(_dev()) for a in _rc_values(case, seed))
    S, ni, N, trap = case["sections"], case["instances"], case["steps"], case["method"] == "trap"
    g, gc = 1.0 / r, (2.0 if trap else 1.0) * cv / _TRAN_H
    inv = _ladder_inverse(g, gc)
    x = torch.zeros(ni, N + 1, S + 2, dtype=torch.float64, device=_dev())
    v = ic = torch.zeros(ni, S, dtype=torch.float64, device=_dev())
    for k in range(1, N + 1):
        b = gc * v + (ic if trap else 0.0)
        b[:, 0] += g[:, 0]
        vn = torch.bmm(inv, b[:, :, None])[:, :, 0]
        if trap:
            ic = gc * (vn - v) - ic
        v = vn
        x[:, k, 0] = -g[:, 0] * (1.0 - v[:, 0])
        x[:, k, 1] = 1.0
        x[:, k, 2:] = v
    out = {"x": x.reshape(-1) if case["outputs"] == "device" else x.cpu().numpy(), "status": None}
    return out if case["outputs"] == "device" else dict(out, iterations=None)


def _exact_uneven(case, seed):
    dev = _dev()
    b = _rlc_batch(case, seed)  # its values alone: ladder i's rows are V1, R1, L1, C1, R2, ...
    ni, N = case["instances"], case["steps"]
    sec = (np.asarray(b.n_unknowns) - 2) // 3
    m = int(sec.max())
    R, L, C = np.ones((ni, m)), np.ones((ni, m)), np.ones((ni, m))
    for i, s in enumerate(sec):
        p = b.params[b.elem_offset[i] + 1:b.elem_offset[i + 1], 0].reshape(s, 3)
        R[i, :s], L[i, :s], C[i, :s] = p.T
    R, L, C = (torch.from_numpy(a).to(dev) for a in (R, L, C))
    have = torch.arange(m, device=dev)[None] < torch.from_numpy(sec).to(dev)[:, None]
    h = _RLC_H
    zl, gc = 2.0 * L / h, 2.0 * C / h
    g = torch.where(have, 1.0 / (R + zl), torch.zeros_like(R))
    inv = _ladder_inverse(g, gc)
    n = 3 * torch.from_numpy(sec).to(dev) + 2
    off = torch.cumsum(n * (N + 1), 0) - n * (N + 1)
    x = torch.zeros(int((n * (N + 1)).sum()), dtype=torch.float64, device=dev)
    k = torch.arange(m, device=dev)[None]
    row = (off[:, None] + 2 + 3 * k)[have]  # V(m_k), then I(L_k), V(n_k)
    nrow = n[:, None].expand(-1, m)[have]
    v, ic, il, vl = (torch.zeros(ni, m, dtype=torch.float64, device=dev) for _ in range(4))
    for s in range(1, N + 1):
        t = s * h
        vin = t / 1e-9 if t < 1e-9 else 1.0 if t < 11e-9 else max(0.0, 1.0 - (t - 11e-9) / 1e-9)
        j = g * (zl * il + vl)
        b = j - torch.cat([j[:, 1:], torch.zeros_like(j[:, :1])], 1) + gc * v + ic
        b[:, 0] += g[:, 0] * vin
        vn = torch.bmm(inv, b[:, :, None])[:, :, 0]
        left = torch.cat([torch.full_like(vn[:, :1], vin), vn[:, :-1]], 1)
        iln = g * (left - vn) + j
        vm = left - R * iln
        ic, vl, il, v = gc * (vn - v) - ic, vm - vn, iln, vn
        at = row + s * nrow
        x[at], x[at + 1], x[at + 2] = vm[have], il[have], v[have]
        x[off + s * n] = -il[:, 0]
        x[off + s * n + 1] = vin
    return {"x": x, "status": None}


def _exact_adjoint(case, seed):
    r, cv = (torch.from_numpy(a).to(_dev()).requires_grad_() for a in _rc_values(case, seed))
    S, ni, N = case["sections"], case["instances"], case["steps"]
    with torch.enable_grad():
        g, gc = 1.0 / r, 2.0 * cv / _ADJ_H
        inv = _ladder_inverse(g, gc)
        src = torch.cat([g[:, :1], torch.zeros_like(g[:, 1:])], 1)
        v = ic = torch.zeros(ni, S, dtype=torch.float64, device=_dev())
        J = torch.zeros(ni, dtype=torch.float64, device=_dev())
        for s in range(1, N + 1):
            vn = torch.bmm(inv, (gc * v + ic + src)[:, :, None])[:, :, 0]
            ic = gc * (vn - v) - ic
            v = vn
            J = J + (0.5 if s == N else 1.0) * _ADJ_H * v.mean(1)
        gr, gcv = torch.autograd.grad(J.sum(), (r, cv))
    grad = torch.zeros(ni, 2 * S + 1, dtype=torch.float64, device=_dev())
    grad[:, 1::2], grad[:, 2::2] = gr, gcv
    return {"J": J.detach(), "gradient": grad}


def exact(case, seed):
    f = {"op": _exact_op, "ac": _exact_ac, "tran": _exact_tran, "tran_uneven": _exact_uneven,
         "adjoint": _exact_adjoint}.get(case["kind"])
    return f(case, seed) if f else None
