"""CPU: the plan's factorisation by pivot levels against its row-by-row factor
program. Both subtract the same products from a slot in the same order, so in
plain FP64 (no fused operations) the factors and the forward substitution agree
bit for bit; every index stays inside its array, and no entry of a level reads
what the same level writes."""
import numpy as np
import pytest

import plan_emulator as pe
from conftest import active_netlist


def netlists():
    from krets_amd import workloads as W
    rng = np.random.default_rng(9)
    mesh = ["V1 n0_0 0 1"]
    for i in range(6):
        for j in range(6):
            if i < 5:
                mesh.append(f"RA{i}{j} n{i}_{j} n{i + 1}_{j} {rng.uniform(10, 99)}")
            if j < 5:
                mesh.append(f"RB{i}{j} n{i}_{j} n{i}_{j + 1} {rng.uniform(10, 99)}")
            mesh.append(f"RC{i}{j} n{i}_{j} 0 1000")
    return {"divider": "V1 a 0 1\nR1 a b 10\nR2 b 0 10\n", "rc70": W.c2_rc_ladder_mc(1, sections=70, seed=1).netlists[0],
            "rlc33": W.c3_rlc_uneven(1, smin=33, smax=33, seed=2).netlists[0], "mesh": "\n".join(mesh) + "\n",
            "rectifier": W.c4_rectifier(1).netlists[0], "active": active_netlist()}


@pytest.mark.parametrize("kind", [pe.DC, pe.AC, pe.TRAN])
@pytest.mark.parametrize("name", ["divider", "rc70", "rlc33", "mesh", "rectifier", "active"])
def test_levels_match_rows(name, kind):
    import krets_amd as kg
    from krets_amd import _lib
    text = netlists()[name]
    c = kg.Circuit(text)
    p = pe.Plan(c.elements, c.n, kind, pe.NESTED, c.params, 1e6)
    if p.status:
        pytest.skip("structurally singular")
    lay = np.zeros(64, np.int32)
    el, pr = np.ascontiguousarray(c.elements), np.ascontiguousarray(c.params)
    _lib.lib().kg_plan_export(el.ctypes.data, len(el), c.n, kind, pe.NESTED, pr.ctypes.data, 1e6, None, 0,
                              lay.ctypes.data, 64)
    ncr, ol, oe, op, os_ = (int(v) for v in lay[len(pe.FIELDS):len(pe.FIELDS) + 5])
    n, nnz, b = p.n, p.nnz, p.b
    rp, col, dg = p.row_ptr, p.col, p.diag
    assert ncr > 0 and ol >= p.L["total"]
    rng = np.random.default_rng(5)
    v0 = rng.standard_normal(nnz)
    v0[dg] += 8.0
    w0 = rng.standard_normal(n)
    # rows
    v, w = v0.copy(), w0.copy()
    fptr = p.arr("fprog_ptr", n + 1)
    for i in range(n):
        fp = p.L["o_fprog"] + int(fptr[i])
        nk = int(b[fp])
        fp += 1
        for _ in range(nk):
            sik, sdk, nu = (int(x) for x in b[fp:fp + 3])
            fp += 3
            v[sik] = v[sik] * v[sdk]
            for _ in range(nu):
                v[b[fp]] = v[b[fp]] - v[sik] * v[b[fp + 1]]
                fp += 2
        v[dg[i]] = 1.0 / v[dg[i]]
    for i in range(n):
        for q in range(rp[i], dg[i]):
            w[i] = w[i] - v[q] * w[col[q]]
    # levels: reads of a phase see the values from before it
    x, y = v0.copy(), w0.copy()
    lvl = b[ol:ol + 3 * ncr + 3]
    npair = int(b[oe + 2 * int(lvl[3 * ncr]) + 1])
    for l in range(ncr):
        vals = np.concatenate([x, y])
        new = {}
        for e in range(lvl[3 * l], lvl[3 * l + 3]):
            code, p0, p1 = int(b[oe + 2 * e]), int(b[oe + 2 * e + 1]), int(b[oe + 2 * e + 3])
            s = code & 0xffff
            assert s < nnz + n and s not in new and 0 <= p0 <= p1 <= npair
            assert (s >= nnz) == (e >= lvl[3 * l + 1])
            acc = vals[s]
            for q in range(p0, p1):
                u = int(b[op + q]) & 0xffffffff
                acc = acc - vals[u & 0xffff] * vals[u >> 16]
            new[s] = 1.0 / acc if code & 0x10000 else acc
        for s, a in new.items():
            if s < nnz:
                x[s] = a
            else:
                y[s - nnz] = a
        for q in range(lvl[3 * l + 2], lvl[3 * l + 5]):
            u = int(b[os_ + q]) & 0xffffffff
            x[u & 0xffff] = x[u & 0xffff] * x[u >> 16]
    assert np.array_equal(x, v) and np.array_equal(y, w)
