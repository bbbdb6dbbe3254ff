"""CPU: the looped form of the generated FP64 AC lane kernel (chains too long
for registers), run lane by lane on the host against the oracle.

The lengths cover every remainder of the loop's four rows, on both orders
(one chain from the far end; two chains from both ends), with the source at
either end of the elimination (so that the forward substitution is zero or
not along the chain). The workspace is exactly as large as the launch asks
for, with a guard band behind it. Tolerance: 1e-12 normwise, as for the
register form of the same solves."""
import ctypes
import os
import re
import shutil
import subprocess
import tempfile

import numpy as np
import pytest

from test_jit import HOST_SHIM, ebase, nerr, source

DRIVER = r"""
extern "C" int words() { return KG_LOOP_WORDS; }
extern "C" void run_host(const double* prm, const double* eb, const double* fr, int nf, long long nsys,
                         double* out, int* st, double* err, unsigned long long* fixq, long long fixcap, double* ws,
                         int grid) {
  gridDim.x = grid;
  for (unsigned b = 0; b < gridDim.x; b++)
    for (unsigned t = 0; t < 64; t++) {
      blockIdx.x = b;
      threadIdx.x = t;
      KERNEL(prm, eb, fr, nf, nsys, out, st, err, 2, 0.0, fixq, fixcap, (Z*)ws);
    }
}
"""


def run(src, params, elements, freqs, n, grid):
    d = tempfile.mkdtemp()
    try:
        cpp, so = os.path.join(d, "k.cpp"), os.path.join(d, "k.so")
        name = re.search(r"void __launch_bounds__\(64\) (\w+)\(", src).group(1)
        open(cpp, "w").write(HOST_SHIM + src + DRIVER.replace("KERNEL", name))
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-ffp-contract=off", cpp, "-o", so],
                       check=True, capture_output=True)
        L = ctypes.CDLL(so)
        P, I, Q = ctypes.c_void_p, ctypes.c_int, ctypes.c_longlong
        L.run_host.argtypes = [P, P, P, I, Q, P, P, P, P, Q, P, I]
        ni, nf = params.shape[0], len(freqs)
        prm, eb = np.ascontiguousarray(params), np.ascontiguousarray(ebase(elements, params))
        fr = np.ascontiguousarray(freqs, np.float64)
        nw = 2 * 64 * L.words() * grid
        ws = np.full(nw + 4096, 7.25)
        out = np.full(ni * nf * n * 2 + 64, 7.25)
        st, err = np.zeros(ni, np.int32), np.zeros(ni)
        fixq = np.zeros(1 + ni * nf, np.uint64)
        L.run_host(prm.ctypes.data, eb.ctypes.data, fr.ctypes.data, nf, ni * nf, out.ctypes.data, st.ctypes.data,
                   err.ctypes.data, fixq.ctypes.data, ni * nf, ws.ctypes.data, grid)
        assert (ws[nw:] == 7.25).all() and (out[ni * nf * n * 2:] == 7.25).all()
        x = out[:ni * nf * n * 2].reshape(ni, nf, n, 2)
        return x[..., 0] + 1j * x[..., 1], st, err, int(fixq[0]), L.words()
    finally:
        shutil.rmtree(d)


def ladder(sections, far):
    """RC ladder, driven at its first node or (far) at its last."""
    t = [f"V1 {'n%d' % sections if far else 'n0'} 0 DC 0 AC 1"]
    for k in range(sections):
        t += [f"R{k + 1} n{k} n{k + 1} {1000 + 7 * k}", f"C{k + 1} n{k + 1} 0 {1e-9 * (1 + 0.01 * k)}"]
    return "\n".join(t + ["R0 n0 0 5000"]) + "\n"


@pytest.mark.parametrize("far", [False, True])
@pytest.mark.parametrize("order", [2, -1])  # minimum degree, balanced
@pytest.mark.parametrize("sections", [20, 21, 22, 23, 54, 200])
def test_looped_chain_vs_oracle(oracle, sections, order, far):
    import krets_amd as kg
    text = ladder(sections, far)
    c = kg.Circuit(text)
    r, src = source(c, 2, order)
    if order < 0 and sections < 22 and r < 0:  # two chains of fewer than eight iterations
        assert "chain" in src
        return
    assert r > 0, src
    f = np.geomspace(10.0, 1e6, 67)
    params = np.stack([c.params, c.params])
    x, st, err, queued, words = run(src, params, c.elements, f, c.n, 2)  # 134 systems: two of three blocks' grid
    assert (st == 0).all() and queued == 0 and words >= sections - 14
    xr = oracle.Circuit(text).ac(f)
    for i in range(2):
        assert max(nerr(x[i, j], xr[j]) for j in range(len(f))) < 1e-12
    if sections <= 54:  # the register form's growth figure, row by row the same
        r, full = source(c, 0)
        if r > 0 and order == 2:
            from test_jit import host_run
            _, _, e2 = host_run(full, params, c.elements, f, c.n)
            assert np.array_equal(err, e2)


def test_looped_declines():
    import krets_amd as kg
    from krets_amd import workloads as W
    r, why = source(kg.Circuit("V1 a 0 AC 1\nR1 a b 10\nC1 b 0 1e-9\n"), 2)
    assert r < 0 and "chain" in why
    r, why = source(kg.Circuit(W.c4_rectifier(1).netlists[0]), 2)
    assert r < 0 and "diode" in why
