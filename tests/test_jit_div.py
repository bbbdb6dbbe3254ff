"""CPU: the generated lane kernels' division by a constant, kg_div(a, n, 1/n):
equal to a / n bit for bit over the voltages and thermal voltages that a diode
sees, and where the quotient leaves the range of a double."""
import ctypes
import re
import subprocess

import numpy as np


def test_kg_div_is_a_division(tmp_path):
    import krets_amd as kg
    from krets_amd import _lib
    from krets_amd import workloads as W
    c = kg.Circuit(W.c4_rectifier(1).netlists[0])
    el, pr = np.ascontiguousarray(c.elements), np.ascontiguousarray(c.params)
    buf = ctypes.create_string_buffer(1 << 20)
    assert _lib.lib().kg_jit_lte_source(el.ctypes.data, len(el), c.n, pr.ctypes.data, 1e-6, buf, len(buf)) > 0
    fn = re.search(r"double kg_div\(.*?\n\}\n", buf.value.decode(), re.S).group(0)
    src, so = tmp_path / "d.cpp", tmp_path / "d.so"
    src.write_text("static " + fn + 'extern "C" void run(const double* a, const double* n, double* q, long k) {\n'
                   "  for (long i = 0; i < k; i++) q[i] = kg_div(a[i], n[i], 1.0 / n[i]);\n}\n")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-ffp-contract=off", str(src), "-o", str(so)], check=True,
                   capture_output=True)
    L = ctypes.CDLL(str(so))
    rng = np.random.default_rng(3)
    vt = 1.380649e-23 * 300.0 / 1.602176634e-19
    n = vt * rng.uniform(0.5, 5.0, 200000)
    a = rng.choice([-1.0, 1.0], len(n)) * 10.0 ** rng.uniform(-280, 308, len(n))
    far = np.array([0.0, 1.7e308, 1e307, 5e306, 4.7e306, np.inf])
    a[:12] = np.concatenate([far, -far])
    a[12:100000] = rng.uniform(-60.0, 60.0, 99988)
    q = np.zeros_like(a)
    L.run(ctypes.c_void_p(a.ctypes.data), ctypes.c_void_p(n.ctypes.data), ctypes.c_void_p(q.ctypes.data),
          ctypes.c_long(len(a)))
    with np.errstate(over="ignore"):
        assert np.array_equal(q, a / n)
