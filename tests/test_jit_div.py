"""CPU: the generated lane kernels' division by a constant, kg_div(a, n, 1/n):
equal to a / n bit for bit over the voltages and thermal voltages that a diode
sees, and kg_div_low also where the quotient lies below the range of a double
(a diode far in reverse in the clean modes; krets' mode limits the voltage)."""
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
    src_text = buf.value.decode()
    assert "kg_div_low(v, nvt" in src_text and "kg_div(v, nvt" not in src_text  # step control: clean mode only
    fns = [re.search(r"double %s\(.*?\n\}\n" % f, src_text, re.S).group(0) for f in ("kg_div", "kg_div_low")]
    src, so = tmp_path / "d.cpp", tmp_path / "d.so"
    src.write_text("".join("static " + f for f in fns) +
                   'extern "C" void run(const double* a, const double* n, double* q, double* ql, long k) {\n'
                   "  for (long i = 0; i < k; i++) {\n    q[i] = kg_div(a[i], n[i], 1.0 / n[i]);\n"
                   "    ql[i] = kg_div_low(a[i], n[i], 1.0 / n[i]);\n  }\n}\n")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-ffp-contract=off", str(src), "-o", str(so)], check=True,
                   capture_output=True)
    L = ctypes.CDLL(str(so))
    rng = np.random.default_rng(3)
    vt = 1.380649e-23 * 300.0 / 1.602176634e-19
    n = vt * rng.uniform(0.5, 5.0, 200000)
    a = rng.choice([-1.0, 1.0], len(n)) * 10.0 ** rng.uniform(-280, 306, len(n))
    a[:100000] = rng.uniform(-60.0, 60.0, 100000)
    q, ql = np.zeros_like(a), np.zeros_like(a)
    p = lambda x: ctypes.c_void_p(x.ctypes.data)
    L.run(p(a), p(n), p(q), p(ql), ctypes.c_long(len(a)))
    assert np.array_equal(q, a / n) and np.array_equal(ql, a / n)
    a, n = -np.array([1.7e308, 1e307, 5e306, 4.7e306, 1.7e308]), vt * np.array([1.0, 1.0, 1.0, 1.0, 0.5])
    L.run(p(a), p(n), p(q), p(ql), ctypes.c_long(len(a)))
    with np.errstate(over="ignore"):
        assert np.array_equal(ql[:len(a)], a / n) and np.isinf(ql[:len(a)]).all()
