"""GPU: a backward pass belongs to the batch of its forward pass. After another
load it is refused, in each form (stored trajectory, checkpoints in LDS, level
by level), where it had taken the new batch's sizes for the old one's states;
a new forward pass serves the new batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tps,precision", [(0, 0), (3064, 0), (64, 0), (16, 1)])
def test_backward_after_another_load_is_refused(oracle, tps, precision):
    import krets_amd as kg
    from krets_amd import workloads as W
    print(f"[gpu case] backward after another load, tps={tps} precision={precision}", flush=True)
    cfg = kg.SolverConfig(compat=False, threads_per_system=tps)
    ctx = kg.Context()
    for sections in (8, 30):
        b = W.c5_rc_ladder(2, sections=sections, seed=5)
        b.load(ctx)
        with pytest.raises(kg.KretsGpuError, match="no forward pass"):
            ctx.adjoint_backward()
        c = np.zeros(b.n_unknowns)
        c[b.names.index("V(n3)")] = 1.0
        ctx.adjoint_forward(1e-9, 40, c, precision=precision, config=cfg)
    g, st = ctx.adjoint_backward()
    _, gr = oracle.Circuit(b.netlists[0]).adjoint(1e-9, 40, c, method=kg.TRAP)
    assert (st == 0).all() and np.max(np.abs(g[0] - gr)) < 1e-9 * np.max(np.abs(gr))
