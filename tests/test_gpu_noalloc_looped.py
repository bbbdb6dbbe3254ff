"""GPU: the allocation-free AC sweep where the looped lane kernel serves the
batch. It must return what kg_ac_sweep returns bit for bit (the kernel takes
any grid, so the workspace that the scratch array holds is enough), with the
mapping asked for and with the tuned one, in both precisions, for more blocks
than the array has workspaces for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_zz_no_alloc import check_pair, noalloc_call


def ladder(ni, sections):
    from krets_amd import workloads as W
    return W.c2_rc_ladder_mc(ni, sections=sections, seed=9)


# 200 sections: some 40 workspaces in 8 MiB; 65 x 101 systems are 103 blocks. 2000: four workspaces, ten blocks.
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("ni,sections,nf,tps", [(65, 200, 101, 0), (65, 200, 101, 2021), (65, 200, 101, 2031),
                                                (3, 30, 21, 2021), (2, 2000, 300, 2021)])
def test_noalloc_matches_ac_sweep_looped(prec, ni, sections, nf, tps):
    import krets_amd as kg
    print(f"[gpu case] no-alloc looped {ni} x {nf}, {sections} sections, prec={prec} tps={tps}", flush=True)
    b = ladder(ni, sections)
    ctx = kg.Context()
    b.load(ctx)
    f = np.geomspace(10.0, 1e5, nf)
    fs = f[np.linspace(0, nf - 1, 20).round().astype(int)]  # same range: the same plans
    check_pair(kg, ctx, b.n_unknowns, f, fs, prec, kg.SolverConfig(threads_per_system=tps))
