"""GPU: an AC sweep with a mapping asked for defers its operating point to a
captured graph, and the plans that the mapping adds meanwhile move the table of
plans. The deferred launch reads the table where it is then: the graph's
results are those of the eager calls, bit for bit, over many frequency ranges
(each adds plans)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("uneven,tps", [(True, 1), (False, 2021), (False, 2031)])
def test_deferred_operating_point_reads_the_moved_table(oracle, uneven, tps):
    import krets_amd as kg
    from krets_amd import workloads as W
    print(f"[gpu case] deferred operating point, uneven={uneven} tps={tps}", flush=True)
    nets = [W.c2_rc_ladder_mc(1, sections=s, seed=11).netlists[0] for s in ((3, 17, 30) if uneven else (150,) * 3)]
    cs = [kg.Circuit(t) for t in nets]
    cfg, got = kg.SolverConfig(threads_per_system=tps), []
    for graphs in (True, False):
        ctx = kg.Context()
        if uneven:
            ctx.load(np.concatenate([c.elements for c in cs]), np.concatenate([c.params for c in cs]),
                     [c.n for c in cs], np.cumsum([0] + [len(c.elements) for c in cs]))
        else:
            ctx.load(cs[0].elements, np.stack([c.params for c in cs]), cs[0].n)
        ctx.use_graphs(graphs)
        runs = []
        for k in range(24):
            for _ in range(2):
                x, st, _ = ctx.ac_sweep(np.geomspace(10.0, 1e4 * (k + 1), 9), config=cfg)
            assert (st == 0).all()
            runs.append([np.array(v) for v in x])
        got.append(runs)
    for p, q in zip(*got):
        assert all(np.array_equal(u, v) for u, v in zip(p, q))
    f = np.geomspace(10.0, 24e4, 9)
    for i in range(3):
        xr = oracle.Circuit(nets[i]).ac(f)
        assert max(np.linalg.norm(got[0][-1][i][j] - xr[j]) / np.linalg.norm(xr[j]) for j in range(9)) < 1e-12
