"""A group whose runs are rebuilt by different kernels: planes of 226 rows walker
by walker through the group's shared list, planes of 28 rows plane by plane.
Rows, parameters and walker states of two SR steps equal those of the runs
stepped alone, bit for bit, with periodic rebuilds in both runs."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import torch
    torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    import mvmc_hip
    return mvmc_hip


@pytest.mark.parametrize("graph_rounds", [0, 2])
def test_mixed_group_matches_runs_alone(M, tmp_path, graph_rounds):
    import lattice
    small = lattice.write_workload("square8", os.path.join(str(tmp_path), "a"), seed=3, warmup=1, interval=4,
                                   overrides=dict(L=6, nup=14, spgl=1, ntrans=2, walkers=5))
    large = lattice.write_workload("square16", os.path.join(str(tmp_path), "b"), seed=4, warmup=1, interval=4,
                                   cg_max_iter=25, overrides=dict(L=16, nup=113, spgl=1, ntrans=1, walkers=3))
    infos, W = [small, large], [5, 3]
    print(f"group of Nsize {[i['nsize'] for i in infos]}, graph rounds {graph_rounds}", flush=True)
    g = M.EnsembleGroup([i["namelist"] for i in infos], [i["initial"] for i in infos], W)
    g.set_graph(graph_rounds)
    rows_g = [g.opt_step() for _ in range(2)]
    for r, info in enumerate(infos):
        e = M.Ensemble(info["namelist"], info["initial"], walkers=W[r])
        rows_a, rebuilt = [], 0
        for _ in range(2):
            rows_a.append(e.opt_step())
            rebuilt += e.timings()["rebuilt"]
        assert rebuilt > 0, r
        for k in range(2):
            assert np.array_equal(rows_g[k][r], rows_a[k]), (r, k, rows_g[k][r], rows_a[k])
        assert np.array_equal(np.concatenate(g.runs[r].params()), np.concatenate(e.params())), r
        for w in range(W[r]):
            a, b = g.runs[r].walker(w), e.walker(w)
            assert np.array_equal(a["ele_idx"], b["ele_idx"]) and np.array_equal(a["rng"], b["rng"]), (r, w)
            assert a["rng_idx"] == b["rng_idx"] and tuple(a["counter"]) == tuple(b["counter"]), (r, w)
        e.close()
    g.close()
