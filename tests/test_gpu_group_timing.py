"""Timings of a group's SR-CG solves: runs whose operator is past one launch are
solved one after the other, each timed over its own solve alone."""
import os

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import torch
    torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    import mvmc_hip
    return mvmc_hip


def test_solve_times_do_not_overlap(M, tmp_path):
    import lattice
    W, R = 64, 3
    infos = [lattice.write_workload("square16", os.path.join(str(tmp_path), f"r{k}"), seed=5 + k, warmup=1, interval=1,
                                    overrides=dict(L=8, nup=12, spgl=1, ntrans=1, walkers=W)) for k in range(R)]
    print(f"group of {R} runs, {W} walkers each", flush=True)
    g = M.EnsembleGroup([i["namelist"] for i in infos], [i["initial"] for i in infos], [W] * R)
    for _ in range(2):
        g.opt_step()
        t = [e.timings() for e in g.runs]
        assert all(x["cg_na"] > 640 and x["cg_iter"] > 20 for x in t)
        # disjoint intervals inside the group's SR phase, whatever the clock
        assert sum(x["cg_ms"] for x in t) <= 1e3 * g.timings()["sr_s"]
    g.close()
