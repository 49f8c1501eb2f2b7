"""Sampler chain against the oracle at the sizes where the sweep kernel
changes form: lanes per plane below and above a plane's columns (columns per
lane in the rank-update pass), Jastrow table and projection parameters inside
and outside their LDS copies (ns 64 / 100, nproj 256), the touched-parameter
bitmap (nproj > 512), rows shorter than a wave.  Bit-exact: the chain is
integer and ordered double arithmetic."""
import sys

import numpy as np
import pytest

import oracle_py as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import torch
    torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    import mvmc_hip
    return mvmc_hip


# workload, sites per side, spins up, planes = spgl * ntrans, exchange, Jastrow classes
@pytest.mark.parametrize("name,L,nup,spgl,ntrans,ex,jast", [
    ("chain16", 6, 3, 1, 1, 0, "nn"),
    ("chain16", 12, 5, 2, 2, 1, "nn"),
    ("chain16", 34, 17, 2, 1, 0, "nn"),
    ("square8", 6, 13, 1, 4, 0, "distance"),
    ("square8", 8, 33 - 1, 2, 4, 1, "distance"),
    ("square16", 8, 25, 2, 4, 0, "sublattice"),
    ("square8", 10, 49, 1, 1, 0, "distance"),
    ("square16", 12, 60, 1, 4, 0, "sublattice"),
])
def test_chain_matches_oracle(M, tmp_path, name, L, nup, spgl, ntrans, ex, jast):
    import lattice
    W = 2
    ov = dict(L=L, nup=nup, spgl=spgl, ntrans=ntrans, jastrow=jast)
    info = lattice.write_workload(name, str(tmp_path / "m"), sr_steps=1, warmup=2, interval=3, ex_update_path=ex,
                                  overrides=ov)
    print(f"{name} L={L} n={2 * nup} planes={spgl * ntrans} ex={ex}: chain vs oracle", flush=True)
    sys.stdout.flush()
    O.set_math(1)
    ens = M.Ensemble(info["namelist"], info["initial"], walkers=W)
    try:
        run = O.Run(info["namelist"], info["initial"], walkers=W)
        run.sample()
        ens.sample()
        for w in range(W):
            sg, so = ens.walker(w), run.walker(w)
            assert np.array_equal(sg["ele_idx"], so["ele_idx"]), w
            assert np.array_equal(sg["rng"], so["rng"]) and sg["rng_idx"] == so["rng_idx"], w
            assert list(sg["counter"]) == list(so["counter"][:4]), w
    finally:
        O.set_math(0)
        ens.close()
