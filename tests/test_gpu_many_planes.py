"""More QP planes than a workgroup has threads (256): placement, rebuilds and
the chain of a small model against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle_py as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nup,spgl,ex", [(2, 256, 0), (2, 257, 0), (1, 300, 1)])
def test_chain_matches_oracle(tmp_path, nup, spgl, ex):
    import torch
    torch.zeros(1, device="cuda")
    import lattice
    import mvmc_hip
    info = lattice.write_workload("chain16", str(tmp_path), seed=3, warmup=2, interval=2, ex_update_path=ex,
                                  overrides=dict(L=12, nup=nup, spgl=spgl, ntrans=1, walkers=2, jastrow="distance"))
    print(f"{info['nqp']} planes of {2 * nup} rows, exchange {ex}", flush=True)
    O.set_math(1)
    try:
        run = O.Run(info["namelist"], info["initial"], walkers=2)
        ens = mvmc_hip.Ensemble(info["namelist"], info["initial"], walkers=2)
        for _ in range(2):
            run.sample()
            ens.sample()
            for w in range(2):
                sg, so = ens.walker(w), run.walker(w)
                assert np.array_equal(sg["ele_idx"], so["ele_idx"]), w
                assert np.array_equal(sg["rng"], so["rng"]) and sg["rng_idx"] == so["rng_idx"], w
                assert list(sg["counter"]) == list(so["counter"][:4]), w
        ens.close()
    finally:
        O.set_math(0)
