"""SR-CG of small operators (one launch) against the oracle at the edges of
its split: columns per lane (64 k + 0, 1), rows per chunk of 32 and per group
of 4 or 2, chunks beyond one per wave, both preconditioners."""
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


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("na,rows", [(1, 5), (63, 31), (64, 33), (65, 257), (128, 38), (192, 300), (193, 6), (320, 65),
                                     (321, 64), (448, 101), (449, 70), (640, 255), (641, 40)])
def test_solve_matches_oracle(M, na, rows, variant):
    import torch
    print(f"cg na={na} rows={rows} variant={variant}", flush=True)
    rng = np.random.default_rng(1000 * na + rows)
    o = rng.standard_normal((rows, na))
    mean = o.mean(axis=0)
    diag = (o * o).mean(axis=0) - mean * mean
    g = rng.standard_normal(na)
    dev = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")
    for limit in (1, 23):
        x = torch.zeros(na, dtype=torch.float64, device="cuda")
        st = M.sr_cg_solve(dev(o), dev(mean), dev(diag), dev(g), x, na, 1, rows, 1.0 / rows, 1e-2, 1e-9, limit, variant)
        sto, xo, _, _ = O.cg_solve(mean, diag, o, g, 1.0 / rows, 1e-2, 1e-9, limit, bool(variant))
        assert st == sto
        assert np.array_equal(x.cpu().numpy(), xo)
