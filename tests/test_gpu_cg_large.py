"""SR-CG of operators past one launch, whole solves against the oracle bit for
bit: the first sizes past that line, several superchunks of rows, their fold in the tail (up to 8000 partials)
and apart, the column counts per lane of the chunk pass (two rows at a time up
to 4096 columns, one above, the wide form past 8192), the dot products past
the tail's LDS (8000); iteration limits on both sides of a residual refresh."""
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
@pytest.mark.parametrize("na,rows", [(20, 8192), (64, 1281), (128, 1025), (192, 769), (320, 513), (448, 257),
                                     (640, 257), (642, 40), (700, 1100), (1999, 2048), (2000, 2048), (2500, 600), (4096, 545),
                                     (4097, 513), (6144, 70), (6145, 33), (8000, 40), (8001, 70), (8193, 35)])
def test_solve_matches_oracle(M, na, rows, variant):
    import torch
    print(f"cg na={na} rows={rows} variant={variant}", flush=True)
    rng = np.random.default_rng(1000 * na + rows)
    o = rng.standard_normal((rows, na))
    mean = o.mean(axis=0)
    diag = (o * o).mean(axis=0) - mean * mean
    g = rng.standard_normal(na)
    dev = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")
    for limit in (2, 22):
        x = torch.zeros(na, dtype=torch.float64, device="cuda")
        st = M.sr_cg_solve(dev(o), dev(mean), dev(diag), dev(g), x, na, 1, rows, 1.0 / rows, 1e-2, 1e-9, limit, variant)
        sto, xo, _, _ = O.cg_solve(mean, diag, o, g, 1.0 / rows, 1e-2, 1e-9, limit, bool(variant))
        assert st == sto
        assert np.array_equal(x.cpu().numpy(), xo)


@pytest.mark.parametrize("na,rows", [(8, 32), (700, 64)])
def test_negative_iteration_limit_is_refused(M, na, rows):
    import torch
    print(f"cg na={na} rows={rows} limit -1", flush=True)
    o = torch.randn(rows, na, dtype=torch.float64, device="cuda")
    v = torch.ones(na, dtype=torch.float64, device="cuda")
    with pytest.raises(M.BackendError):
        M.sr_cg_solve(o, v, v, v, torch.zeros_like(v), na, 1, rows, 1.0 / rows, 1e-2, 1e-9, -1, 0)
