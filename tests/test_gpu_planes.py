"""Edges of the plane kernels behind mvmc_pfinv_f64 / mvmc_pfinv_c128 (one
plane per wave up to 104 rows, complex up to 64; four waves per plane above):
the sizes on both sides of every block count and of the changes of kernel,
with random planes, integer planes (ties and exact zeros in the pivot
search), a plane with a NaN, a zero and a non-finite one: Pfaffians, statuses
and inverses equal to the oracle's bit for bit (both are the same operation
sequence, so no tolerance), out of place, in place and through the
no-allocation entry."""
import sys

import numpy as np
import pytest

import oracle_py as O

pytestmark = pytest.mark.gpu


def log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def M():
    import torch
    torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    import mvmc_hip
    return mvmc_hip


def _planes(n, cplx):
    rng = np.random.default_rng(7000 + n + (500 if cplx else 0))
    a = rng.standard_normal((9, n, n))
    a[3:5] = rng.integers(-1, 2, (2, n, n))
    if cplx:
        b = rng.standard_normal((9, n, n))
        b[3:5] = rng.integers(-1, 2, (2, n, n))
        a = a + 1j * b
    a = a - a.transpose(0, 2, 1)
    a[5] = 0.0
    a[6] *= 1e300
    a[7][0, n - 1] = np.nan
    a[7][n - 1, 0] = np.nan
    return np.ascontiguousarray(a)


def _same(x, y):
    return np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("cplx,n", [(False, n) for n in (2, 8, 10, 14, 18, 24, 26, 38, 40, 42, 50, 56, 58, 64, 66, 72,
                                                        74, 80, 82, 90, 96, 104, 106, 112, 114, 146, 162, 178, 210,
                                                        224)] +
                         [(True, n) for n in (2, 8, 10, 18, 26, 34, 42, 50, 58, 64, 66, 80, 82, 98, 114, 130, 146,
                                              160)])
def test_plane_kernels_at_their_edges(M, cplx, n):
    import torch
    planes = _planes(n, cplx)
    count = len(planes)
    for order in ((0, 1) if cplx else (0,)):
        log(f"planes n={n} complex={cplx} order={order}")
        pf_o, inv_o, st_o = O.pfinv_c128(planes, order) if cplx else O.pfinv(planes)
        assert st_o[5] > 0 and (st_o[:3] == 0).all()
        ran = []
        for form in ("out", "in place") + (() if cplx else ("no allocation",)):
            dp = torch.tensor(planes, device="cuda")
            pf = torch.zeros(count, dtype=dp.dtype, device="cuda")
            st = torch.zeros(count, dtype=torch.int32, device="cuda")
            inv = dp if form == "in place" else torch.full_like(dp, 5.0)
            if cplx:
                M.pfaffian_inverse_batched_c128(dp, pf, inv, st, n, count, order)
            elif form == "no allocation":
                M.pfaffian_inverse_batched_noalloc(dp, pf, inv, st, n, count)
            else:
                M.pfaffian_inverse_batched(dp, pf, inv, st, n, count)
            torch.cuda.synchronize()
            ran.append(form)
            assert np.array_equal(st.cpu().numpy(), st_o), form
            fin = np.isfinite(pf_o)
            assert _same(pf.cpu().numpy()[fin], pf_o[fin]), form
            assert np.array_equal(np.isfinite(pf.cpu().numpy()), fin), form
            assert _same(inv.cpu().numpy(), inv_o), form
        assert len(ran) == (2 if cplx else 3)
