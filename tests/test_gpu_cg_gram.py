"""SR-CG of the precision form, whose products come from the FP32 Gram of the
samples, in one launch (271 parameters) and in launches (421): the solution of
22 iterations, a residual refresh among them, equals bit for bit that of the
same iteration on the host, which forms every sum in the kernels' order."""
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


def _tree(p):
    """Pairwise over the last axis, halves first."""
    while p.shape[-1] > 1:
        h = p.shape[-1] // 2
        p = p[..., :h] + p[..., h:]
    return p[..., 0]


def _strided(prod, lanes):
    """Partials of `lanes` strided lanes, then the tree."""
    pad = -prod.shape[-1] % lanes
    prod = np.concatenate([prod, np.zeros(prod.shape[:-1] + (pad,))], axis=-1)
    prod = prod.reshape(prod.shape[:-1] + (-1, lanes))
    acc = np.zeros(prod.shape[:-2] + (lanes,))
    for k in range(prod.shape[-2]):
        acc = acc + prod[..., k, :]
    return _tree(acc)


def _solve(G, mean, diag, g, inv_w, shift, max_it, precond):
    dot = lambda a, b: _strided(a * b, 256)

    def apply(v):
        return inv_w * _strided(G * v, 64) - dot(mean, v) * mean + shift * diag * v

    den = (1.0 + shift) * diag
    assert np.abs(den).min() > 1e-12
    x = np.zeros_like(g)
    r = g - apply(x) if precond else g.copy()
    d = r / den if precond else r.copy()
    delta = dot(r, d)
    for it in range(max_it):
        q = apply(d)
        alpha = delta / dot(d, q)
        x = x + alpha * d
        r = g - apply(x) if (it + 1) % 20 == 0 else r - alpha * q
        src = r / den if precond else r
        dn = dot(r, src)
        beta = dn / delta
        d = src + beta * d
        delta = dn if precond else delta * beta
    return x


@pytest.mark.parametrize("precond", [False, True])
@pytest.mark.parametrize("L,nup,na", [(8, 28, 271), (10, 42, 421)])
def test_gram_solve(M, tmp_path, L, nup, na, precond):
    import lattice
    import torch
    W, limit, shift, dt = 40, 22, 1e-3, 0.01
    info = lattice.write_workload("square8", str(tmp_path), seed=7, warmup=2, interval=2, cg_max_iter=limit, step_dt=dt,
                                  sta_del=shift, overrides=dict(L=L, nup=nup, spgl=1, ntrans=1, walkers=W))
    path = os.path.join(str(tmp_path), "modpara.def")
    with open(path) as f:
        text = f.read().split("\n")
    text = [("NSRCG 2" if precond else "NSRCG 1") if t.split()[:1] == ["NSRCG"] else t for t in text]
    with open(path, "w") as f:
        f.write("\n".join(t for t in text if t) + "\nNSRCGFallback 0\nDSROptCGTol 0.0\n")
    print(f"FP32 Gram CG, L={L}, precond={precond}", flush=True)
    ens = M.Ensemble(info["namelist"], info["initial"], walkers=W)
    ens.set_precision("mixed")
    ens.sample()
    ens.measure()
    oo, ho = ens.operands()
    O = np.concatenate([ens.o_store(w) for w in range(W)])
    ens.sr_cg()
    _, x = ens.cg()
    size = ens.size
    var = oo[size:] - oo[:size] * oo[:size]
    assert ens.timings()["cg_na"] == len(x)
    active = 1 + np.flatnonzero(var[1:] >= var[1:].max() * 1e-10)
    assert len(active) == len(x) == na
    mean, diag = oo[active], var[active]
    g = -(2.0 * dt) * (ho[active] - ho[0] * oo[active])
    pack = np.ascontiguousarray(O[:, active], dtype=np.float32)
    out = torch.zeros((na, na), dtype=torch.float64, device="cuda")
    M.sr_gram_real_f32(torch.tensor(pack, device="cuda"), out, na, W)
    G = out.cpu().numpy()
    assert np.array_equal(G, G.astype(np.float32))
    want = _solve(G, mean, diag, g, 1.0 / ens.energy()[0], shift, limit, precond)
    assert np.array_equal(x, want), np.abs(x - want).max() / np.abs(want).max()
    ens.close()
