"""The work that users of this library have it do, as cases to be timed.

A user of the library either runs whole optimisation steps of a walker
ensemble (sample, measure, SR update), or calls its stages on their own data:
the batched skew-symmetric Pfaffian + inverse, the measurement of given
configurations, the derivative form, the SR solves.  The listed cases take
each of these once over the sizes in use, from calls of a few microseconds
to the 16 x 16 lattice; draw() gives more of the same ranges.  All models come from the
library's own generator (mvmc-rs_amd/lattice.py).

Steps are taken from the same parameters each time (set_params, as a
parameter scan or a restarted run does), so a pass is the same work however
many passes came before it; the walkers go on from their last configuration.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mvmc-rs_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import lattice  # noqa: E402
import mvmc_hip  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # a few small planes at a time: a host program that asks for one small model's planes, call by call
        dict(name="pfinv_n16", kind="pfinv", n=16, count=64, complex=False, order=0),
        # the planes of a mid-sized lattice (10 x 10 near half filling), an odd batch
        dict(name="pfinv_n98", kind="pfinv", n=98, count=1777, complex=False, order=0),
        # the planes of the 16 x 16 lattice (112 + 112 electrons)
        dict(name="pfinv_n224", kind="pfinv", n=224, count=1024, complex=False, order=0),
        # complex planes of a 12 x 12 lattice with flux, in the production sampler's order
        dict(name="pfinv_c128_n144", kind="pfinv", n=144, count=768, complex=True, order=1),
        # the 16-site chain as it is configured: 256 walkers, 16 sweeps a sample; launches and latency
        dict(name="chain16_step", kind="step", lattice="chain16", L=16, nup=8, spgl=1, ntrans=1, walkers=256,
             interval=16, samples=1, ex=0, precision="fp64", direct=False),
        # the 8 x 8 lattice, 4096 walkers, the precision form (FP32 inverse and FP32 samples in SR)
        dict(name="square8_step_mixed", kind="step", lattice="square8", L=8, nup=32, spgl=2, ntrans=4, walkers=4096,
             interval=2, samples=1, ex=0, precision="mixed", direct=False),
        # the 16 x 16 t-t'-U lattice: sampling and measurement at fixed parameters (an energy evaluation)
        dict(name="square16_energy", kind="energy", lattice="square16", L=16, nup=112, spgl=2, ntrans=4, walkers=512,
             interval=2, samples=1, ex=0, precision="fp64"),
        # lattices of uneven size stepped as one group
        dict(name="uneven_group", kind="group", walkers=256, interval=2),
        # measurement of configurations that the caller brings (host arrays in and out), an odd count
        dict(name="square8_configs", kind="configs", lattice="square8", L=8, nup=32, spgl=2, ntrans=4, walkers=1024,
             count=999),
        # log|psi| of sampled configurations and its vector-Jacobian product (forward and backward)
        dict(name="square8_vjp", kind="vjp", lattice="square8", L=8, nup=30, spgl=2, ntrans=4, walkers=1024,
             form="adjoint"),
        # direct SR from stored samples: Gram, S and g, Cholesky solve
        dict(name="sr_direct", kind="direct", na=1111, rows=4096, f32=False),
        # SR-CG from stored samples
        dict(name="sr_cg", kind="cg", na=2099, rows=8192, variant=0),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pfinv", "pfinv", "pfinv", "step", "energy", "group", "configs", "vjp", "direct", "cg"])
    if kind == "pfinv":
        cplx = rng.random() < 0.3
        n = 2 * _logint(rng, 2, 80 if cplx else 128)
        most = 768 * 144 ** 3 / n ** 3 if cplx else 1024 * 224 ** 3 / n ** 3
        return dict(kind="pfinv", n=n, count=max(1, min(4096, _logint(rng, 8, max(9, most)))), complex=cplx,
                    order=rng.choice([0, 1]) if cplx else 0)
    if kind in ("step", "energy", "configs", "vjp"):
        if rng.random() < 0.4:
            L = 2 * rng.randint(3, 16)
            c = dict(kind=kind, lattice="chain16", L=L, nup=max(2, L // 2 - rng.randint(0, 1)), spgl=rng.choice([1, 2]),
                     ntrans=rng.choice([1, 2]), walkers=_logint(rng, 16, 1024))
        else:
            L = rng.choice([4, 6, 8, 10])
            c = dict(kind=kind, lattice="square8", L=L, nup=L * L // 2 - rng.randint(0, L * L // 8),
                     spgl=rng.choice([1, 2]), ntrans=rng.choice([1, 4]), walkers=_logint(rng, 16, 1024 if L <= 8 else 256))
        if kind == "configs":
            c["count"] = max(1, c["walkers"] - rng.randint(0, 7))
        elif kind == "vjp":
            c["form"] = rng.choice(["adjoint", "rows"])
        else:
            c.update(interval=rng.choice([2, 4]), samples=rng.choice([1, 1, 2]), ex=rng.choice([0, 0, 0, 1]),
                     precision=rng.choice(["fp64", "fp64", "mixed"]))
            if kind == "step":
                c["direct"] = rng.random() < 0.3
        return c
    if kind == "group":
        return dict(kind="group", walkers=_logint(rng, 16, 256), interval=rng.choice([1, 2]))
    if kind == "direct":
        return dict(kind="direct", na=_logint(rng, 20, 1111), rows=_logint(rng, 256, 8192), f32=rng.random() < 0.4)
    return dict(kind="cg", na=_logint(rng, 20, 4000), rows=_logint(rng, 256, 8192), variant=rng.choice([0, 1]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    return g


def _files(case, seed, out_dir):
    """The model's input files: the library's generator with this case's sizes."""
    kw = dict(interval=case.get("interval", 2), nvmc_sample=case.get("samples", 1), ex_update_path=case.get("ex", 0))
    ov = dict(L=case["L"], nup=case["nup"], spgl=case["spgl"], ntrans=case["ntrans"], walkers=case["walkers"])
    return lattice.write_workload(case["lattice"], out_dir, seed=int(seed) % (1 << 31), warmup=2,
                                  rnd_seed=1 + int(seed) % 100003, overrides=ov, **kw)


def _configs(case, seed):
    """Random configurations, electron -> site, spin up first."""
    ns = case["L"] if case["lattice"] == "chain16" else case["L"] ** 2
    r = np.random.default_rng(int(seed) % (1 << 31))
    order = r.random((case["count"], 2, ns)).argsort(axis=2)[:, :, :case["nup"]]
    return np.ascontiguousarray(order.reshape(case["count"], -1), dtype=np.int32)


def _planes(case, seed):
    n, count = case["n"], case["count"]
    a = torch.randn(count, n, n, generator=_gen(seed), device=DEV,
                    dtype=torch.complex128 if case["complex"] else torch.float64)
    return ((a - a.transpose(1, 2)) / math.sqrt(2 * n)).contiguous()


def _samples(rows, na, seed, dtype=torch.float64):
    """Log-derivative samples [rows][na]: parameters of different scale about nonzero means."""
    g = _gen(seed)
    scale = torch.exp(torch.rand(na, generator=g, device=DEV, dtype=torch.float64) * math.log(20.0)) / 20.0
    mean = torch.randn(na, generator=g, device=DEV, dtype=torch.float64) * 0.5
    o = torch.randn(rows, na, generator=g, device=DEV, dtype=torch.float64)
    return ((o + mean) * scale).to(dtype).contiguous()


def _cg_operands(case, seed):
    na, rows = case["na"], case["rows"]
    pack = _samples(rows, na, seed)
    mean = pack.mean(dim=0)
    diag = (pack * pack).mean(dim=0) - mean * mean
    e = torch.randn(rows, generator=_gen(seed + 1), device=DEV, dtype=torch.float64)
    g = -0.02 * ((pack * e[:, None]).mean(dim=0) - e.mean() * mean)
    return pack, mean.contiguous(), diag.contiguous(), g.contiguous()


CG = dict(shift=1e-3, tol=1e-9, max_it=60)  # a fixed number of iterations bounds the step, as NSROptCGMaxIter does


def prepare(case, seed):
    k = case["kind"]
    if k == "pfinv":
        planes = _planes(case, seed)
        return dict(case=case, planes=planes, pf=torch.zeros(case["count"], dtype=planes.dtype, device=DEV),
                    inv=torch.zeros_like(planes), status=torch.zeros(case["count"], dtype=torch.int32, device=DEV))
    if k == "direct":
        na, rows = case["na"], case["rows"]
        o = _samples(rows, na, seed, torch.float32 if case["f32"] else torch.float64)
        store = torch.cat([torch.ones(rows, 1, dtype=o.dtype, device=DEV), o], dim=1) / math.sqrt(rows)
        n = na + 1
        e = torch.randn(rows, generator=_gen(seed + 1), device=DEV, dtype=torch.float64)
        ho = (store.double() * e[:, None]).sum(dim=0) / math.sqrt(rows)
        return dict(case=case, store=store.contiguous(), ho=ho.contiguous(),
                    map=torch.arange(na, dtype=torch.int32, device=DEV),
                    gram=torch.zeros(n, n, dtype=torch.float64, device=DEV),
                    s=torch.zeros(na, na, dtype=torch.float64, device=DEV),
                    g=torch.zeros(na, dtype=torch.float64, device=DEV))
    if k == "cg":
        pack, mean, diag, g = _cg_operands(case, seed)
        return dict(case=case, pack=pack, mean=mean, diag=diag, g=g, x=torch.zeros_like(g))
    torch.zeros(1, device=DEV)  # torch brings the GPU up before the library does
    with tempfile.TemporaryDirectory() as d:
        if k == "group":
            infos = lattice.write_uneven_batch(d, seed=int(seed) % (1 << 31), walkers=case["walkers"], runs_per_side=1,
                                               interval=case["interval"], warmup=2, rnd_seed=1 + int(seed) % 100003)
            grp = mvmc_hip.EnsembleGroup([i["namelist"] for i in infos], [i["initial"] for i in infos],
                                         [case["walkers"]] * len(infos))
            return dict(case=case, group=grp, start=[e.params() for e in grp.runs])
        info = _files(case, seed, d)
        ens = mvmc_hip.Ensemble(info["namelist"], info["initial"], walkers=case["walkers"])
    s = dict(case=case, ens=ens, start=ens.params())
    if case.get("precision") == "mixed":
        ens.set_precision("mixed")
    if k == "configs":
        s["ele_idx"] = _configs(case, seed)
    if k == "vjp":
        ens.sample()
        s["cot"] = np.random.default_rng(int(seed) % (1 << 31)).standard_normal(case["walkers"]) / case["walkers"]
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _result(ens):
    oo, ho = ens.operands()
    proj, slater = ens.params()
    return dict(energy=ens.energy(), oo=oo, ho=ho, proj=proj, slater=slater)


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "pfinv":
        if c["complex"]:
            mvmc_hip.pfaffian_inverse_batched_c128(s["planes"], s["pf"], s["inv"], s["status"], c["n"], c["count"],
                                                   order=c["order"])
        else:
            mvmc_hip.pfaffian_inverse_batched(s["planes"], s["pf"], s["inv"], s["status"], c["n"], c["count"])
        return dict(pf=s["pf"], inv=s["inv"], status=s["status"])
    if k == "direct":
        n = c["na"] + 1
        (mvmc_hip.sr_gram_real_f32 if c["f32"] else mvmc_hip.sr_gram_real)(s["store"], s["gram"], n, c["rows"])
        mvmc_hip.sr_assemble_s_g(s["gram"], s["ho"], s["map"], c["na"], n, 1, 1e-3, 0.01, s["s"], s["g"])
        info = mvmc_hip.sr_cholesky_solve(s["s"], s["g"], c["na"])
        return dict(gram=s["gram"], x=s["g"], info=info)
    if k == "cg":
        status = mvmc_hip.sr_cg_solve(s["pack"], s["mean"], s["diag"], s["g"], s["x"], c["na"], c["rows"], 1,
                                      1.0 / c["rows"], CG["shift"], CG["tol"], CG["max_it"], variant=c["variant"])
        return dict(x=s["x"], status=status)
    if k == "group":
        for e, p in zip(s["group"].runs, s["start"]):
            e.set_params(*p)
        rows = s["group"].opt_step()
        return dict(rows=rows, runs=[_result(e) for e in s["group"].runs])
    ens = s["ens"]
    if k == "configs":
        e, o, ok = ens.measure_configs(s["ele_idx"])
        return dict(e=e, o=o, ok=ok)
    if k == "vjp":
        if c["form"] == "rows":
            ens.measure()
            return dict(grad=ens.vjp(s["cot"]), energy=ens.energy())
        return dict(log_psi=ens.log_psi(), grad=ens.vjp_adjoint(s["cot"]))
    ens.set_params(*s["start"])
    if k == "energy":
        ens.sample()
        ens.measure()
        return _result(ens)
    if c["direct"]:
        ens.sample()
        ens.measure()
        skipped = ens.sr_direct()
        return dict(_result(ens), skipped=skipped)
    row = ens.opt_step()
    return dict(_result(ens), row=row)


# ---------------------------------------------------------------------------
# the work that a pass cannot do without
# ---------------------------------------------------------------------------
def _pf_flops(n, cplx=False):
    # LTL of a skew matrix n^3/3 multiply-adds' worth, its inverse n^3
    return (4.0 if cplx else 1.0) * (2.0 * n ** 3 / 3.0 + n ** 3)


def _model(case):
    ns = case["L"] if case["lattice"] == "chain16" else case["L"] ** 2
    return ns, 2 * case["nup"], case["spgl"] * case["ntrans"]


def _sweep_work(ns, n, nqp, walkers, interval, outer):
    """Proposals: a row of the inverse and of the Slater table each; the update of a third of them that
    is accepted: the inverse read and written."""
    props = walkers * interval * ns * outer
    b = props * nqp * 2 * n * 8 + props / 3 * nqp * n * n * 16
    f = props * nqp * 2 * n + props / 3 * nqp * n * n * 6
    return b, f


def work(case):
    k = case["kind"]
    if k == "pfinv":
        n, c = case["n"], case["count"]
        size = 16 if case["complex"] else 8
        return dict(bytes=2.0 * c * n * n * size, flops=c * _pf_flops(n, case["complex"]))
    if k == "direct":
        n, rows, size = case["na"] + 1, case["rows"], 4 if case["f32"] else 8
        return dict(bytes=rows * n * size + 2.0 * n * n * 8, flops=float(rows) * n * n + n ** 3 / 3.0)
    if k == "cg":
        it = CG["max_it"]
        # one pass over the samples for each iteration
        return dict(bytes=float(case["rows"]) * case["na"] * 8 * it, flops=4.0 * case["rows"] * case["na"] * it)
    if k == "group":
        b = f = 0.0
        for L in lattice.UNEVEN_SIDES:
            ns, n, nqp = L * L, int(0.875 * L * L), 4
            x, y = _sweep_work(ns, n, nqp, case["walkers"], case["interval"], 2)
            b, f = b + x, f + y + case["walkers"] * nqp * 2 * _pf_flops(n)
        return dict(bytes=b, flops=f)
    ns, n, nqp = _model(case)
    planes = case["walkers"] * nqp
    if k in ("configs", "vjp"):
        return dict(bytes=planes * n * n * 8.0 * 2, flops=planes * _pf_flops(n) * (2 if k == "vjp" else 1))
    b, f = _sweep_work(ns, n, nqp, case["walkers"], case["interval"], case["samples"] + 1)
    return dict(bytes=b, flops=f + planes * (1 + case["samples"]) * _pf_flops(n))


# ---------------------------------------------------------------------------
# the same in 64 bits, without the library
# ---------------------------------------------------------------------------
def _pfaffian(a):
    """Pfaffians of a batch of skew planes: Parlett-Reid with pivoting, in torch."""
    a = a.clone()
    b, n = a.shape[0], a.shape[1]
    at = torch.arange(b, device=a.device)
    pf = torch.ones(b, dtype=a.dtype, device=a.device)
    for k in range(0, n - 1, 2):
        p = a[:, k + 1:, k].abs().argmax(dim=1) + k + 1
        row, other = a[:, k + 1].clone(), a[at, p].clone()
        a[:, k + 1], a[at, p] = other, row
        col, other = a[:, :, k + 1].clone(), a[at, :, p].clone()
        a[:, :, k + 1], a[at, :, p] = other, col
        pf = pf * torch.where(p == k + 1, 1.0, -1.0) * a[:, k, k + 1]
        if k + 2 < n:
            t = a[:, k, k + 2:] / a[:, k, k + 1, None]
            v = a[:, k + 2:, k + 1]
            u = t[:, :, None] * v[:, None, :]
            a[:, k + 2:, k + 2:] += u - u.transpose(1, 2)
    return pf


def _numbers(path, skip, cols):
    with open(path) as f:
        rows = [x.split() for x in f.readlines()[skip:]]
    return [r for r in rows if len(r) == cols]


def _exact_configs(case, seed):
    """Local energy and log-derivatives of the configurations from the model's input files alone."""
    ns, n, nqp = _model(case)
    ne, nleg, nmp = case["nup"], case["spgl"], case["ntrans"]
    with tempfile.TemporaryDirectory() as d:
        info = _files(case, seed, d)
        trans = np.array(_numbers(os.path.join(d, "trans.def"), 5, 6), dtype=float)
        inter = np.array(_numbers(os.path.join(d, "coulombintra.def"), 5, 2), dtype=float)
        jidx = np.full((ns, ns), -1)
        for i, j, c in np.array(_numbers(os.path.join(d, "jastrowidx.def"), 5, 3), dtype=int):
            jidx[i, j] = c
        oidx = np.zeros((ns, ns), dtype=int)
        for i, j, c in np.array(_numbers(os.path.join(d, "orbitalidx.def"), 5, 3), dtype=int):
            oidx[i, j] = c
        tmap = np.zeros((nmp, ns), dtype=int)
        for k, i, j, _ in np.array(_numbers(os.path.join(d, "qptransidx.def"), 5, 4), dtype=int):
            tmap[k, i] = j
        frozen = any(r[1] == "0" for r in _numbers(os.path.join(d, "jastrowidx.def"), 5 + ns * (ns - 1), 2))
        para = np.array(_numbers(info["initial"], 1, 3), dtype=float)[:, 0]
    ng, nj = info["n_gutz"], info["n_jast"]
    proj, orb = para[:ng + nj].copy(), para[ng + nj:].copy()
    if not frozen:
        proj -= proj.mean()
    orb *= 4.0 / np.abs(orb).max()
    w = np.ones(nqp)
    cs, cc, ss = np.zeros(nleg), np.ones(nleg), np.zeros(nleg)
    if nleg > 1:
        x, gw = np.polynomial.legendre.leggauss(nleg)
        beta, gw = np.pi / 2 * (x + 1), np.pi / 2 * gw
        cs, cc, ss = np.cos(beta / 2) * np.sin(beta / 2), np.cos(beta / 2) ** 2, np.sin(beta / 2) ** 2
        w = np.tile(0.5 * np.sin(beta) * gw, nmp)
    # Slater tables [nqp][2 ns][2 ns], and the derivative of each entry by the orbitals f_ij and f_ji
    S = np.zeros((nqp, 2 * ns, 2 * ns))
    for q in range(nqp):
        t, p = tmap[q // nleg], q % nleg
        fij = orb[oidx[np.ix_(t, t)]]
        fji = fij.T
        S[q, :ns, :ns], S[q, :ns, ns:] = -(fij - fji) * cs[p], fij * cc[p] + fji * ss[p]
        S[q, ns:, :ns], S[q, ns:, ns:] = -fij * ss[p] - fji * cc[p], (fij - fji) * cs[p]
    T = lambda a: torch.as_tensor(a, device=DEV)  # noqa: E731
    S, w = T(S), T(w)
    cfg = T(_configs(case, seed).astype(np.int64))
    rs = cfg + torch.cat([torch.zeros(ne), torch.full((ne,), ns)]).long().to(DEV)
    count = cfg.shape[0]
    occ = torch.zeros(count, 2 * ns, dtype=torch.float64, device=DEV).scatter_(1, rs, 1.0)
    who = torch.zeros(count, 2 * ns, dtype=torch.int64, device=DEV).scatter_(1, rs, torch.arange(n, device=DEV).expand(count, n))
    m = occ[:, :ns] + occ[:, ns:] - 1.0
    double = occ[:, :ns] * occ[:, ns:]
    J = T(np.where(jidx >= 0, proj[ng + np.maximum(jidx, 0)], 0.0))
    Jm = m @ J
    e = double @ T(inter[:, 1])
    o = torch.zeros(count, info["npara"] + 1, dtype=torch.float64, device=DEV)
    o[:, 0] = 1.0
    o[:, 1] = double.sum(dim=1)
    pairs = T(np.triu(np.ones((ns, ns)), 1))
    for a in range(0, count, 64):
        z = slice(a, min(count, a + 64))
        mm = (m[z, :, None] * m[z, None, :] * pairs).reshape(-1, ns * ns)
        cls = T(np.where(jidx >= 0, jidx, 0).reshape(-1))
        o[z, 1 + ng:1 + ng + nj] = torch.zeros(mm.shape[0], nj, dtype=torch.float64, device=DEV).index_add_(1, cls, mm)
        r = rs[z]
        A = S[:, r[:, :, None], r[:, None, :]]  # [nqp][b][n][n]
        pf = _pfaffian(A.reshape(-1, n, n)).reshape(nqp, -1)
        X = torch.linalg.inv(A)
        part = w[:, None] * pf
        part = part / part.sum(dim=0)
        # hop of electron k to (site, spin): the new row of A against column k of its inverse
        ratio = torch.zeros(r.shape[0], 2 * ns, n, dtype=torch.float64, device=DEV)
        bar = torch.zeros(r.shape[0], nqp, 2 * ns, 2 * ns, dtype=torch.float64, device=DEV)
        b = torch.arange(r.shape[0], device=DEV)
        for q in range(nqp):
            rows = S[q][:, r].permute(1, 0, 2).contiguous()  # [b][2 ns][n]
            ratio += part[q][:, None, None] * torch.matmul(rows, X[q].contiguous())
            bar[b[:, None, None], q, r[:, :, None], r[:, None, :]] = part[q][:, None, None] * X[q].transpose(1, 2) / 2
        for q in range(nqp):
            t, p = tmap[q // nleg], q % nleg
            g = bar[:, q]
            fij = -g[:, :ns, :ns] * cs[p] + g[:, :ns, ns:] * cc[p] - g[:, ns:, :ns] * ss[p] + g[:, ns:, ns:] * cs[p]
            fji = g[:, :ns, :ns] * cs[p] + g[:, :ns, ns:] * ss[p] - g[:, ns:, :ns] * cc[p] - g[:, ns:, ns:] * cs[p]
            both = (fij + fji.transpose(1, 2)).reshape(r.shape[0], -1)
            o[z, 1 + ng + nj:].index_add_(1, T(oidx[np.ix_(t, t)].reshape(-1)), both)
        for i, s, j, _, t, _ in trans:
            i, s, j = int(i), int(s), int(j)
            to, frm = i + s * ns, j + s * ns
            can = occ[z, frm] * (1.0 - occ[z, to])
            lp = proj[0] * (occ[z, i + (1 - s) * ns] - occ[z, j + (1 - s) * ns]) + Jm[z, i] - Jm[z, j] - J[i, j]
            e[z] -= t * can * torch.exp(lp) * ratio[b, to, who[z, frm]]
    return dict(e=e.cpu().numpy(), o=o.cpu().numpy(), ok=None)


def exact(case, seed):
    k = case["kind"]
    if k == "pfinv":
        a = _planes(case, seed).transpose(1, 2).contiguous()  # the library reads planes column by column
        pf = torch.cat([_pfaffian(x) for x in a.split(256)])
        inv = np.linalg.inv(a.cpu().numpy()).transpose(0, 2, 1)
        return dict(pf=pf, inv=np.ascontiguousarray(inv), status=None)
    if k == "direct":
        s = prepare(case, seed)
        st = s["store"].double()
        gram = st.t().contiguous() @ st
        S = gram[1:, 1:] - torch.outer(gram[0, 1:], gram[0, 1:])
        S.diagonal().mul_(1.0 + 1e-3)
        g = -0.02 * (s["ho"][1:] - s["ho"][0] * gram[0, 1:])
        return dict(gram=gram, x=torch.linalg.solve(S, g), info=None)
    if k == "cg":
        pack, mean, diag, g = _cg_operands(case, seed)

        def apply(v):
            return (pack.t() @ (pack @ v)) / case["rows"] - torch.dot(mean, v) * mean + CG["shift"] * diag * v

        pre = (1.0 + CG["shift"]) * diag if case["variant"] else torch.ones_like(diag)
        x, r = torch.zeros_like(g), g.clone()
        d = r / pre
        delta = torch.dot(r, d)
        threshold = CG["tol"] ** 2 * case["na"] ** 2
        for it in range(CG["max_it"]):
            if abs(float(delta)) < threshold:
                break
            q = apply(d)
            alpha = delta / torch.dot(d, q)
            x = x + alpha * d
            r = g - apply(x) if (it + 1) % 20 == 0 else r - alpha * q
            z = r / pre
            new = torch.dot(r, z)
            d = z + new / delta * d
            delta = new
        return dict(x=x, status=None)
    if k == "configs":
        return _exact_configs(case, seed)
    return None  # Markov chains: what they visit has no value apart from the library's own draws
