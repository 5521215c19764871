"""The work that users of this package have it do, as cases that a timing
program can prepare and run through the public entry points.

A case is a dict of plain values with its ``kind``:

* ``box``     one periodic-box catalogue in device memory -> P_l(k)
              (Context.run_device), the call of an analysis of simulations;
* ``batch``   many mocks of uneven sizes in one call (Context.run_batch,
              replayed as a captured graph), the call of a covariance run;
* ``survey``  data and randoms in device memory -> local-line-of-sight
              multipoles (Context.run_survey_device);
* ``cross``   two host catalogues -> both auto spectra and the cross spectrum
              (Context.run_host), uploads included;
* ``alias``   a plain grid with the learned alias correction (the shipped
              networks) in place of the interlaced second grid;
* ``ascii``   a text catalogue -> device records (Ingest.start_ascii);
* ``cnvt``    (RA, Dec, z) -> comoving coordinates in place (cnvt_device).

Inputs are made from the seed alone with torch; ``exact`` evaluates the same
estimators in 64 bits with torch and numpy only.
"""
from __future__ import annotations

import ctypes
import math
import tempfile

import numpy as np
import torch

import powspec_amd as P
from powspec_amd import mlp

SIDE = 1000.0                      # box side of the repository's catalogues
OMEGA_M = 0.31
RA, DEC = (0.0, 60.0), (-30.0, 30.0)
Z_MU, Z_SIGMA, Z_LO, Z_HI = 0.55, 0.08, 0.4, 0.7
NBAR0, P0 = 5e-3, 1e4
POLES = {"0": [0], "02": [0, 2], "024": [0, 2, 4], "0to4": [0, 1, 2, 3, 4]}
GRIDS = [48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512, 640, 768, 1024]


# ---- the cases ------------------------------------------------------------

def _box(grid, npart, assign, intlace, **kw):
    c = dict(kind="box", grid=grid, npart=npart, assign=assign, intlace=intlace,
             poles="024", kbin=0.01, kmax=0.0, log=False, los=2, order="grid",
             weights=False)
    c.update(kw)
    return c


def listed():
    return [
        # a small simulation, one call among thousands of a parameter scan
        dict(_box(64, 20_000, P.CIC, False), name="box 64 CIC 2e4"),
        # the plain configuration: 1e6 particles, CIC, no interlacing
        dict(_box(256, 1_000_000, P.CIC, False), name="box 256 CIC 1e6"),
        # a galaxy or halo list ordered by mass (so random in space), with
        # completeness weights, measured up to k_max = 0.4
        dict(_box(512, 4_000_000, P.TSC, True, order="random", weights=True, kmax=0.4),
             name="box 512 TSC 4e6 shuffled"),
        # a grid size between the powers of two, log bins, line of sight on x,
        # odd poles as well
        dict(_box(640, 6_000_000, P.PCS, True, log=True, kbin=0.05, los=0, poles="0to4"),
             name="box 640 PCS log bins"),
        # the production box: 2e7 clustered particles, PCS, interlaced
        dict(_box(1024, 20_000_000, P.PCS, True, kbin=0.005), name="box 1024 PCS 2e7"),
        # the mocks of a covariance matrix, uneven sizes, one graph replay
        dict(kind="batch", nmock=32, grid=256, nmin=200_000, nmax=3_000_000, assign=P.TSC,
             intlace=True, name="batch 32 x 256 TSC"),
        # a small survey without interlacing, quadrupole only
        dict(kind="survey", grid=256, ndata=200_000, nrand=2_000_000, assign=P.TSC,
             intlace=False, poles="02", name="survey 256 TSC 2e6"),
        # the survey workload: 5e6 objects, 1e8 randoms, CIC, interlaced
        dict(kind="survey", grid=512, ndata=5_000_000, nrand=100_000_000, assign=P.CIC,
             intlace=True, poles="024", name="survey 512 CIC 1e8"),
        # two tracers of one box from host memory, auto and cross spectra
        dict(kind="cross", grid=256, npart=1_000_000, npart2=400_000, assign=P.TSC,
             intlace=True, name="cross 256 TSC host"),
        # the learned correction in place of interlacing
        dict(kind="alias", grid=512, npart=20_000_000, name="alias 512 CIC 2e7"),
        # a text catalogue of a simulation, x y z w
        dict(kind="ascii", lines=1_000_003, name="ascii 1e6 lines"),
        # a random catalogue of a survey to comoving coordinates
        dict(kind="cnvt", n=20_000_001, name="cnvt 2e7"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box", "box", "box", "batch", "survey", "cross", "alias", "ascii",
                       "cnvt"])
    if kind == "box":
        log = rng.random() < 0.25
        return _box(rng.choice(GRIDS), _log_int(rng, 1e4, 2e7), rng.randrange(4),
                    rng.random() < 0.6, log=log, kbin=0.05 if log else rng.choice([0.005, 0.01]),
                    kmax=0.0 if log else rng.choice([0.0, 0.0, 0.2, 0.4]), los=rng.randrange(3),
                    poles=rng.choice(["0", "02", "024", "024", "0to4"]),
                    order=rng.choice(["grid", "random"]), weights=rng.random() < 0.5)
    if kind == "batch":
        grid = rng.choice([64, 128, 192, 256])
        nmin = _log_int(rng, 2e4, 4e5)
        return dict(kind="batch", nmock=rng.randrange(2, 33), grid=grid, nmin=nmin,
                    nmax=int(nmin * rng.uniform(1.5, 7.0)), assign=rng.randrange(1, 4),
                    intlace=rng.random() < 0.7)
    if kind == "survey":
        nd = _log_int(rng, 5e4, 2e6)
        return dict(kind="survey", grid=rng.choice([128, 192, 256, 320, 384, 512]), ndata=nd,
                    nrand=int(nd * rng.uniform(5, 30)), assign=rng.randrange(1, 4),
                    intlace=rng.random() < 0.6, poles=rng.choice(["0", "02", "024"]))
    if kind == "cross":
        n = _log_int(rng, 1e5, 1.5e6)
        return dict(kind="cross", grid=rng.choice([128, 192, 256, 320]), npart=n,
                    npart2=int(n * rng.uniform(0.2, 1.0)), assign=rng.randrange(1, 4),
                    intlace=rng.random() < 0.6)
    if kind == "alias":
        return dict(kind="alias", grid=rng.choice([256, 384, 512]), npart=_log_int(rng, 2e6, 2e7))
    if kind == "ascii":
        return dict(kind="ascii", lines=_log_int(rng, 1e4, 2e6))
    return dict(kind="cnvt", n=_log_int(rng, 1e4, 5e7))


# ---- inputs ---------------------------------------------------------------

class Records:
    """psh_data records (x, y, z, w) held by a torch tensor [n, 4]."""

    def __init__(self, t):
        self.tensor = t
        self.ptr = ctypes.c_void_p(t.data_ptr())
        self.nbytes = t.numel() * 8


def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(n, g):
    return torch.rand(n, generator=g, dtype=torch.float64, device="cuda")


def _clustered(npart, seed, order="grid", weights=False):
    """About npart particles of a lognormal field in [0, SIDE)^3 with a
    redshift-space shift along z, in the order of the generator's cells or
    shuffled."""
    g = _rng(seed)
    ng = 64 if npart < 300_000 else (128 if npart < 3_000_000 else 256)
    kf = 2 * math.pi / SIDE
    kx = torch.fft.fftfreq(ng, d=1.0 / ng, device="cuda") * kf
    kz = torch.arange(ng // 2 + 1, device="cuda") * kf
    k2 = kx[:, None, None] ** 2 + kx[None, :, None] ** 2 + kz[None, None, :] ** 2
    k = torch.sqrt(k2).clamp_min(kf)
    pk = 1e4 * (k / 0.1) ** -1.5 * torch.exp(-((k / 0.5) ** 2))
    dk = torch.fft.rfftn(torch.randn((ng, ng, ng), generator=g, device="cuda"))
    dk = dk * torch.sqrt(pk * (ng / SIDE) ** 3) * (k2 > 0)
    delta = torch.fft.irfftn(dk, s=(ng, ng, ng))
    psi = torch.fft.irfftn(dk * (1j * kz / k2.clamp_min(kf * kf)), s=(ng, ng, ng))
    lam = npart / ng ** 3 * torch.exp(delta - 0.5 * delta.var())
    counts = torch.poisson(lam, generator=g).to(torch.int64).reshape(-1)
    cell = torch.repeat_interleave(torch.arange(ng ** 3, device="cuda"), counts)
    n = cell.numel()
    h = SIDE / ng
    d = torch.empty((n, 4), dtype=torch.float64, device="cuda")
    d[:, 0] = (cell // (ng * ng) + _uniform(n, g)) * h
    d[:, 1] = (cell // ng % ng + _uniform(n, g)) * h
    d[:, 2] = (cell % ng + _uniform(n, g)) * h + 0.8 * psi.reshape(-1)[cell]
    d[:, :3] = torch.remainder(d[:, :3], SIDE).clamp_max(SIDE * (1 - 4e-16) - 1e-9 * SIDE)
    d[:, 3] = 0.5 + _uniform(n, g) if weights else 1.0
    if order == "random":
        d = d[torch.randperm(n, generator=g, device="cuda")].contiguous()
    return d


def _distance(z):
    """Comoving distance [Mpc/h] in flat LCDM, 64-point Gauss-Legendre."""
    x, w = np.polynomial.legendre.leggauss(64)
    out = torch.zeros_like(z)
    for a, b in zip(x, w):
        out += float(b) / torch.sqrt(OMEGA_M * (1 + 0.5 * z * (1 + float(a))) ** 3 + 1 - OMEGA_M)
    return out * (0.5 * 2997.92458) * z


def _sky(n, g):
    """RA, Dec [deg], z of a sky cap with a truncated Gaussian n(z)."""
    ra = RA[0] + (RA[1] - RA[0]) * _uniform(n, g)
    s0, s1 = (math.sin(math.radians(v)) for v in DEC)
    dec = torch.rad2deg(torch.asin(s0 + (s1 - s0) * _uniform(n, g)))
    pa, pb = (0.5 * math.erfc(-(v - Z_MU) / Z_SIGMA / math.sqrt(2)) for v in (Z_LO, Z_HI))
    z = Z_MU + Z_SIGMA * math.sqrt(2) * torch.erfinv(2 * (pa + (pb - pa) * _uniform(n, g)) - 1)
    return ra, dec, z


def _survey_cat(n, seed):
    """(records in comoving coordinates with FKP weights, n(z))."""
    ra, dec, z = _sky(n, _rng(seed))
    zt = torch.linspace(Z_LO - 0.01, Z_HI + 0.01, 4097, dtype=torch.float64, device="cuda")
    dt = _distance(zt)
    u = (z - zt[0]) * (4096 / (zt[-1] - zt[0]))
    i = u.to(torch.int64).clamp_(0, 4095)
    r = dt[i] + (u - i) * (dt[i + 1] - dt[i])
    del u, i
    nz = NBAR0 * torch.exp(-0.5 * ((z - Z_MU) / Z_SIGMA) ** 2)
    d = torch.empty((n, 4), dtype=torch.float64, device="cuda")
    ra, dec = torch.deg2rad(ra), torch.deg2rad(dec)
    d[:, 0] = r * torch.cos(dec) * torch.cos(ra)
    d[:, 1] = r * torch.cos(dec) * torch.sin(ra)
    d[:, 2] = r * torch.sin(dec)
    d[:, 3] = 1 / (1 + nz * P0)
    return d, nz


def _survey_inputs(case, seed):
    d, _ = _survey_cat(case["ndata"], 2 * seed)
    r, nz = _survey_cat(case["nrand"], 2 * seed + 1)
    a = case["ndata"] / case["nrand"]
    w2 = r[:, 3] ** 2
    return d, r, a, float((d[:, 3] ** 2).sum() + a * a * w2.sum()), float(a * (w2 * nz).sum())


def _batch_inputs(case, seed):
    sizes = np.random.default_rng(seed).integers(case["nmin"], case["nmax"] + 1, case["nmock"])
    return [_clustered(int(n), 1000 * seed + m) for m, n in enumerate(sizes)]


def _ascii_ints(lines, seed):
    """Positions in units of 1e-6 and weights in units of 1e-4."""
    g = _rng(seed)
    v = torch.randint(0, int(SIDE) * 10 ** 6, (lines, 3), generator=g, device="cuda")
    return torch.cat([v, torch.randint(5000, 15000, (lines, 1), generator=g, device="cuda")], 1)


def _ascii_bytes(v):
    """Lines "xxx.xxxxxx yyy.yyyyyy zzz.zzzzzz w.wwww", blank-padded."""
    cols = []
    for a, (whole, frac) in enumerate([(3, 6)] * 3 + [(1, 4)]):
        for k in range(whole - 1, -1, -1):
            q = v[:, a] // 10 ** (k + frac)
            cols.append(torch.where((q == 0) & (k > 0), 32, q % 10 + 48))
        cols.append(torch.full_like(v[:, a], 46))
        for k in range(frac - 1, -1, -1):
            cols.append(v[:, a] // 10 ** k % 10 + 48)
        cols.append(torch.full_like(v[:, a], 10 if a == 3 else 32))
    return torch.stack(cols, 1).to(torch.uint8)


def _conf_kw(case):
    kind = case["kind"]
    kw = dict(gsize=case["grid"], assign=case.get("assign", P.CIC),
              intlace=case.get("intlace", False), kbin=case.get("kbin", 0.01),
              poles=POLES[case.get("poles", "024")])
    if kind == "survey":
        kw.update(issim=False)
    else:
        kw.update(bsize=SIDE)
    if kind == "box":
        kw.update(los=[float(a == case["los"]) for a in range(3)])
        if case["log"]:
            kw.update(logscale=True, kmin=-2.0)
        if case["kmax"] > 0:
            kw.update(kmax=case["kmax"])
    if kind == "cross":
        kw.update(ndata=2, isauto=[True, True], iscross=True)
    return kw


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("box", "alias"):
        s["data"] = Records(_clustered(case["npart"], seed, case.get("order", "grid"),
                                       case.get("weights", False)))
        s["n"] = len(s["data"].tensor)
        s["wsum"] = float(s["data"].tensor[:, 3].sum())
    elif kind == "batch":
        cats = _batch_inputs(case, seed)
        s["offsets"] = np.concatenate([[0], np.cumsum([len(c) for c in cats])]).tolist()
        s["wsums"] = [float(len(c)) for c in cats]
        s["data"] = Records(torch.cat(cats))
    elif kind == "survey":
        d, r, s["alpha"], s["shot"], s["norm"] = _survey_inputs(case, seed)
        s["data"], s["rand"] = Records(d), Records(r)
    elif kind == "cross":
        s["data"] = [_clustered(n, 2 * seed + c).cpu().numpy()
                     for c, n in enumerate((case["npart"], case["npart2"]))]
    elif kind == "ascii":
        s["file"] = tempfile.NamedTemporaryFile(prefix="psh_case_", suffix=".txt")
        _ascii_bytes(_ascii_ints(case["lines"], seed)).cpu().numpy().tofile(s["file"].name)
        s["out"] = Records(torch.empty((case["lines"], 4), dtype=torch.float64, device="cuda"))
        s["ingest"] = P.Ingest()
    else:
        ra, dec, z = _sky(case["n"], _rng(seed))
        s["sky"] = torch.stack([ra, dec, z, torch.ones_like(z)], 1)
        s["out"] = Records(torch.empty_like(s["sky"]))
        s["cnvt"] = P.make_cnvt(omega_m=OMEGA_M)
    if kind not in ("ascii", "cnvt"):
        s["ctx"] = P.Context(P.make_conf(**_conf_kw(case)), nmock_max=case.get("nmock", 1))
    if kind == "alias":
        s["ctx"].set_mu_cells(mlp.NMU)
        s["ctx"].set_alias_mlp(mlp.load_params())
    torch.cuda.synchronize()      # the library's streams do not wait for torch's
    return s


def run(s):
    kind = s["kind"]
    if kind in ("box", "alias"):
        return s["ctx"].run_device(s["data"], s["n"], s["wsum"])
    if kind == "batch":
        res = s["ctx"].run_batch(s["data"], s["offsets"], s["wsums"], graph=True)
        return {q: np.stack([r[q] for r in res]) for q in ("k", "km", "cnt", "lcnt")} | {
            "pl": np.stack([r["pl"][0] for r in res])}
    if kind == "survey":
        return s["ctx"].run_survey_device(s["data"], len(s["data"].tensor), s["rand"],
                                          len(s["rand"].tensor), s["alpha"], s["shot"],
                                          s["norm"])
    if kind == "cross":
        return s["ctx"].run_host(s["data"])
    if kind == "ascii":
        s["ingest"].start_ascii(s["file"].name, s["out"], len(s["out"].tensor),
                                fmtr="%lf %lf %lf %lf", wcomp=4)
        r = s["ingest"].wait()
        return {"records": s["out"].tensor, "n": r["n"], "sumw": r["sumw"]}
    s["out"].tensor.copy_(s["sky"])          # the conversion is in place
    order = P.cnvt_device(s["cnvt"], [(s["out"], len(s["sky"]))])
    return {"records": s["out"].tensor, "order": order}


def work(case):
    """Inputs read once and outputs written once; the FFTs, the windows and
    about 20 operations per mode and pole."""
    kind = case["kind"]
    if kind == "ascii":
        return {"bytes": case["lines"] * (40.0 + 32.0), "flops": case["lines"] * 80.0}
    if kind == "cnvt":
        return {"bytes": case["n"] * 56.0, "flops": case["n"] * 200.0}
    n = {"box": lambda: case["npart"], "alias": lambda: case["npart"],
         "batch": lambda: case["nmock"] * (case["nmin"] + case["nmax"]) / 2,
         "survey": lambda: case["ndata"] + case["nrand"],
         "cross": lambda: case["npart"] + case["npart2"]}[kind]()
    N = float(case["grid"])
    poles = POLES[case.get("poles", "024")]
    grids = 2 if case.get("intlace") else 1
    fields = {"batch": case.get("nmock", 1), "cross": 2}.get(kind, 1)
    fft = 2.5 * N ** 3 * math.log2(N ** 3)
    flops = fields * (grids * fft + 10.0 * N ** 3 * len(poles))
    flops += grids * n * 2.0 * (case.get("assign", P.CIC) + 1) ** 3
    if kind == "survey":
        flops += sum(2 * l + 1 for l in poles[1:]) * (fft + 20.0 * N ** 3)
    nb = N / (2 * SIDE) * 2 * math.pi / case.get("kbin", 0.01)
    return {"bytes": 32.0 * n + 8.0 * fields * nb * (4 + 2 * len(poles)), "flops": flops}


# ---- the same in 64 bits --------------------------------------------------

def _window(x, assign):
    """First cell and weights of a particle along one axis."""
    i = x.floor()
    d = x - i
    if assign == P.NGP:
        return i + (d >= 0.5), [torch.ones_like(d)]
    if assign == P.CIC:
        return i, [1 - d, d]
    if assign == P.TSC:
        up = d >= 0.5
        d = d - up.to(d.dtype)
        return i - 1 + up, [0.5 * (0.5 - d) ** 2, 0.75 - d * d, 0.5 * (0.5 + d) ** 2]
    return i - 1, [(1 - d) ** 3 / 6, (4 - 6 * d * d + 3 * d ** 3) / 6,
                   (1 + 3 * (d + d * d - d ** 3)) / 6, d ** 3 / 6]


def _mesh(cats, N, L, corner, assign):
    """Density of [(records, scale)] on the N^3 grid with its corner there."""
    rho = torch.zeros(N ** 3, dtype=torch.float64, device="cuda")
    for d, scale in cats:
        for part in torch.split(d, 1 << 23):
            ax = []
            for a in range(3):
                p = part[:, a]
                p = torch.where(p >= corner[a] + L[a], p - L[a], p)
                b, w = _window((p - corner[a]) * N / L[a], assign)
                ax.append((b.to(torch.int64), w))
            wt = part[:, 3] * scale
            for i, wx in enumerate(ax[0][1]):
                ix = torch.remainder(ax[0][0] + i, N) * N
                for j, wy in enumerate(ax[1][1]):
                    iy = (ix + torch.remainder(ax[1][0] + j, N)) * N
                    for k, wz in enumerate(ax[2][1]):
                        rho.index_add_(0, iy + torch.remainder(ax[2][0] + k, N),
                                       wt * wx * wy * wz)
    return rho.view(N, N, N)


def _freq(N):
    i = torch.arange(N, dtype=torch.float64, device="cuda")
    return torch.where(i <= N // 2, i, i - N)


def _field(cats, N, L, bmin, assign, intlace):
    """F(k) of the catalogues' density, interlaced when asked for."""
    F = torch.fft.rfftn(_mesh(cats, N, L, bmin, assign))
    if not intlace:
        return F
    G = torch.fft.rfftn(_mesh(cats, N, L, [b - 0.5 * l / N for b, l in zip(bmin, L)], assign))
    ph = torch.exp(1j * math.pi / N * _freq(N))
    G *= ph[:, None, None]
    G *= ph[None, :, None]
    G *= ph[None, None, : N // 2 + 1]
    F += G
    F *= 0.5
    return F


def _alias(N, assign, intlace):
    """Alias factors per signed index; the series is used for all small or
    negative arguments, as the estimator defines them."""
    out = []
    for s in _freq(N).tolist():
        x = s * math.pi / N
        t = x * x
        if intlace:
            f = x / math.sin(x) if x > 0.01 else 1 + t / 6 + 7 * t * t / 360 + 31 * t ** 3 / 15120
            out.append(f ** (2 * (assign + 1)))
            continue
        f = (math.sin(x) if x > 0.01 else (1 - t / 6 + t * t / 120 - t ** 3 / 5040) * x) ** 2
        out.append([1.0, 1 / (1 - 2 / 3 * f), 1 / (1 - f + 2 / 15 * f * f),
                    1 / (1 - 4 / 3 * f + 0.4 * f * f - 4 / 315 * f ** 3)][assign])
    return torch.tensor(out, dtype=torch.float64, device="cuda")


def _legendre(l, x):
    a, b = torch.ones_like(x), x
    for n in range(1, l + 1):
        a, b = b, ((2 * n + 1) * x * b - n * a) / (n + 1)
    return a


def _bins(N, L, kw):
    log = kw.get("logscale", False)
    kmin, dk, kmax = kw.get("kmin", 0.0), kw["kbin"], kw.get("kmax", -1.0)
    kny = math.pi * N / max(L)
    if log:
        kny = math.log10(kny)
    top = min(kny, kmax) if kmax > 0 else kny
    nb = int(math.floor((top - kmin) / dk + 0.5))
    if kmin + dk * nb > kny:
        nb -= 1
    return nb, kmin + dk * np.arange(nb + 1)


def _modes(N, L, kw):
    """Slabs of modes: (slab, bin, multiplicity, |k|, alias, mu) with the bin
    nb outside the binning."""
    nb, edge = _bins(N, L, kw)
    M = N // 2
    k = [_freq(N) * (2 * math.pi / l) for l in L]
    al = _alias(N, kw["assign"], kw["intlace"])
    mult = torch.full((M + 1,), 2.0, dtype=torch.float64, device="cuda")
    mult[0] = mult[M] = 1.0
    los = kw.get("los", [0, 0, 1])
    kz = k[2][: M + 1]
    step = max(1, (1 << 26) // (N * (M + 1)))
    for i in range(0, N, step):
        sl = slice(i, min(N, i + step))
        kx = k[0][sl][:, None, None]
        k2 = (kx ** 2 + k[1][None, :, None] ** 2) + kz[None, None, :] ** 2
        km = torch.sqrt(k2)
        mu = (kx * los[0] + k[1][None, :, None] * los[1] + kz[None, None, :] * los[2])
        mu = mu / km.clamp_min(1e-300)
        q = 0.5 * torch.log10(k2) if kw.get("logscale") else km
        b = ((q - float(edge[0])) / kw["kbin"]).clamp(0, nb).to(torch.int64)
        b = torch.where((q >= float(edge[0])) & (q < float(edge[-1])) & (b < nb), b, nb)
        a = al[sl][:, None, None] * al[None, :, None] * al[None, None, : M + 1]
        yield sl, b, mult.expand_as(km), km, a, mu


def _sum(b, w, nb):
    return torch.bincount(b.reshape(-1), weights=w.reshape(-1), minlength=nb + 1)[:nb]


def _legsums(N, L, kw, nmu=1):
    """Mode counts, mean |k| and Legendre sums of the bins."""
    nb, edge = _bins(N, L, kw)
    cnt, km = (torch.zeros(nb, dtype=torch.float64, device="cuda") for _ in range(2))
    lc = torch.zeros((len(kw["poles"]), nb), dtype=torch.float64, device="cuda")
    for _, b, m, k, _, mu in _modes(N, L, kw):
        cnt += _sum(b, m, nb)
        km += _sum(b, k * m, nb)
        m = m * (k > 0)
        for n, l in enumerate(kw["poles"]):
            lc[n] += _sum(b, (m if l % 2 == 0 else m * (m == 1)) * _legendre(l, mu), nb)
    return cnt, km / cnt.clamp_min(1), lc


def _power(N, L, kw, F, G=None, nmu=1):
    """Raw sums of Re(F G*) alias mult L_l(mu) per pole, bin and |mu| cell."""
    nb, _ = _bins(N, L, kw)
    out = torch.zeros((len(kw["poles"]), nb * nmu), dtype=torch.float64, device="cuda")
    for sl, b, m, k, a, mu in _modes(N, L, kw):
        f, g = F[sl], F[sl] if G is None else G[sl]
        p = (f.real * g.real + f.imag * g.imag) * a * m * (k > 0)
        if nmu > 1:
            b = b * nmu + (mu.abs() * nmu).clamp(0, nmu - 1).to(torch.int64) * (b < nb)
        for n, l in enumerate(kw["poles"]):
            out[n] += _sum(b, (p if l % 2 == 0 else p * (m == 1)) * _legendre(l, mu), nb * nmu)
    return out


def _np(t):
    return t.cpu().numpy()


def _box_pl(raw, cnt, lc, poles, wsum, shot=True):
    vol = SIDE ** 3
    v = raw / (wsum * wsum / vol) / cnt.clamp_min(1)
    if shot:
        v = v - vol / wsum * lc / cnt.clamp_min(1)
    v = torch.where(cnt > 0, v, 0.0)
    return _np(v * torch.tensor([2 * l + 1.0 for l in poles], device="cuda")[:, None])


def _axis(N, L, kw, km):
    """k, edges and mean k as the estimator reports them (with log bins the
    lower edges and mean k follow from the rescaled centres)."""
    nb, e = _bins(N, L, kw)
    c = 0.5 * (e[1:] + e[:-1])
    if not kw.get("logscale"):
        return c, e, _np(km)
    c = 10.0 ** c
    return c, np.append(10.0 ** c, 10.0 ** e[-1]), 10.0 ** c


def _ylm(l, m, x, y, z):
    """Real Y_lm of unit vectors, without the Condon-Shortley phase."""
    am = abs(m)
    a = math.prod(range(2 * am - 1, 0, -2)) * torch.ones_like(z)
    b = (2 * am + 1) * z * a
    for n in range(am + 1, l + 1):
        a, b = b, ((2 * n + 1) * z * b - (n + am) * a) / (n - am + 1)
    c, s = torch.ones_like(x), torch.zeros_like(x)
    for _ in range(am):
        c, s = c * x - s * y, s * x + c * y
    nrm = (2 * l + 1) / (4 * math.pi) * math.factorial(l - am) / math.factorial(l + am)
    return math.sqrt(nrm * (2 if m else 1)) * a * (s if m < 0 else c)


def _unit(x, y, z):
    r = torch.sqrt(x * x + y * y + z * z).clamp_min(1e-300)
    return x / r, y / r, z / r


def _survey_exact(case, kw, seed):
    d, r, alpha, shot, norm = _survey_inputs(case, seed)
    N, poles = case["grid"], kw["poles"]
    lo = torch.minimum(d[:, :3].amin(0), r[:, :3].amin(0)).tolist()
    hi = torch.maximum(d[:, :3].amax(0), r[:, :3].amax(0)).tolist()
    L = [math.ceil((b - a) * 1.02 / 10) * 10.0 for a, b in zip(lo, hi)]
    bmin = [(a + b - l) * 0.5 for a, b, l in zip(lo, hi, L)]
    cats = [(d, 1.0), (r, -alpha)]
    if kw["intlace"]:
        F = _field(cats, N, L, bmin, kw["assign"], True)
        rho = torch.fft.irfftn(F, s=(N, N, N))
    else:
        rho = _mesh(cats, N, L, bmin, kw["assign"])
        F = torch.fft.rfftn(rho)
    nb, _ = _bins(N, L, kw)
    M = N // 2
    cnt, km, _ = _legsums(N, L, dict(kw, poles=[0]))
    S = torch.zeros((len(poles), nb), dtype=torch.float64, device="cuda")
    for sl, b, m, _, a, _ in _modes(N, L, kw):
        S[0] += _sum(b, (F[sl].real ** 2 + F[sl].imag ** 2) * a * m, nb)
    idx = torch.arange(N, dtype=torch.float64, device="cuda")
    pos = [(idx + bmin[a] * N / L[a]) * L[a] for a in range(3)]
    fr = [_freq(N) / l for l in L]
    for n, l in enumerate(poles[1:], 1):
        for mm in range(-l, l + 1):
            W = torch.empty_like(rho)
            for i in range(N):
                u = _unit(*torch.broadcast_tensors(pos[0][i], pos[1][:, None], pos[2][None, :]))
                W[i] = rho[i] * _ylm(l, mm, *u)
            W[0, 0] = rho[0, 0]
            W = torch.fft.rfftn(W)
            for sl, b, m, _, a, _ in _modes(N, L, kw):
                q = torch.broadcast_tensors(fr[0][sl][:, None, None], fr[1][None, :, None],
                                            fr[2][None, None, : M + 1])
                y = torch.where((q[0] == 0) & (q[1] == 0), 1.0, _ylm(l, mm, *_unit(*q)))
                f, g = F[sl], W[sl]
                S[n] += _sum(b, (f.real * g.real + f.imag * g.imag) * y * a * m, nb)
            del W
    c = cnt.clamp_min(1)
    S[0] = (S[0] / c - shot) / norm
    S[1:] *= 4 * math.pi / norm / c
    k, e, km = _axis(N, L, kw, km)
    return {"k": k, "kedge": e, "km": km, "pl": [_np(S), None]}


def _alias_exact(case, kw, seed):
    N, L, nmu = case["grid"], [SIDE] * 3, mlp.NMU
    d = _clustered(case["npart"], seed)
    wsum = float(len(d))
    cells = _power(N, L, kw, _field([(d, 1.0)], N, L, [0.0] * 3, P.CIC, False), nmu=nmu)
    cnt, km, lc = _legsums(N, L, kw)
    nb, e = _bins(N, L, kw)
    cells = cells.view(3, nb, nmu)
    S = cells[0].sum(1)
    p = _np(S / (wsum * wsum / SIDE ** 3) / cnt.clamp_min(1) / (SIDE ** 3 / wsum))
    kny = math.pi * N / SIDE
    k = 0.5 * (e[1:] + e[:-1])
    X = np.zeros((nb, nmu, 32))
    for q in range(16):
        b0, b1 = (kny * (0.25 + 0.75 * (q + t) / 16) for t in (0, 1))
        sel = (k >= b0) & (k < b1) & (p > 0)
        near = np.argmin(np.where(p > 0, np.abs(k - 0.5 * (b0 + b1)), np.inf))
        X[..., 6 + q] = math.log10(p[sel].mean() if sel.any() else p[near])
    X[..., 0] = (k / kny)[:, None]
    X[..., 1] = (np.arange(nmu) + 0.5) / nmu
    X[..., 2 + P.CIC] = 1.0
    X[..., 22] = np.log10(np.where(p > 0, p, 1.0))[:, None]
    share = _np(cells[0] * nmu / S.clamp_min(1e-300)[:, None])
    X[..., 23] = np.clip(np.log10(np.maximum(share, 1e-300)), -2.0, 2.0)
    X = X.reshape(-1, 32)
    f = 0.0
    nets = mlp.load_params().astype(np.float64)
    for net in nets:
        u = mlp.unpack(net)
        h = X
        for n in (1, 2, 3):
            h = np.maximum(h @ u[f"W{n}"] + u[f"b{n}"], 0.0)
        f = f + (h @ u["W4"] + u["b4"])[:, 0] / len(nets)
    f = np.where(np.repeat(p > 0, nmu), f, 0.0)
    raw = (cells * torch.from_numpy(np.exp(f)).cuda().view(nb, nmu)).sum(2)
    kk, e, km = _axis(N, L, kw, km)
    return {"k": kk, "kedge": e, "km": km, "lcnt": _np(lc),
            "pl": [_box_pl(raw, cnt, lc, kw["poles"], wsum), None]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "ascii":
        v = _ascii_ints(case["lines"], seed).to(torch.float64)
        v[:, :3] /= 1e6
        v[:, 3] /= 1e4
        return {"records": v, "n": None, "sumw": math.fsum(v[:, 3].tolist())}
    if kind == "cnvt":
        ra, dec, z = _sky(case["n"], _rng(seed))
        r = _distance(z)
        ra, dec = torch.deg2rad(ra), torch.deg2rad(dec)
        xyz = [r * torch.cos(dec) * torch.cos(ra), r * torch.cos(dec) * torch.sin(ra),
               r * torch.sin(dec), torch.ones_like(z)]
        return {"records": torch.stack(xyz, 1), "order": None}
    kw = dict(_conf_kw(case))
    if kind == "survey":
        return _survey_exact(case, kw, seed)
    if kind == "alias":
        return _alias_exact(case, kw, seed)
    N, L, zero = case["grid"], [SIDE] * 3, [0.0] * 3
    cnt, km, lc = _legsums(N, L, kw)
    k, e, km = _axis(N, L, kw, km)

    def pl(d):
        F = _field([(d, 1.0)], N, L, zero, kw["assign"], kw["intlace"])
        return _box_pl(_power(N, L, kw, F), cnt, lc, kw["poles"], float(d[:, 3].sum())), F

    if kind == "box":
        v = pl(_clustered(case["npart"], seed, case["order"], case["weights"]))[0]
        return {"k": k, "kedge": e, "km": km, "lcnt": _np(lc), "pl": [v, None]}
    if kind == "batch":
        v = np.stack([pl(d)[0] for d in _batch_inputs(case, seed)])
        rep = [np.repeat(a[None], len(v), 0) for a in (k, km, _np(lc))]
        return {"k": rep[0], "km": rep[1], "lcnt": rep[2], "pl": v}
    cats = [_clustered(n, 2 * seed + c) for c, n in enumerate((case["npart"], case["npart2"]))]
    (v0, F0), (v1, F1) = pl(cats[0]), pl(cats[1])
    w = math.sqrt(float(len(cats[0])) * float(len(cats[1])))
    x = _box_pl(_power(N, L, kw, F0, F1), cnt, lc, kw["poles"], w, shot=False)
    return {"k": k, "kedge": e, "km": km, "lcnt": _np(lc), "pl": [v0, v1], "xpl": x}
