"""Timed cases: the calls a user of this package makes, over the range of sizes
and options they are made with.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)`
one more of the same ranges.  `prepare(case, seed)` builds what the caller has
in hand before the call, `run(state)` makes one pass through the package's
entry points and returns its outputs, `work(case)` counts the bytes and
operations the pass cannot do without, and `exact(case, seed)` evaluates the
same outputs in 64 bits with plain torch.

Kinds of call:

* host_cape  - `core.calc_cape` on numpy arrays (the drop-in call);
* host_srh   - `core.calc_srh` on numpy arrays;
* cape       - `_hip.cape` on device tensors;
* srh        - `_hip.srh` on device tensors;
* combined   - `_hip.cape_srh` on device tensors (CAPE and helicity together);
* ragged     - a `RaggedPlan`'s replay (mixed level counts, sources, adiabats);
* train      - one training step of the warm start's surrogate.
"""
import math

import numpy as np
import torch

from xcape_amd import _hip, core, ragged, surrogate, synthetic

SOURCES = {1: 'surface', 2: 'most-unstable', 3: 'mixed-layer'}
ADIABATS = {1: 'pseudo-liquid', 2: 'reversible-liquid', 3: 'pseudo-ice', 4: 'reversible-ice'}
PINC = 500.0
ML_DEPTH = 500.0
DEPTH = 3000.0
P_TOP = 100.0        # [hPa] the uppermost level of the pressure grids


def listed():
    return [
        # one station's sounding, the smallest call there is: latency of one
        # column's ascent and of the host call around it
        dict(name='sounding_mu', kind='host_cape', grid='sigma', ncol=1, nk=60, source=2,
             adiabat=1),
        # a handful of reanalysis points with winds, float64 as read from files
        dict(name='points_17_srh', kind='host_srh', grid='pressure', ncol=17, nk=37, f64=True),
        # a small model domain from numpy, every default of calc_cape
        dict(name='domain_64x64x40_sb', kind='host_cape', grid='sigma', ncol=4096, nk=40,
             source=1, adiabat=1),
        # a regional domain of odd size, already on the device, warm start
        dict(name='regional_121x97x50_mu_warm', kind='cape', grid='sigma', ncol=121 * 97, nk=50,
             source=2, adiabat=3, warm=True, fast=False, levels=False),
        # the reanalysis grid on pressure levels, reference method
        dict(name='pressure_1024x512x37_sb', kind='cape', grid='pressure', ncol=1024 * 512, nk=37,
             source=1, adiabat=1, warm=False, fast=False, levels=False),
        # the same grid, mixed-layer parcels, warm start, with the LFC and EL
        dict(name='pressure_1024x512x37_ml_warm_lfc', kind='cape', grid='pressure',
             ncol=1024 * 512, nk=37, source=3, adiabat=1, warm=True, fast=False, levels=True),
        # a half-degree globe on model levels, reference method, fast math
        dict(name='globe_720x361x91_mu_ice_fast', kind='cape', grid='sigma', ncol=720 * 361,
             nk=91, source=2, adiabat=3, warm=False, fast=True, levels=False),
        # the headline workload: CAPE/CIN with the warm start, and the helicity
        dict(name='combined_2048x1024x137', kind='combined', grid='sigma', ncol=2048 * 1024,
             nk=137, source=2, adiabat=3, warm=True),
        # mixed soundings (30 to 137 levels, every source, two adiabats) kept
        # in a plan that is replayed
        dict(name='ragged_200k_warm', kind='ragged', ncol=200_000, warm=True),
        # the helicity chain alone
        dict(name='srh_1024x512x137', kind='srh', grid='sigma', ncol=1024 * 512, nk=137),
        # a large grid from numpy: the transfers with the ascent under them
        dict(name='host_360x181x137_mu_ice', kind='host_cape', grid='sigma', ncol=360 * 181,
             nk=137, source=2, adiabat=3),
        # one training step of the surrogate at its default batch
        dict(name='train_step_16384', kind='train', n=16384),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(('host_cape', 'host_srh', 'cape', 'cape', 'cape', 'combined', 'srh',
                       'ragged', 'train'))
    grid = rng.choice(('sigma', 'pressure'))
    nk = rng.choice((30, 40, 60, 91, 137, rng.randint(24, 137)))
    if grid == 'pressure':
        nk = rng.randint(20, 60)
    source, adiabat = rng.randint(1, 3), rng.choice((1, 1, 2, 3, 3, 4))
    if kind == 'host_cape':
        return dict(kind=kind, grid=grid, ncol=_log_int(rng, 1, 60_000), nk=nk, source=source,
                    adiabat=adiabat)
    if kind == 'host_srh':
        return dict(kind=kind, grid=grid, ncol=_log_int(rng, 1, 60_000), nk=nk,
                    f64=rng.random() < 0.5)
    if kind == 'cape':
        return dict(kind=kind, grid=grid, ncol=_log_int(rng, 100, 600_000), nk=nk, source=source,
                    adiabat=adiabat, warm=rng.random() < 0.5, fast=rng.random() < 0.2,
                    levels=rng.random() < 0.25)
    if kind == 'combined':
        return dict(kind=kind, grid=grid, ncol=_log_int(rng, 1000, 1_200_000), nk=nk,
                    source=source, adiabat=adiabat, warm=rng.random() < 0.7)
    if kind == 'srh':
        return dict(kind=kind, grid=grid, ncol=_log_int(rng, 100, 1_000_000), nk=nk)
    if kind == 'ragged':
        return dict(kind=kind, ncol=_log_int(rng, 500, 200_000), warm=rng.random() < 0.5)
    return dict(kind=kind, n=_log_int(rng, 1000, 70_000))


# ---------------------------------------------------------------------------
# inputs

def _tvirt(t, td, p):
    es = 611.2 * torch.exp(17.67 * (td - 273.15) / (td - 29.65))
    return t * (1.0 + 0.608 * 0.622 * es / torch.clamp(p - es, min=1.0))


def _columns(grid, ncol, nk, seed, winds):
    """Synthetic soundings as (ncol, nk) float32 tensors on the device, hPa and
    degC: surface pressure 950-1020 hPa, surface temperature 12-32 degC, a
    lapse rate of 5.5-8 K/km up to a tropopause at 11-15 km, hydrostatic
    heights; sheared winds with 1 m/s noise.  Sigma grids run from 0.995 to
    0.1 of the surface pressure; pressure grids share levels from 1000 to
    100 hPa, with NaN below the ground."""
    g = torch.Generator(device='cuda')
    g.manual_seed(seed)
    f64 = dict(dtype=torch.float64, device='cuda')

    def uniform(lo, hi):
        return lo + (hi - lo) * torch.rand(ncol, generator=g, **f64)
    ps, ts = uniform(95000.0, 102000.0), uniform(285.0, 305.0)
    lapse, ztrop = uniform(5.5e-3, 8.0e-3), uniform(11000.0, 15000.0)
    d0, gd = uniform(1.0, 15.0), uniform(1.0e-3, 4.0e-3)
    if grid == 'sigma':
        sig = torch.linspace(0.995, 0.1, nk, **f64).tolist()
    else:
        lev = torch.linspace(100000.0, 100.0 * P_TOP, nk, **f64)
        # a level is below the ground by the float32 values the caller holds
        ps32, lev32 = (ps / 100.0).float(), (lev / 100.0).float()
    # float32 level-major buffers, handed over column-contiguous
    names = ('p', 't', 'td') if grid == 'sigma' else ('t', 'td')
    out = {k: torch.empty((nk, ncol), dtype=torch.float32, device='cuda') for k in names}
    zs = torch.empty((nk, ncol), **f64) if winds else None
    z, p_prev = torch.zeros(ncol, **f64), ps
    tv_prev = _tvirt(ts, ts - d0, ps)
    for k in range(nk):
        pk = ps * sig[k] if grid == 'sigma' else torch.minimum(lev[k], ps)
        lnr = torch.log(p_prev / pk) * (synthetic.RD / synthetic.G)
        zk = z + tv_prev * lnr
        for _ in range(3):
            tk = ts - lapse * torch.minimum(zk, ztrop)
            tv = _tvirt(tk, tk - (d0 + gd * zk), pk)
            zk = z + 0.5 * (tv_prev + tv) * lnr
        tk = ts - lapse * torch.minimum(zk, ztrop)
        tdk = tk - (d0 + gd * zk)
        tv_prev, z, p_prev = _tvirt(tk, tdk, pk), zk, pk
        below = None if grid == 'sigma' else lev32[k] > ps32
        for name, a in (('p', pk / 100.0), ('t', tk - 273.15), ('td', tdk - 273.15)):
            if name in out:
                out[name][k] = a if below is None else torch.where(below, float('nan'), a)
        if winds:
            zs[k] = zk
    if winds:
        u0, s, th = uniform(-5.0, 10.0), uniform(0.0, 0.01), uniform(0.0, 2.0 * math.pi)

        def shear(h):
            return s * torch.clamp(h, max=6000.0) + 0.5 * s * torch.clamp(h - 6000.0, min=0.0)
        for name, base, f in (('u', u0, torch.cos(th)), ('v', 0.0 * u0, torch.sin(th))):
            a = torch.empty((nk, ncol), dtype=torch.float32, device='cuda')
            for k in range(nk):
                noise = torch.randn(ncol, generator=g, **f64)
                a[k] = base + shear(zs[k]) * f + noise
                if grid == 'pressure':
                    a[k] = torch.where(lev32[k] > ps32, float('nan'), a[k])
            out[name] = a
            out[name + 's'] = (base + s * 2.0 * f).float()
    out = {k: (a.t().contiguous() if a.ndim == 2 else a) for k, a in out.items()}
    if grid == 'pressure':
        out['p'] = lev32
    out.update(ps=(ps / 100.0).float(), ts=(ts - 273.15).float(), tds=(ts - d0 - 273.15).float())
    return out


SFC = ('ps', 'ts', 'tds')
WIND_ARGS = ('p', 't', 'td', 'u', 'v', 'ps', 'ts', 'tds', 'us', 'vs')
CAPE_ARGS = ('p', 't', 'td') + SFC


def _inputs(case, seed):
    winds = case['kind'] in ('host_srh', 'srh', 'combined')
    return _columns(case['grid'], case['ncol'], case['nk'], seed, winds)


def _train_inputs(case, seed):
    """Normalised network inputs with a smooth target, and an optimiser in the
    middle of a run (its moments already built up)."""
    g = torch.Generator(device='cuda')
    g.manual_seed(seed)
    n = case['n']
    u = torch.randn((n, 3), generator=g, device='cuda')
    t = torch.tanh(u[:, 0] - 0.5 * u[:, 1] * u[:, 2]) + 0.3 * u[:, 2] \
        + 0.05 * torch.randn(n, generator=g, device='cuda')
    theta = torch.as_tensor(surrogate.init_params(seed % 1000), device='cuda')
    m = 1e-3 * torch.randn(theta.shape, generator=g, device='cuda')
    v = 1e-6 + 1e-5 * torch.rand(theta.shape, generator=g, device='cuda')
    return dict(u=u, t=t.contiguous(), theta=theta, m=m, v=v)


ADAM = dict(step=500, lr=1e-3, b1=0.9, b2=0.999, eps=1e-8, wd=0.0)


def _load_surrogate():
    # a program that uses the warm start loads the packaged network once
    if not _hip.lib().xcape_surrogate_loaded():
        surrogate.Surrogate.load().activate()


def prepare(case, seed):
    kind = case['kind']
    if kind == 'train':
        return dict(case=case, **_train_inputs(case, seed))
    if case.get('warm'):
        _load_surrogate()
    if kind == 'ragged':
        batch = ragged.RaggedBatch.from_dict(synthetic.ragged_columns(case['ncol'], seed))
        cfg = dict(ragged.DEFAULT, cols=64) if case['warm'] else dict(ragged.DEFAULT)
        return dict(case=case, batch=batch,
                    plan=ragged.RaggedPlan(batch, PINC, ML_DEPTH, warm_start=case['warm'], **cfg))
    c = _inputs(case, seed)
    if kind in ('host_cape', 'host_srh'):
        dt = np.float64 if case.get('f64') else np.float32
        c = {k: np.ascontiguousarray(a.cpu().numpy().astype(dt)) for k, a in c.items()}
    return dict(case=case, **c)


# ---------------------------------------------------------------------------
# one pass

def run(s):
    case = s['case']
    kind = case['kind']
    if kind == 'host_cape':
        return core.calc_cape(*(s[k] for k in CAPE_ARGS), source=SOURCES[case['source']],
                              ml_depth=ML_DEPTH, adiabat=ADIABATS[case['adiabat']], pinc=PINC,
                              vertical_lev=case['grid'])
    if kind == 'host_srh':
        return core.calc_srh(*(s[k] for k in WIND_ARGS), depth=DEPTH, vertical_lev=case['grid'],
                             output_var='all')
    if kind == 'cape':
        return _hip.cape(*(s[k] for k in CAPE_ARGS), pinc=PINC, source=case['source'],
                         ml_depth=ML_DEPTH, adiabat=case['adiabat'],
                         p_shared=case['grid'] == 'pressure', fast_math=case['fast'],
                         warm_start=case['warm'], levels=case['levels'])
    if kind == 'srh':
        return _hip.srh(*(s[k] for k in WIND_ARGS), depth=DEPTH,
                        p_shared=case['grid'] == 'pressure')
    if kind == 'combined':
        return _hip.cape_srh(*(s[k] for k in WIND_ARGS), pinc=PINC, source=case['source'],
                             ml_depth=ML_DEPTH, adiabat=case['adiabat'], depth=DEPTH,
                             p_shared=case['grid'] == 'pressure', warm_start=case['warm'])
    if kind == 'ragged':
        s['plan'].run()
        b = s['batch']
        return b.cape, b.cin, b.mulev, b.zmulev
    loss, grad = surrogate.loss_grad(s['theta'], s['u'], s['t'])
    P = _hip._ptr
    _hip.check(_hip.lib().xcape_mlp_adam(
        P(s['theta']), P(grad), P(s['m']), P(s['v']), ADAM['step'], ADAM['lr'], ADAM['b1'],
        ADAM['b2'], ADAM['eps'], ADAM['wd'], surrogate._stream()))
    return dict(loss=loss, grad=grad, theta=s['theta'], m=s['m'], v=s['v'])


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _substeps(case, nk):
    """Sub-steps of a column's ascent over nk levels: every layer takes one
    more than it holds whole pinc steps."""
    if case['grid'] == 'sigma':
        dp = 98500.0 * 0.895 / max(nk - 1, 1)
    else:
        dp = 100.0 * (1000.0 - P_TOP) / max(nk - 1, 1)
    return nk * (1 + int(dp / PINC))


def _ascent_ops(nk, sub, source, adiabat):
    """Operations of one column: the environment, the theta-e scan below
    500 hPa, buoyancy and trapezoids per level, set-up and one evaluation of
    the moist-adiabat map per sub-step."""
    ice = adiabat >= 3
    return 26 * (nk + 1) + (26 * nk * 0.55 if source == 2 else 0) + 35 * nk \
        + sub * (6 + (74 if ice else 69))


def work(case):
    kind = case['kind']
    if kind == 'train':
        n, h, npar = case['n'], 64, surrogate.nparams()
        return dict(bytes=4 * (4 * n + 7 * npar + 1), flops=n * (3 * 2 * h * (h + 3 + 1) + 30 * h))
    if kind == 'ragged':
        n = case['ncol']
        b = f = 0.0
        for nk in synthetic.RAGGED_NLEVS:
            c = dict(grid='sigma')
            b += n / 5 * (4 * (3 * nk + 3) + 16 + 8)
            for source in (1, 2, 3):
                for adiabat in (1, 3):
                    f += n / 30 * _ascent_ops(nk, _substeps(c, nk), source, adiabat)
        return dict(bytes=b, flops=f)
    n, nk = case['ncol'], case['nk']
    esz = 8 if case.get('f64') else 4
    narr = 2 + (case['grid'] == 'sigma')
    b = f = 0.0
    if kind in ('host_cape', 'cape', 'combined'):
        b += 16 + (8 if case.get('levels') else 0)
        f += _ascent_ops(nk, _substeps(case, nk), case['source'], case['adiabat'])
    if kind in ('host_srh', 'srh', 'combined'):
        # two logarithms, an exponential and five divisions per level up to 6 km
        narr += 2
        b += 2 * esz + 16 + 24
        f += 0.53 * nk * 120
    return dict(bytes=n * (b + esz * (narr * nk + 3)), flops=n * f)


# ---------------------------------------------------------------------------
# the same outputs in 64 bits: Bryan's getcape, the hypsometric heights,
# Bunkers motion and storm-relative helicity over whole batches, level by level

G, CP, RD, RV = 9.81, 1005.7, 287.04, 461.5
XLV, XLS, T0, CPV, CPL, CPI = 2501000.0, 2836017.0, 273.15, 1875.0, 4190.0, 2118.636


def _qv(a, b, p, t):
    es = 611.2 * torch.exp(a * (t - 273.15) / (t - b))
    return RD / RV * es / (p - es)


def _qvs(p, t):
    return _qv(17.67, 29.65, p, t)


def _thetae(p, t, td, q):
    tl = 56.0 + 1.0 / (1.0 / (td - 56.0) + 0.00125 * torch.log(t / td))
    tl = torch.where(td - t >= -0.1, t, tl)
    return t * (100000.0 / p) ** (0.2854 * (1.0 - 0.28 * q)) \
        * torch.exp((3376.0 / tl - 2.54) * q * (1.0 + 0.81 * q))


def _map(x, p2, pi2, logp, t1, th1, qv1, ql1, qi1, qt, ice):
    """The moist-adiabat map at iterate x: its image and the parcel state."""
    t2 = x * pi2
    fliq = torch.where(ice, torch.clamp((t2 - 233.15) / 40.0, 0.0, 1.0), 1.0)
    fice = 1.0 - fliq
    qv2 = torch.minimum(qt, fliq * _qvs(p2, t2) + fice * _qv(21.8745584, 7.66, p2, t2))
    qi2 = torch.clamp(fice * (qt - qv2), min=0.0)
    ql2 = torch.clamp(qt - qv2 - qi2, min=0.0)
    tb, qvb, qlb, qib = 0.5 * (t1 + t2), 0.5 * (qv1 + qv2), 0.5 * (ql1 + ql2), 0.5 * (qi1 + qi2)
    lhv = XLV + (CPL - CPV) * T0 - (CPL - CPV) * tb
    lhs = XLS + (CPI - CPV) * T0 - (CPI - CPV) * tb
    cpm = CP + CPV * qvb + CPL * qlb + CPI * qib
    th2 = th1 * torch.exp((lhv * (ql2 - ql1) + lhs * (qi2 - qi1)) / (cpm * tb)
                          + ((RD + RV * qvb) / cpm - RD / CP) * logp)
    return th2, t2, qv2, ql2, qi2


def _getcape64(p, t, td, nk, source, adiabat, levels):
    """p, t, td: (K, n) float64 in Pa and K, row 0 the surface; nk, source and
    adiabat per column.  Entries at rows >= nk are never used."""
    K, n = p.shape
    dev = p.device
    col = torch.arange(n, device=dev)
    pi = (p / 100000.0) ** (RD / CP)
    q = _qvs(p, td)
    th = t / pi
    thv = th * (1.0 + RV / RD * q) / (1.0 + q)
    dz = torch.zeros_like(p)
    dz[1:] = -CP / G * 0.5 * (thv[1:] + thv[:-1]) * (pi[1:] - pi[:-1])
    z = torch.cumsum(dz, 0)
    zero = torch.zeros(n, dtype=torch.float64, device=dev)
    kmax = torch.zeros(n, dtype=torch.int64, device=dev)
    best = zero.clone()
    mu = (source == 2) & (p[0] >= 50000.0)
    for k in range(K):
        use = mu & (k < nk) & (p[k] >= 50000.0)
        the = _thetae(p[k], t[k], td[k], q[k])
        use &= the > best
        best, kmax = torch.where(use, the, best), torch.where(use, k, kmax)
    # mixed layer: trapezoid means of theta and q up to ML_DEPTH
    mix = source == 3
    ath, aqv = zero.clone(), zero.clone()
    open_ = mix & (z[min(1, K - 1)] <= ML_DEPTH)
    ath, aqv = torch.where(mix & ~open_, th[0], ath), torch.where(mix & ~open_, q[0], aqv)
    for k in range(1, K):
        here = open_ & (k < nk)
        top = here & (z[k] > ML_DEPTH)
        h = torch.where(top, ML_DEPTH, z[k]) - z[k - 1]
        w = (ML_DEPTH - z[k - 1]) / (z[k] - z[k - 1])
        thk = torch.where(top, th[k - 1] + (th[k] - th[k - 1]) * w, th[k])
        qk = torch.where(top, q[k - 1] + (q[k] - q[k - 1]) * w, q[k])
        ath = torch.where(here, ath + 0.5 * h * (thk + th[k - 1]), ath)
        aqv = torch.where(here, aqv + 0.5 * h * (qk + q[k - 1]), aqv)
        ath, aqv = torch.where(top, ath / ML_DEPTH, ath), torch.where(top, aqv / ML_DEPTH, aqv)
        open_ = open_ & ~top

    def at(a):
        return a[kmax, col]
    th2, qv2, pi2, p2 = at(th), at(q), at(pi), at(p)
    thv0 = at(thv)
    th2, qv2 = torch.where(mix, ath, th2), torch.where(mix, aqv, qv2)
    t2 = torch.where(mix, th2 * pi2, at(t))
    b2 = torch.where(mix, G * (th2 * (1.0 + RV / RD * qv2) / (1.0 + qv2) - thv0) / thv0, 0.0)
    ql2, qi2, qt = zero.clone(), zero.clone(), qv2
    cape, cin, narea = zero.clone(), zero.clone(), zero.clone()
    nan = torch.full_like(zero, float('nan'))
    zout, lfc, el = torch.full_like(zero, -999999.0), nan.clone(), nan.clone()
    ice, pseudo = adiabat >= 3, (adiabat == 1) | (adiabat == 3)
    alive = torch.ones(n, dtype=torch.bool, device=dev)
    for k in range(1, K):
        on = alive & (k > kmax) & (k < nk)
        if not bool(on.any()):
            continue
        dp = p[k - 1] - p[k]
        nloop = torch.where(dp < PINC, 1.0, 1.0 + torch.floor(dp / PINC))
        dp = dp / nloop
        for j in range(int(nloop[on].max())):
            step = on & (j < nloop)
            p2n = p2 - dp
            pi2n = (p2n / 100000.0) ** (RD / CP)
            logp = torch.log(p2n / p2)
            x, left = th2, step
            got = (th2, t2, qv2, ql2, qi2)
            for it in range(101):
                new = _map(x, p2n, pi2n, logp, t2, th2, qv2, ql2, qi2, qt, ice)
                got = tuple(torch.where(left, a, b) for a, b in zip(new, got))
                left = left & ((new[0] - x).abs() > 2e-4)
                if not bool(left.any()):
                    break
                x = torch.where(left, x + 0.3 * (new[0] - x), x)
            alive, on, step = alive & ~left, on & ~left, step & ~left
            cape, cin = torch.where(left, 0.0, cape), torch.where(left, 0.0, cin)
            th2, t2, qv2, ql2, qi2 = got
            p2 = torch.where(step, p2n, p2)
            drop = step & pseudo
            qt = torch.where(drop, qv2, qt)
            ql2, qi2 = torch.where(drop, 0.0, ql2), torch.where(drop, 0.0, qi2)
        b1 = b2
        thv2 = th2 * (1.0 + RV / RD * qv2) / (1.0 + qv2 + ql2 + qi2)
        b2 = torch.where(on, G * (thv2 - thv[k]) / thv[k], b1)
        d = dz[k]
        enter, leave = on & (b2 >= 0.0) & (b1 < 0.0), on & (b2 < 0.0) & (b1 > 0.0)
        neg, pos = on & (b2 < 0.0) & ~leave, on & (b2 >= 0.0) & ~enter
        frac = torch.where(enter, b2, b1) / torch.where(enter, b2 - b1, b1 - b2)
        area = torch.where(enter, 0.5 * b2 * d * frac, zero)
        area = torch.where(leave, 0.5 * b1 * d * frac, area)
        area = torch.where(pos, 0.5 * d * (b1 + b2), area)
        cin = torch.where(enter, cin + narea - 0.5 * b1 * d * (1.0 - frac), cin)
        narea = torch.where(enter | pos, 0.0, torch.where(
            leave, -0.5 * b2 * d * (1.0 - frac),
            torch.where(neg, narea - 0.5 * d * (b1 + b2), narea)))
        cape = cape + torch.clamp(area, min=0.0)
        if levels:
            add = on & (area > 0.0)
            pc = p[k - 1] + (p[k] - p[k - 1]) * (0.0 - b1) / (b2 - b1)
            lfc = torch.where(add & torch.isnan(lfc), torch.where(enter, pc, p[k - 1]), lfc)
            el = torch.where(add, torch.where(leave, pc, p[k]), el)
        zout = torch.where(on, z[k], zout)
        alive = alive & ~(on & (p[k] <= 10000.0) & (b2 < 0.0))
    out = [cape, cin, None, zout]
    return out + [lfc / 100.0, el / 100.0] if levels else out


def _full_columns(c, names):
    """The arrays of `names` ('p' first) as (K, n) float64 rows, the surface
    row first, each column from its first level above the ground; and the
    columns' level counts."""
    d = {k: torch.as_tensor(a, device='cuda').double() for k, a in c.items()}
    n, nk = d['t'].shape
    if d['p'].ndim == 1:
        above = d['p'][None, :] <= d['ps'][:, None]
        first = above.int().argmax(1)
        idx = torch.clamp(torch.arange(nk, device='cuda')[:, None] + first[None, :], max=nk - 1)
        rows = {k: d[k].t().gather(0, idx) for k in names if k != 'p'}
        rows['p'] = d['p'][idx]
        count = nk - first + 1
    else:
        rows = {k: d[k].t() for k in names}
        count = torch.full((n,), nk + 1, device='cuda')
    return [torch.cat((d[k + 's'][None], rows[k])) for k in names], count


def _srh64(c, depth):
    (p, t, td, u, v), nk = _full_columns(c, ('p', 't', 'td', 'u', 'v'))

    def lit(x):           # the reference's single-precision literals
        return float(np.float32(x))
    eps = lit(0.6219800858985514)
    t, td = t + lit(273.15), td + lit(273.15)
    e = lit(6.112) * torch.exp(lit(53.49) - 6808.0 / td - lit(5.09) * torch.log(td))
    w = eps * e / (p - e)
    tv = t * (w + eps) / (eps * (1.0 + w))
    K, n = p.shape
    H = torch.full_like(p, 2.0)
    for k in range(1, K):
        H[k] = H[k - 1] + lit(287.04) * 0.5 * (tv[k] + tv[k - 1]) / lit(-9.80665) \
            * torch.log(p[k] / p[k - 1])
    wind = []
    for a in (u, v):
        got = []
        for i in range(12):
            h = 500.0 * (i + 1)
            x = torch.full((n,), -999999.0, dtype=torch.float64, device=p.device)
            for k in range(1, K):
                f = (h - H[k - 1]) / (H[k] - H[k - 1])
                x = torch.where((k < nk) & (H[k - 1] <= h) & (H[k] > h),
                                (1.0 - f) * a[k - 1] + f * a[k], x)
            got.append(x)
        wind.append((a[0], got))
    (u0, iu), (v0, iv) = wind
    mu, mv = (u0 + sum(iu)) / 13.0, (v0 + sum(iv)) / 13.0
    su = (iu[10] + iu[11]) / 2.0 - (u0 + iu[0]) / 2.0
    sv = (iv[10] + iv[11]) / 2.0 - (v0 + iv[0]) / 2.0
    mag = torch.sqrt(su * su + sv * sv)
    rm, lm = (mu + 7.5 * sv / mag, mv - 7.5 * su / mag), (mu - 7.5 * sv / mag, mv + 7.5 * su / mag)
    srh = []
    for cu, cv in (rm, lm):
        s, done = torch.zeros_like(mu), torch.zeros(n, dtype=torch.bool, device=p.device)
        ub, vb = u[0], v[0]
        for k in range(1, K):
            use = ~done & (k < nk)
            top = use & (H[k] > depth)
            f = (depth - H[k]) / (H[k - 1] - H[k])
            uk = torch.where(top, u[k] + (u[k - 1] - u[k]) * f, u[k])
            vk = torch.where(top, v[k] + (v[k - 1] - v[k]) * f, v[k])
            s = torch.where(use, s + (uk - cu) * (vk - vb) - (vk - cv) * (uk - ub), s)
            ub, vb, done = torch.where(use, uk, ub), torch.where(use, vk, vb), done | top
        srh.append(torch.where(done, -s, 0.0))
    return srh, rm, lm, (mu, mv)


def _bf16(a):
    return a.float().bfloat16().double()


def _train64(case, seed):
    """The step in 64 bits, with the network's BF16 weights and first hidden
    activations rounded as the network defines them."""
    s = {k: a.double() for k, a in _train_inputs(case, seed).items()}
    h = 64
    theta, x, n = s['theta'], s['u'], case['n']
    w1, b1, w2, b2, w3, b3 = torch.split(theta, [3 * h, h, h * h, h, h, 1])
    w1, w2, w3 = _bf16(w1).view(h, 3), _bf16(w2).view(h, h), _bf16(w3)
    c, a = math.sqrt(2.0 / math.pi), 0.044715

    def gelu(z):
        return 0.5 * z * (1.0 + torch.tanh(c * (z + a * z ** 3)))

    def slope(z):
        r = torch.tanh(c * (z + a * z ** 3))
        return 0.5 * (1.0 + r) + 0.5 * z * (1.0 - r * r) * c * (1.0 + 3.0 * a * z * z)
    z1 = x @ w1.t() + b1
    h1 = _bf16(gelu(z1))
    z2 = h1 @ w2.t() + b2
    h2 = gelu(z2)
    r = h2 @ w3 + b3 - s['t']
    dy = 2.0 * r / n
    d2 = dy[:, None] * w3 * slope(z2)
    d1 = (d2 @ w2) * slope(z1)
    grad = torch.cat(((d1.t() @ x).flatten(), d1.sum(0), (d2.t() @ h1).flatten(), d2.sum(0),
                      h2.t() @ dy, dy.sum()[None]))
    k = ADAM
    m = k['b1'] * s['m'] + (1.0 - k['b1']) * grad
    v = k['b2'] * s['v'] + (1.0 - k['b2']) * grad * grad
    step = (m / (1.0 - k['b1'] ** k['step'])) \
        / (torch.sqrt(v / (1.0 - k['b2'] ** k['step'])) + k['eps'])
    return dict(loss=(r * r).mean()[None], grad=grad, theta=theta - k['lr'] * step, m=m, v=v)


def _ragged64(case, seed):
    b = synthetic.ragged_columns(case['ncol'], seed)
    dev = dict(device='cuda')
    nlev = torch.as_tensor(b['nlev'], **dev).long()
    off = torch.as_tensor(b['offsets'], **dev)[:-1]
    row = torch.arange(int(nlev.max()), **dev)[:, None]
    idx = off[None, :] + torch.minimum(row, nlev[None, :] - 1)
    full = []
    for k in ('p', 't', 'td'):
        a = torch.as_tensor(b[k], **dev).double()
        full.append(torch.cat((torch.as_tensor(b[k + 's'], **dev).double()[None], a[idx])))
    return _getcape64(100.0 * full[0], 273.15 + full[1], 273.15 + full[2], nlev + 1,
                      torch.as_tensor(b['source'], **dev), torch.as_tensor(b['adiabat'], **dev),
                      False)


def exact(case, seed):
    kind = case['kind']
    if kind == 'train':
        return _train64(case, seed)
    if kind == 'ragged':
        return _ragged64(case, seed)
    c = _inputs(case, seed)
    out = []
    if kind in ('host_cape', 'cape', 'combined'):
        (p, t, td), nk = _full_columns(c, ('p', 't', 'td'))
        n = p.shape[1]
        src = torch.full((n,), case['source'], device='cuda')
        adi = torch.full((n,), case['adiabat'], device='cuda')
        out = _getcape64(100.0 * p, 273.15 + t, 273.15 + td, nk, src, adi,
                         bool(case.get('levels')))
        del p, t, td
        if kind == 'host_cape' and case['source'] != 2:
            out = out[:2]
    if kind in ('host_srh', 'srh', 'combined'):
        srh, rm, lm, mean = _srh64(c, DEPTH)
        if kind == 'host_srh':
            out = [*srh, *rm, *lm, *mean]
        else:
            out += [*srh] + [torch.stack(x, 1) for x in (rm, lm, mean)]
    return out
