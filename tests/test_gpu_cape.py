"""GPU parity of the CAPE/CIN kernels against the oracle and the reference's
goldens.  Calls go through the C-ABI (xcape_amd._hip -> libxcape_hip.so)."""
import numpy as np
import pytest

from tests.tolerances import cape_ok, cape_tol, ill_conditioned_and_matched
from xcape_amd import synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def hip():
    from xcape_amd import _hip
    assert _hip.device_count() >= 1, 'no HIP device visible'
    return _hip


def _report(name, got, ref):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    d = np.abs(got - ref)
    bad = ~cape_ok(got, ref)
    print(f'{name}: max|d|={d.max():.4g} exact={np.mean(got == ref):.3f} '
          f'outside_tol={bad.sum()}/{bad.size}', flush=True)
    return bad


def _mu_tie(o, p, t, td, ps, ts, tds, lv_a, lv_b):
    """True when the theta-e of two candidate MU levels agree to 4 ulp."""
    pa = np.concatenate([[ps], p])
    ta = np.concatenate([[ts], t])
    tda = np.concatenate([[tds], td])

    def the(k):
        pk, tk, tdk = pa[k - 1] * 100.0, ta[k - 1] + 273.15, tda[k - 1] + 273.15
        pk, tk, tdk = np.float32(pk), np.float32(tk), np.float32(tdk)
        q = o.lib().xo_getqvs_f32
        import ctypes
        q.restype = ctypes.c_float
        q.argtypes = [ctypes.c_float, ctypes.c_float]
        qq = q(pk, tdk)
        f = o.lib().xo_getthe_f32
        f.restype = ctypes.c_float
        f.argtypes = [ctypes.c_float] * 4
        return f(pk, tk, tdk, qq)
    a, b = the(lv_a), the(lv_b)
    return abs(a - b) <= 4 * np.spacing(np.float32(max(a, b)))


def test_soundings_goldens(hip, soundings, oracle_lib):
    """Reference test_calc_cape_sigma (test/test_core.py:68-116): 13 soundings,
    SB pinc 100, ML 500 m pinc 1000, MU pinc 100; |d| < 1.5 like the
    reference's decimal=0, plus the 0.5 J/kg / 0.1 % bar against the oracle."""
    s = soundings
    P, T, TD = s['pressure'], s['temperature'], s['dewpoint']
    args = (P[:, 1:], T[:, 1:], TD[:, 1:], P[:, 0], T[:, 0], TD[:, 0])
    cases = [(1, 100., 'SB_CAPE_pinc100', 'SB_CIN_pinc100'),
             (3, 1000., 'ML_CAPE_pinc1000_mldepth500', 'ML_CIN_pinc1000_mldepth500'),
             (2, 100., 'MU_CAPE_pinc100', 'MU_CIN_pinc100')]
    for src, pinc, kc, ki in cases:
        c, ci, mu, z = hip.cape(*args, pinc=pinc, source=src, ml_depth=500., adiabat=1)
        oc, oci, omu, oz = oracle_lib.cape(*args, pinc=pinc, source=src, ml_depth=500.,
                                           adiabat=1)
        assert np.all(np.abs(c - s[kc]) < 1.5), (kc, c, s[kc])
        assert np.all(np.abs(ci - s[ki]) < 1.5), (ki, ci, s[ki])
        assert not _report(f'snd src{src} cape', c, oc).any()
        assert not _report(f'snd src{src} cin', ci, oci).any()
        if src == 2:
            assert np.array_equal(mu, s['MU_lv_pinc100'].astype(np.int32))
            assert np.all(np.abs(z - s['MU_z_pinc100']) < 1.5)
            np.testing.assert_array_equal(mu, omu)


def test_era5_goldens(hip, era5, oracle_lib):
    """Reference test_calc_cape_pressure (test/test_core.py:120-170):
    17 ERA5 columns, SB / ML 300 m / MU at pinc 500."""
    e = era5
    lev = e['level']
    st = oracle_lib.start_levels(lev, e['sfc_p'])
    for src, key in ((1, 'sp500'), (3, 'ml300p500'), (2, 'mup500')):
        for start in (st, None):     # host-computed and device-computed start levels
            c, ci, mu, z = hip.cape(lev, e['t'], e['td'], e['sfc_p'], e['sfc_t'], e['sfc_td'],
                                    pinc=500., source=src, ml_depth=300., adiabat=1,
                                    p_shared=True, start_lev=start)
            assert np.all(np.abs(c - e['sfc_cape' + key]) < 1.5)
            assert np.all(np.abs(ci - e['sfc_cin' + key]) < 1.5)
            oc, oci, _, _ = oracle_lib.cape(None, e['t'], e['td'], e['sfc_p'], e['sfc_t'],
                                            e['sfc_td'], 500., src, 300., 1, p1d=lev,
                                            start_lev=st)
            assert not _report(f'era5 src{src} cape', c, oc).any()
            assert not _report(f'era5 src{src} cin', ci, oci).any()


@pytest.mark.parametrize('adiabat', [1, 2, 3, 4])
@pytest.mark.parametrize('source', [1, 2, 3])
def test_sigma_synthetic(hip, oracle_lib, source, adiabat):
    """64x64 sigma columns (40 levels) from the seeded generator, every
    source and adiabat, against the FP32 oracle."""
    c = synthetic.sigma_columns(4096, 40, 1000)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    g = hip.cape(*args, pinc=500., source=source, ml_depth=500., adiabat=adiabat, stats=True)
    o = oracle_lib.cape(*args, pinc=500., source=source, ml_depth=500., adiabat=adiabat,
                        stats=True)
    print('gpu stats', g[4], 'oracle stats', o[4])
    bad_c = _report(f'sigma s{source} a{adiabat} cape', g[0], o[0])
    bad_i = _report(f'sigma s{source} a{adiabat} cin', g[1], o[1])
    assert not bad_c.any() and not bad_i.any()
    mism = np.nonzero(g[2] != o[2])[0]
    for i in mism:
        assert _mu_tie(oracle_lib, c['p'][i], c['t'][i], c['td'][i], c['ps'][i], c['ts'][i],
                       c['tds'][i], g[2][i], o[2][i]), (i, g[2][i], o[2][i])
    assert g[4]['columns'] == o[4]['columns']


@pytest.mark.parametrize('adiabat', [1, 3])
@pytest.mark.parametrize('source', [1, 2, 3])
@pytest.mark.parametrize('warm', [False, 'extrapolation'])
def test_pressure_synthetic(hip, oracle_lib, source, adiabat, warm):
    """37 fixed pressure levels with NaN below ground, device start levels
    (columns of different level counts), plain and warm-started."""
    c = synthetic.pressure_columns(4096, 1001)
    st = oracle_lib.start_levels(c['p'], c['ps'])
    g = hip.cape(c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'], pinc=500.,
                 source=source, ml_depth=500., adiabat=adiabat, p_shared=True,
                 warm_start=warm)
    o = oracle_lib.cape(None, c['t'], c['td'], c['ps'], c['ts'], c['tds'], 500., source, 500.,
                        adiabat, p1d=c['p'], start_lev=st)
    assert np.all(np.isfinite(g[0])) and np.all(np.isfinite(g[1]))
    assert not _report(f'pres s{source} a{adiabat} {warm} cape', g[0], o[0]).any()
    assert not _report(f'pres s{source} a{adiabat} {warm} cin', g[1], o[1]).any()


def test_fp64_matches_fp64_oracle(hip, oracle_lib):
    c = synthetic.sigma_columns(2048, 40, 1000)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    for src in (1, 2, 3):
        g = hip.cape(*args, pinc=500., source=src, adiabat=3, fp64=True)
        o = oracle_lib.cape(*[a.astype(np.float64) for a in args], pinc=500., source=src,
                            adiabat=3, fp64=True)
        d = np.abs(g[0] - o[0])
        print('fp64 max|d|', d.max(), flush=True)
        assert np.all(d <= 1e-6 * np.maximum(1.0, np.abs(o[0])))
        assert np.all(np.abs(g[1] - o[1]) <= 1e-6 * np.maximum(1.0, np.abs(o[1])))


def test_fast_math_within_tolerance(hip, oracle_lib):
    c = synthetic.sigma_columns(4096, 40, 1000)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    for src, adi in ((1, 1), (2, 3), (3, 1)):
        g = hip.cape(*args, pinc=500., source=src, adiabat=adi, fast_math=True)
        o = oracle_lib.cape(*args, pinc=500., source=src, adiabat=adi)
        bad = _report(f'fast s{src} a{adi} cape', g[0], o[0])
        bad |= _report(f'fast s{src} a{adi} cin', g[1], o[1])
        assert not bad.any()


def test_cold_surface_gate(hip):
    """ts <= 0 degC columns return zeros (CAPE_CODE_model_lev.f90:77,83-88)."""
    c = synthetic.sigma_columns(256, 40, 7)
    ts = c['ts'].copy()
    ts[::3] = -1.0
    ts[1] = 0.0
    g = hip.cape(c['p'], c['t'], c['td'], c['ps'], ts, c['tds'], source=2)
    gated = ~(ts > 0)
    assert np.all(g[0][gated] == 0) and np.all(g[1][gated] == 0)
    assert np.all(g[2][gated] == 0) and np.all(g[3][gated] == 0)


def test_device_pointer_path(hip):
    import torch
    c = synthetic.sigma_columns(1024, 40, 11)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    h = hip.cape(*args, source=1)
    dargs = [torch.from_numpy(a).cuda() for a in args]
    d = hip.cape(*dargs, source=1)
    torch.cuda.synchronize()
    for x, y in zip(h, d):
        np.testing.assert_array_equal(x, y.cpu().numpy())


@pytest.mark.parametrize('warm', [False, True])
def test_level_major_input_matches_column_contiguous(hip, warm):
    """(nk, ncol) profiles with XCAPE_LEVEL_MAJOR give the same results as
    the column-contiguous ones (which the library stages level-major), on a
    sigma and on a pressure grid, CAPE and helicity."""
    c = synthetic.sigma_columns(3000, 60, 17, winds=True)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    lm = (c['p'].T.copy(), c['t'].T.copy(), c['td'].T.copy(), c['ps'], c['ts'], c['tds'])
    kw = dict(pinc=500., source=2, adiabat=3, warm_start=warm)
    for x, y in zip(hip.cape(*args, **kw), hip.cape(*lm, level_major=True, **kw)):
        np.testing.assert_array_equal(x, y)
    sa = (c['p'], c['t'], c['td'], c['u'], c['v'], c['ps'], c['ts'], c['tds'], c['us'], c['vs'])
    sl = (c['p'].T.copy(), c['t'].T.copy(), c['td'].T.copy(), c['u'].T.copy(), c['v'].T.copy(),
          c['ps'], c['ts'], c['tds'], c['us'], c['vs'])
    for x, y in zip(hip.srh(*sa), hip.srh(*sl, level_major=True)):
        np.testing.assert_array_equal(x, y)
    pc = synthetic.pressure_columns(2000, 18)
    pa = (np.asarray(pc['p'], np.float32), pc['t'], pc['td'], pc['ps'], pc['ts'], pc['tds'])
    pl = (pa[0], pc['t'].T.copy(), pc['td'].T.copy(), pc['ps'], pc['ts'], pc['tds'])
    for x, y in zip(hip.cape(*pa, p_shared=True, **kw),
                    hip.cape(*pl, p_shared=True, level_major=True, **kw)):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize('adiabat', [1, 3, 4])
@pytest.mark.parametrize('source', [1, 2, 3])
def test_warm_grid_matches_ragged_warm(hip, source, adiabat):
    """A uniform batch through a ragged plan (staged in sorted order, each
    column's level count, source and output slot passed to the warm kernels)
    gives the grid call's warm results and work counters bit for bit."""
    import torch

    from xcape_amd.ragged import RaggedBatch, RaggedPlan
    c = synthetic.sigma_columns(3000, 60, 31, winds=False)
    g = hip.cape(c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'], pinc=500.,
                 source=source, adiabat=adiabat, warm_start='extrapolation', stats=True)
    n = c['t'].shape[0]
    d = dict(offsets=np.arange(n + 1, dtype=np.int64) * 60, p=c['p'].ravel(),
             t=c['t'].ravel(), td=c['td'].ravel(), ps=c['ps'], ts=c['ts'], tds=c['tds'],
             source=np.full(n, source, np.int32), adiabat=np.full(n, adiabat, np.int32))
    b = RaggedBatch.from_dict(d)
    plan = RaggedPlan(b, pinc=500., ml_depth=500., chunk=64, tile=0, cols=256, warm_start=True)
    st = plan.run(stats=True)
    torch.cuda.synchronize()
    r = [x.cpu().numpy() for x in (b.cape, b.cin, b.mulev, b.zmulev)]
    plan.close()
    for x, y in zip(g[:4], r):
        np.testing.assert_array_equal(x, y)
    for key in ('levels', 'substeps', 'iterations', 'fallbacks', 'nonconverged'):
        assert g[4][key] == st[key], key


def test_deep_columns_take_the_tile_transpose(hip):
    """Columns of more than 255 levels are staged by the tiled transpose
    (the slab kernel holds up to 255 levels of 64 columns in LDS): results
    equal the level-major call's."""
    c = synthetic.sigma_columns(500, 300, 41)
    lm = (c['p'].T.copy(), c['t'].T.copy(), c['td'].T.copy(), c['ps'], c['ts'], c['tds'])
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    for warm in (False, 'extrapolation'):
        kw = dict(pinc=500., source=2, adiabat=3, warm_start=warm)
        for x, y in zip(hip.cape(*args, **kw), hip.cape(*lm, level_major=True, **kw)):
            np.testing.assert_array_equal(x, y)


def test_staged_chunks_match_level_major(hip, monkeypatch):
    """Grids larger than one scratch chunk are computed chunk by chunk
    (outputs offset per chunk, 4- or 8-byte elements): forced here to 700
    columns a chunk, 3000 columns give five chunks, the last one partial.
    Column-contiguous (staged) and level-major input, chunked, both equal the
    unchunked level-major call's outputs."""
    c = synthetic.sigma_columns(3000, 60, 23, winds=True)
    lmj = {k: (c[k].T.copy() if c[k].ndim == 2 else c[k]) for k in c}
    cols = ('p', 't', 'td', 'ps', 'ts', 'tds')
    wcols = ('p', 't', 'td', 'u', 'v', 'ps', 'ts', 'tds', 'us', 'vs')
    cases = [dict(), dict(warm_start='extrapolation'), dict(fp64=True), dict(fast_math=True),
             dict(warm_start='extrapolation', fast_math=True)]
    monkeypatch.delenv('XCAPE_STAGE_COLUMNS', raising=False)
    ref = [hip.cape(*(lmj[k] for k in cols), level_major=True, pinc=500., source=2,
                    adiabat=3, **kw) for kw in cases]
    ref_srh = [hip.srh(*(lmj[k] for k in wcols), level_major=True, fp64=f)
               for f in (False, True)]
    ref_fused = hip.cape_srh(*(lmj[k] for k in wcols), pinc=500., source=2, adiabat=3,
                             warm_start='extrapolation', level_major=True)
    monkeypatch.setenv('XCAPE_STAGE_COLUMNS', '700')
    for kw, r in zip(cases, ref):
        for lm in (False, True):
            src = lmj if lm else c
            x = hip.cape(*(src[k] for k in cols), level_major=lm, pinc=500., source=2,
                         adiabat=3, **kw)
            for a, b in zip(x, r):
                np.testing.assert_array_equal(a, b)
    for fp64, r in zip((False, True), ref_srh):
        x = hip.srh(*(c[k] for k in wcols), fp64=fp64)
        for a, b in zip(x, r):
            np.testing.assert_array_equal(a, b)
    x = hip.cape_srh(*(c[k] for k in wcols), pinc=500., source=2, adiabat=3,
                     warm_start='extrapolation')
    for a, b in zip(x, ref_fused):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize('ncol', [1, 63, 700, 2047, 2049])
def test_warm_small_grids(hip, oracle_lib, ncol):
    """Grids smaller than the device: the persistent ascent's grid shrinks to
    the columns (and its work parts with it); every column is computed."""
    c = synthetic.sigma_columns(ncol, 60, 900 + ncol)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    o = oracle_lib.cape(*args, pinc=500., source=2, adiabat=3)
    for warm in ('extrapolation', 'cold'):
        g = hip.cape(*args, pinc=500., source=2, adiabat=3, warm_start=warm)
        assert not _report(f'small {ncol} {warm} cape', g[0], o[0]).any()
        assert not _report(f'small {ncol} {warm} cin', g[1], o[1]).any()
        np.testing.assert_array_equal(g[2], o[2])


@pytest.mark.parametrize('adiabat', [1, 2, 3, 4])
@pytest.mark.parametrize('source', [1, 2, 3])
def test_warm_start_within_tolerance(hip, oracle_lib, source, adiabat):
    """The warm-started iteration converges to the reference's tolerance from
    a predicted first iterate: results stay within 0.5 J/kg / 0.1 % of the
    cold-start oracle and the iteration count drops."""
    c = synthetic.sigma_columns(4096, 137, 1004)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    w = hip.cape(*args, pinc=500., source=source, adiabat=adiabat, warm_start=True, stats=True)
    p = hip.cape(*args, pinc=500., source=source, adiabat=adiabat, stats=True)
    o = oracle_lib.cape(*args, pinc=500., source=source, adiabat=adiabat)
    print('warm', w[4], 'plain', p[4], flush=True)
    assert not _report(f'warm s{source} a{adiabat} cape', w[0], o[0]).any()
    assert not _report(f'warm s{source} a{adiabat} cin', w[1], o[1]).any()
    np.testing.assert_array_equal(w[2], p[2])           # source selection untouched
    assert w[4]['substeps'] == p[4]['substeps'] or source == 2
    assert w[4]['iterations'] < 0.4 * p[4]['iterations']
    assert w[4]['fallbacks'] < 0.1 * w[4]['substeps']


def test_warm_start_fast_math(hip, oracle_lib):
    c = synthetic.sigma_columns(4096, 137, 1004)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    w = hip.cape(*args, pinc=500., source=2, adiabat=3, warm_start=True, fast_math=True)
    o = oracle_lib.cape(*args, pinc=500., source=2, adiabat=3)
    assert not _report('warm fast cape', w[0], o[0]).any()
    assert not _report('warm fast cin', w[1], o[1]).any()


@pytest.mark.parametrize('source', [1, 2, 3])
@pytest.mark.parametrize('adiabat', [1, 3, 4])
def test_lfc_el_against_oracle(hip, oracle_lib, source, adiabat):
    """LFC and EL (xcape_cape_levels_f32; no reference output, the oracle
    restates their definition from the reference's crossing pressure): the
    plain method within 0.05 hPa of the oracle's for 99.5 % of the columns
    (the device's exp/log/pow differ from the host's by an ulp, which moves a
    crossing where the layer's buoyancy barely changes), the warm start within
    1 hPa for 99 % (its fixed points move within the solver tolerance); both
    present exactly where CAPE is positive; asking for them leaves the other
    outputs unchanged."""
    c = synthetic.sigma_columns(3000, 80, 61)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    kw = dict(pinc=500., source=source, adiabat=adiabat)
    o = oracle_lib.cape(*args, levels=True, **kw)
    for warm, tol, share in ((False, 0.05, 0.995), ('extrapolation', 1.0, 0.99)):
        g = hip.cape(*args, warm_start=warm, levels=True, **kw)
        base = hip.cape(*args, warm_start=warm, **kw)
        for x, y in zip(g[:4], base):
            np.testing.assert_array_equal(x, y)
        pos = g[0] > 0
        np.testing.assert_array_equal(np.isfinite(g[4]), pos)
        np.testing.assert_array_equal(np.isfinite(g[5]), pos)
        assert np.all(g[4][pos] >= g[5][pos])
        both = pos & (o[0] > 0)
        assert np.mean(pos == (o[0] > 0)) >= 0.999
        for name, x, y in (('lfc', g[4], o[4]), ('el', g[5], o[5])):
            d = np.abs(x[both] - y[both])
            print(f'{name} s{source} a{adiabat} {warm}: max {d.max():.3g} '
                  f'within {np.mean(d <= tol):.4f}', flush=True)
            assert np.mean(d <= tol) >= share


def test_lfc_el_pressure_grid_and_small(hip, oracle_lib):
    """Shared pressure levels with start levels, and a grid of 37 columns,
    warm-started (the persistent ascent on a small grid)."""
    c = synthetic.pressure_columns(2000, 1003)
    st = oracle_lib.start_levels(c['p'], c['ps'])
    o = oracle_lib.cape(None, c['t'], c['td'], c['ps'], c['ts'], c['tds'], 500., 2, 500., 3,
                        p1d=c['p'], start_lev=st, levels=True)
    g = hip.cape(c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'], pinc=500., source=2,
                 adiabat=3, p_shared=True, levels=True)
    both = (g[0] > 0) & (o[0] > 0)
    assert both.sum() > 100
    assert np.mean(np.abs(g[4][both] - o[4][both]) <= 0.05) >= 0.995
    assert np.mean(np.abs(g[5][both] - o[5][both]) <= 0.05) >= 0.995
    s = synthetic.sigma_columns(37, 60, 62)
    a = (s['p'], s['t'], s['td'], s['ps'], s['ts'], s['tds'])
    w = hip.cape(*a, pinc=500., source=1, adiabat=1, warm_start='extrapolation', levels=True)
    r = oracle_lib.cape(*a, pinc=500., source=1, adiabat=1, levels=True)
    np.testing.assert_array_equal(np.isfinite(w[4]), w[0] > 0)
    pos = (w[0] > 0) & (r[0] > 0)
    assert np.all(np.abs(w[4][pos] - r[4][pos]) <= 1.0)


def test_lfc_el_fp64(hip, oracle_lib):
    """xcape_cape_levels_f64 (the FP64 re-run's LFC and EL) against the
    oracle's FP64 run: the same columns with positive area, LFC and EL within
    1e-3 hPa (the device's and the host's double exp/log/pow differ by an
    ulp, far below the FP32 spread); its CAPE, CIN and levels equal
    xcape_cape_f64's."""
    c = synthetic.sigma_columns(2000, 80, 63)
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    for source, adiabat in ((1, 1), (3, 3)):
        kw = dict(pinc=500., source=source, adiabat=adiabat)
        g = hip.cape(*args, fp64=True, levels=True, **kw)
        base = hip.cape(*args, fp64=True, **kw)
        for x, y in zip(g[:4], base):
            np.testing.assert_array_equal(x, y)
        assert g[4].dtype == np.float64
        o = oracle_lib.cape(*args, fp64=True, levels=True, **kw)
        pos = g[0] > 0
        assert pos.sum() > 100
        np.testing.assert_array_equal(pos, o[0] > 0)
        np.testing.assert_array_equal(np.isfinite(g[4]), pos)
        for x, y in ((g[4], o[4]), (g[5], o[5])):
            d = np.abs(x[pos] - y[pos])
            print(f'fp64 levels s{source} a{adiabat}: max {d.max():.3g}', flush=True)
            assert np.all(d <= 1e-3)


def test_cin_disagreements_only_where_the_reference_is_ill_conditioned(hip, oracle_lib):
    """On the 2048x1024x137 grid, every variant's CAPE agrees with the plain
    accurate kernel within max(0.5 J/kg, 0.1 %) everywhere.  CIN may not
    agree only where the reference's own CIN is ill-conditioned: it commits
    the accumulated CIN on the first entry into positive buoyancy
    (CAPE_CODE_model_lev.f90:509-523), so a layer whose buoyancy is within
    rounding of zero commits it under one rounding, or one accepted iterate,
    and not under another.  There the oracle's own runs (FP64, perturbed
    library, perturbed accepted iterates) disagree beyond the tolerance, and
    each variant is within tolerance of one of them.  Such columns are
    rare."""
    import torch
    ncol = 2048 * 1024
    inp = synthetic.sigma_columns_torch(ncol, 137, 4004, device='cuda')
    cols = [inp[k] for k in ('p', 't', 'td', 'ps', 'ts', 'tds')]
    lm = [inp[k].t().contiguous() for k in ('p', 't', 'td')] + \
         [inp[k] for k in ('ps', 'ts', 'tds')]
    kw = dict(pinc=500., source=2, adiabat=3, level_major=True)
    ref = hip.cape(*lm, **kw)
    for extra in (dict(warm_start=True), dict(fast_math=True),
                  dict(fast_math=True, warm_start=True)):
        got = hip.cape(*lm, **kw, **extra)
        tol = [(1e-3 * r.double().abs()).clamp(min=0.5) for r in ref[:2]]
        dcape = (got[0].double() - ref[0].double()).abs()
        dcin = (got[1].double() - ref[1].double()).abs()
        assert bool((dcape <= tol[0]).all()), extra
        off = torch.nonzero(dcin > tol[1]).flatten()
        print(extra, 'CIN outside tolerance:', off.tolist(), flush=True)
        assert len(off) <= ncol // 10000, extra
        if len(off):
            host = [x[off].cpu().numpy() for x in cols]
            o = off.cpu().numpy()

            def run(c, **kw):
                j = np.searchsorted(o, c)
                return oracle_lib.cape(*(a[j] for a in host), pinc=500., source=2, adiabat=3,
                                       **kw)
            ill, matched = ill_conditioned_and_matched(
                run, o, [(got[0][off].cpu().numpy(), got[1][off].cpu().numpy()),
                         (ref[0][off].cpu().numpy(), ref[1][off].cpu().numpy())])
            assert ill.all() and matched.all(), (extra, o, ill, matched)
    torch.cuda.synchronize()


@pytest.mark.parametrize('warm', [False, True])
def test_pressure_per_column_with_start_levels(hip, oracle_lib, warm):
    """loopcape_pl (CAPE_CODE_pressure_lev.f90:4-84): pressure per column on a
    pressure grid, each column from its own start level.  Against the oracle
    (pinned bit-exact to the compiled loopcape_pl on the CPU); with the shared
    levels repeated per column, equal to the shared-levels call."""
    c = synthetic.pressure_columns(3000, 1013)
    st = oracle_lib.start_levels(c['p'], c['ps'])
    rng = np.random.default_rng(11)
    p2 = (c['p'][None, :] * (1.0 + 0.001 * rng.uniform(-1.0, 1.0, (3000, 1)))).astype(np.float32)
    kw = dict(pinc=500., source=2, adiabat=3, warm_start=warm)
    g = hip.cape(p2, c['t'], c['td'], c['ps'], c['ts'], c['tds'], start_lev=st, **kw)
    o = oracle_lib.cape(p2, c['t'], c['td'], c['ps'], c['ts'], c['tds'], 500., 2, 500., 3,
                        start_lev=st)
    assert np.all(np.isfinite(g[0])) and np.all(np.isfinite(g[1]))
    assert not _report(f'pressure per column warm={warm} cape', g[0], o[0]).any()
    assert not _report(f'pressure per column warm={warm} cin', g[1], o[1]).any()
    assert np.mean(g[2] == o[2]) >= 0.999
    tiled = np.tile(np.asarray(c['p'], np.float32), (3000, 1))
    a = hip.cape(tiled, c['t'], c['td'], c['ps'], c['ts'], c['tds'], start_lev=st, **kw)
    b = hip.cape(c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'], p_shared=True,
                 start_lev=st, **kw)
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)
    with pytest.raises(RuntimeError):
        hip.srh(p2, c['t'], c['td'], c['t'], c['td'], c['ps'], c['ts'], c['tds'], c['ts'],
                c['tds'], start_lev=st)


@pytest.fixture(scope='module')
def pressure_grid():
    return synthetic.pressure_columns(1024 * 512, 2024)


@pytest.mark.parametrize('source', [1, 3, 2])
def test_pressure_grid_full_size(hip, oracle_lib, pressure_grid, source):
    """The pressure-level configuration at its full size: 1024x512 columns x
    37 fixed levels, pseudo-liquid, the shared-levels path with start levels
    from the device's own rule, for each of its three runs: surface,
    mixed-layer (500 m) and most-unstable.  Size-independent checks on every
    column (outputs finite and non-negative, MUlev inside the column, the
    warm start within tolerance of the plain method for CAPE, CIN only where
    CAPE vanishes, the same MUlev, host arrays streamed equal to device
    arrays), and a random sample of 2000 columns against the oracle."""
    import torch
    n = 1024 * 512
    c = pressure_grid
    args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
    kw = dict(pinc=500., source=source, ml_depth=500., adiabat=1, p_shared=True)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in args]
    plain = [x.cpu().numpy() for x in hip.cape(*dev, **kw)]
    warm = [x.cpu().numpy() for x in hip.cape(*dev, warm_start=True, **kw)]
    host = hip.cape(*args, **kw)
    torch.cuda.synchronize()
    for x, y in zip(host, plain):
        np.testing.assert_array_equal(x, y)
    assert np.all(np.isfinite(plain[0])) and np.all(np.isfinite(plain[1]))
    assert (plain[0] >= 0).all() and (plain[1] >= 0).all()
    assert cape_ok(warm[0], plain[0]).all()
    off = np.nonzero(~cape_ok(warm[1], plain[1]))[0]
    print(f'pressure grid source {source}: CIN outside tolerance', off.tolist(), flush=True)
    assert len(off) <= n // 10000
    if len(off):
        # where the warm start and the plain method disagree on CIN, the
        # reference's own CIN is ill-conditioned (committed at a near-zero
        # buoyancy crossing: it turns on the last bit of the C library or on
        # the iterate accepted within the convergence tolerance), and each
        # of them is within tolerance of one of the oracle's runs
        def run(cols, **kw):
            return oracle_lib.cape(None, c['t'][cols], c['td'][cols], c['ps'][cols],
                                   c['ts'][cols], c['tds'][cols], 500., source, 500., 1,
                                   p1d=c['p'], start_lev=oracle_lib.start_levels(
                                       c['p'], c['ps'][cols]), **kw)
        ill, matched = ill_conditioned_and_matched(
            run, off, [(warm[0][off], warm[1][off]), (plain[0][off], plain[1][off])])
        assert ill.all() and matched.all(), (off, ill, matched)
    np.testing.assert_array_equal(warm[2], plain[2])
    live = c['ts'] > 0
    if source == 2:
        # the most-unstable level: 1 (the surface) .. the column's last level
        assert (plain[2][live] >= 1).all() and (plain[2][live] <= len(c['p']) + 1).all()
    else:
        # no most-unstable search: the reference's -999999
        assert (plain[2][live] == -999999).all()
    idx = np.sort(np.random.default_rng(5).choice(n, 2000, replace=False))
    st = oracle_lib.start_levels(c['p'], c['ps'][idx])
    o = oracle_lib.cape(None, c['t'][idx], c['td'][idx], c['ps'][idx], c['ts'][idx],
                        c['tds'][idx], 500., source, 500., 1, p1d=c['p'], start_lev=st)
    assert not _report('pressure grid sample cape', plain[0][idx], o[0]).any()
    assert not _report('pressure grid sample cin', plain[1][idx], o[1]).any()
    np.testing.assert_array_equal(plain[2][idx], o[2])


def test_staging_of_unaligned_and_even_level_inputs(hip):
    """The staging transpose copies 16 bytes per lane when the profiles are
    16-byte aligned and the level count odd, 4 bytes otherwise: device
    inputs starting 4 bytes into an allocation, and an even level count,
    give the results of aligned copies of the same columns."""
    import torch
    for nk in (137, 40):
        c = synthetic.sigma_columns(3001, nk, 77)
        args = (c['p'], c['t'], c['td'], c['ps'], c['ts'], c['tds'])
        kw = dict(pinc=500., source=2, adiabat=3, warm_start=True)
        ref = [x.cpu() for x in hip.cape(*[torch.from_numpy(a).cuda() for a in args], **kw)]
        # the same columns at an odd float offset into a larger buffer
        shifted = []
        for a in args[:3]:
            buf = torch.empty(a.size + 1, dtype=torch.float32, device='cuda')
            view = buf[1:].view(a.shape)
            view.copy_(torch.from_numpy(a))
            assert view.data_ptr() % 16 != 0
            shifted.append(view)
        got = hip.cape(*shifted, *[torch.from_numpy(a).cuda() for a in args[3:]], **kw)
        for x, y in zip(got, ref):
            assert torch.equal(x.cpu(), y), nk


def test_warm_parts_match_one_launch(hip, monkeypatch):
    """Warm-started grids of 2^20 column-contiguous columns or more are staged
    in four parts, each part's setup pass beside the next part's copies, then
    one ascent over every column; forced here down to 128 columns (3000
    columns: parts of 768, the last of 696).  Every output (LFC/EL too), the
    per-column kernel counts and the fused call's helicity equal the one-launch
    call's: the extrapolation, the surrogate's first iterates, the cold loop,
    fast math, sigma and shared pressure levels.  Last in this file: it loads
    the surrogate."""
    from xcape_amd import surrogate
    surrogate.Surrogate.load().activate()
    c = synthetic.sigma_columns(3000, 137, 37, winds=True)
    pc = synthetic.pressure_columns(3000, 38)
    cols = ('p', 't', 'td', 'ps', 'ts', 'tds')
    wcols = ('p', 't', 'td', 'u', 'v', 'ps', 'ts', 'tds', 'us', 'vs')
    kw0 = dict(pinc=500., source=2, adiabat=3)
    cases = [dict(warm_start='extrapolation', stats=True), dict(warm_start=True, stats=True),
             dict(warm_start='cold', stats=True), dict(warm_start='extrapolation', levels=True),
             dict(warm_start=True, fast_math=True, stats=True)]

    def run():
        out = [hip.cape(*(c[k] for k in cols), **kw0, **kw) for kw in cases]
        out.append(hip.cape(*(pc[k] for k in cols), pinc=500., source=1, adiabat=1,
                            p_shared=True, warm_start=True, stats=True))
        for ws in ('extrapolation', True):
            out.append(hip.cape_srh(*(c[k] for k in wcols), **kw0, depth=3000., warm_start=ws,
                                    stats=True))
        return out

    monkeypatch.delenv('XCAPE_STAGE_COLUMNS', raising=False)
    monkeypatch.delenv('XCAPE_WARM_PIPE_COLUMNS', raising=False)
    ref = run()
    monkeypatch.setenv('XCAPE_WARM_PIPE_COLUMNS', '128')
    got = run()
    for x, r in zip(got, ref):
        assert len(x) == len(r)
        for a, b in zip(x, r):
            if isinstance(b, dict):
                # the per-column counts (the wave-level ones follow the columns'
                # packing into waves)
                per_col = [k for k in b if k not in ('wave_trips', 'blocks')]
                assert {k: a[k] for k in per_col} == {k: b[k] for k in per_col}
            else:
                np.testing.assert_array_equal(a, b)
    assert got[0][-1]['columns'] == 3000


@pytest.mark.parametrize('levels', [False, True])
@pytest.mark.parametrize('ncol', [1, 2, 65, 1023, 1025, 5000, 33000])
def test_warm_small_launches_match_the_large(hip, ncol, levels):
    """A warm ascent of fewer columns than the device has lanes spreads them
    over its waves, a few to each; a column's result does not depend on it."""
    import torch
    c = synthetic.sigma_columns(70000, 24, 19)
    args = [torch.from_numpy(np.ascontiguousarray(c[k])).cuda()
            for k in ('p', 't', 'td', 'ps', 'ts', 'tds')]
    kw = dict(pinc=700., source=2, adiabat=3, warm_start=True, levels=levels)
    whole = hip.cape(*args, **kw)
    part = hip.cape(*(a[:ncol] for a in args), **kw)
    for w, p in zip(whole, part):
        np.testing.assert_array_equal(p.cpu().numpy(), w[:ncol].cpu().numpy())


@pytest.mark.parametrize('adiabat', [1, 2, 3, 4])
@pytest.mark.parametrize('ncol,nk', [(1, 60), (63, 40), (1024, 40), (1025, 33), (2111, 40),
                                     (65537, 24), (131072, 20), (131073, 20)])
def test_small_launches_match_the_large_loop(hip, adiabat, ncol, nk):
    """Plain launches of at most two waves per SIMD spread their columns over
    the waves and iterate with a loop of their own; counted launches always
    take the large grids' loop.  Same columns, same bits, on both sides of the
    limit and with a partly filled last wave."""
    import torch
    c = synthetic.sigma_columns_torch(ncol, nk, 7 * ncol + adiabat)
    args = [c[k] for k in ('p', 't', 'td', 'ps', 'ts', 'tds')]
    kw = dict(pinc=500., source=1 + adiabat % 3, adiabat=adiabat)
    small = hip.cape(*args, **kw)
    large = hip.cape(*args, stats=True, **kw)
    for a, b in zip(small, large[:4]):
        assert torch.equal(a, b)
    assert large[4]['columns'] == ncol


@pytest.mark.parametrize('adiabat', [1, 2, 3, 4])
@pytest.mark.parametrize('mode', [dict(fast_math=True), dict(fp64=True)])
@pytest.mark.parametrize('ncol', [1, 1025, 4096, 4097, 20011, 131072])
def test_small_launches_match_the_large_in_fast_math_and_fp64(hip, mode, adiabat, ncol):
    """Fast math and FP64 spread a small launch's columns over the waves too,
    in a kernel of their own (fast reversible-liquid launches of up to 4 columns
    a wave, the others of up to 64): on both sides of these limits a column's
    result is that of a launch larger than all of them, bit for bit."""
    import torch
    c = synthetic.sigma_columns_torch(131073, 16, 40 + adiabat)
    args = [c[k] for k in ('p', 't', 'td', 'ps', 'ts', 'tds')]
    kw = dict(pinc=2500., source=1 + adiabat % 3, adiabat=adiabat, **mode)
    whole = hip.cape(*args, **kw)
    part = hip.cape(*(a[:ncol].contiguous() for a in args), **kw)
    for w, p in zip(whole, part):
        assert torch.equal(p, w[:ncol])


@pytest.mark.parametrize('adiabat', [1, 2, 3, 4])
@pytest.mark.parametrize('ncol', [1, 63, 2111, 131072])
def test_three_loops_agree(hip, ncol, adiabat):
    """The accurate mode's loops: a launch of more than two waves per SIMD
    leaves lanes and phases out, a counted one below that leaves out lanes, an
    uncounted one nothing.  A column's result is the same in each, bit for
    bit, columns that stop at the iteration limit and NaN levels included."""
    import edge_cases
    import torch
    c = synthetic.sigma_columns_torch(131073, 30, 90 + adiabat)
    args = [c[k] for k in ('p', 't', 'td', 'ps', 'ts', 'tds')]
    for a, e in zip(args, edge_cases.grid()):
        a[:128] = torch.from_numpy(e).cuda()
    kw = dict(pinc=500., source=1 + adiabat % 3, adiabat=adiabat)
    whole = hip.cape(*args, **kw)
    part = [a[:ncol].contiguous() for a in args]
    few = hip.cape(*part, **kw)
    counted = hip.cape(*part, stats=True, **kw)
    for w, f, m in zip(whole, few, counted):
        w = w[:ncol].nan_to_num(nan=-7e7)
        assert torch.equal(f.nan_to_num(nan=-7e7), w)
        assert torch.equal(m.nan_to_num(nan=-7e7), w)
