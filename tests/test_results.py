"""Results finalisation and multi-sim reduction (covasim/sim.py:764-1001, covasim/run.py:220-303).

CPU: the numpy restatement (oracle/results_ref.py) is pinned by closed forms: cumulative flows of
constant series, the doubling time of an exact exponential, r_eff's mean infectious duration on a
hand-built population, the smoothing kernel's binomial spread of an impulse.
GPU: cvk_finalize equals the restatement on real runs (single sims and a batch): bit for bit on
flows, stocks and derived states, within 1e-13 relative on the doubling time (log) and 1e-5
relative on r_eff (the reference averages float32 dates in float32, the device in float64).
cvk_reduce equals numpy's quantile / mean / std over the sims.
"""

import os
import subprocess

import numpy as np
import pytest

from oracle import results_ref as rr


def test_smooth_spreads_an_impulse_binomially():
    x = np.zeros(11)
    x[5] = 16.0
    y = rr.smooth(x, 2)
    assert np.array_equal(y[3:8], [1, 4, 6, 4, 1])
    assert y.sum() == 16.0
    c = rr.smooth(np.full(9, 3.0), 1)
    assert np.array_equal(c[1:-1], np.full(7, 3.0)) and c[0] == c[-1] == 2.25  # zero beyond the ends


def test_doubling_time_of_an_exponential():
    t = np.arange(30)
    cum = 10.0 * 2.0 ** (t / 5.0)
    d = rr.compute_doubling(cum)
    assert np.all(np.isnan(d[:3]))
    assert np.allclose(d[3:], 5.0, rtol=1e-12)
    slow = rr.compute_doubling(10.0 * 2.0 ** (t / 100.0))
    assert np.all(slow[3:] == 30)  # capped at max_doubling_time
    flat = rr.compute_doubling(np.full(10, 7.0))
    assert np.all(np.isnan(flat))


def test_r_eff_mean_infectious_duration():
    nan = np.nan
    d_inf = np.array([2, 5, 8, nan], np.float32)
    d_rec = np.array([10, nan, 20, nan], np.float32)
    d_dead = np.array([nan, 15, nan, nan], np.float32)
    new = np.array([4.0, 6.0, 0.0, 3.0, 1.0])
    imp = np.array([0.0, 2.0, 0.0, 0.0, 0.0])
    ninf = np.array([2.0, 4.0, 0.0, 3.0, 2.0])
    # outcomes 10, 20, 15 (mean 15) of agents infectious on days 2, 8, 5 (mean 5): 10 days
    r = rr.compute_r_eff(new, imp, ninf, d_inf, d_rec, d_dead, initial_period_par=0, smoothing=0)
    assert np.allclose(r, 10 * np.array([2.0, 1.0, 0.0, 1.0, 0.5]))
    r2 = rr.compute_r_eff(new, imp, ninf, d_inf, d_rec, d_dead, initial_period_par=2.5, smoothing=0)
    assert np.allclose(r2, [15.0, 10.0, 0.0, 10.0, 5.0])  # day 0 averages days 0..1
    r3 = rr.compute_r_eff(new, imp, ninf, d_inf, d_rec, d_dead, initial_period_par=0, smoothing=1)
    assert np.allclose(r3, [20.0, 10.0, 5.0, 6.25, 5.0])  # ends kept, interior (0.25, 0.5, 0.25)
    none = rr.compute_r_eff(new, imp, ninf, d_inf, np.full(4, nan, np.float32), np.full(4, nan, np.float32), 0, 2)
    assert np.all(none == 0)


def test_finalize_closed_forms():
    from covasim_amd import _lib
    npts, nv = 6, 1
    counts = np.zeros((npts, _lib.R_COLS), np.uint32)
    col = _lib.R_COL
    counts[:, col['new_infections']] = 2
    counts[:, col['new_deaths']] = [0, 0, 1, 0, 1, 0]
    counts[:, col['new_recoveries']] = 1
    counts[:, col['n_exposed']] = 10
    counts[:, col['n_infectious']] = 4
    counts[:, col['n_recovered']] = np.arange(npts)
    counts[:, col['n_alive']] = 100
    counts_f = np.zeros((npts, _lib.RF_COLS))
    nan = np.full(5, np.nan, np.float32)
    R = rr.finalize(counts, counts_f, col, _lib.R_BYVAR, _lib.MAX_VARIANTS, nv, 100.0, 5, False, None, nan, nan, nan,
                    0.0)
    assert np.array_equal(R['cum_infections'], 2.0 * np.arange(1, npts + 1) + 5)
    assert np.array_equal(R['n_alive'], 100 - np.array([0, 0, 1, 1, 2, 2.0]))
    assert np.array_equal(R['n_susceptible'], R['n_alive'] - 10 - np.arange(1, npts + 1))
    assert np.array_equal(R['prevalence'], 10 / R['n_alive'])
    assert np.array_equal(R['n_removed'], np.arange(1, npts + 1) + R['cum_deaths'])
    W = rr.finalize(counts, counts_f, col, _lib.R_BYVAR, _lib.MAX_VARIANTS, nv, 100.0, 5, True, None, nan, nan, nan,
                    0.0)
    assert np.array_equal(W['n_susceptible'], W['n_alive'] - 10)  # waning: recovered agents count as susceptible


def test_finalize_pop_infected_on_every_variant_row():
    """sim.py:785-786 adds pop_infected to cum_infections_by_variant as a whole (n_variants, npts)
    array, so every variant's row carries it, not only the wild type's."""
    from covasim_amd import _lib
    npts, nv = 5, 3
    counts = np.zeros((npts, _lib.R_COLS), np.uint32)
    base = _lib.R_BYVAR  # new_infections_by_variant columns
    counts[:, base + 0] = 3
    counts[:, base + 1] = [0, 0, 1, 2, 0]
    counts[:, base + 2] = 0
    counts_f = np.zeros((npts, _lib.RF_COLS))
    nan = np.full(4, np.nan, np.float32)
    R = rr.finalize(counts, counts_f, _lib.R_COL, _lib.R_BYVAR, _lib.MAX_VARIANTS, nv, 50.0, 7, False, None, nan,
                    nan, nan, 0.0)
    cum = R['variant']['cum_infections_by_variant']
    assert np.array_equal(cum[0], 3.0 * np.arange(1, npts + 1) + 7)
    assert np.array_equal(cum[1], np.array([0, 0, 1, 3, 3.0]) + 7)
    assert np.array_equal(cum[2], np.full(npts, 7.0))


@pytest.fixture(scope='module')
def smooth_schedule(tmp_path_factory):
    """The program that runs the device's smoothing on the CPU, a thread at a time between barriers."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = str(tmp_path_factory.mktemp('smooth') / 'smooth_schedule')
    subprocess.run(['g++', '-std=c++17', '-O1', '-pthread', '-I', os.path.join(root, 'covasim_amd', 'csrc'), '-o', exe,
                    os.path.join(root, 'tests', 'golden', 'smooth_schedule.cpp')], check=True)
    return exe


@pytest.mark.parametrize('descending', [0, 1])
@pytest.mark.parametrize('rounds', [0, 1, 2, 3, 8])
def test_smoothing_needs_no_luck_in_the_schedule(smooth_schedule, rounds, descending):
    """However far a thread runs ahead of the others between two barriers, the values are the restatement's."""
    for npts, threads in [(3, 2), (10, 4), (33, 32), (65, 64)]:
        raw = np.random.default_rng(npts).uniform(0.5, 2.0, npts)
        text = f'{npts} {rounds} {threads} {descending}\n' + '\n'.join(f'{x:.17g}' for x in raw)
        out = subprocess.run([smooth_schedule], input=text, capture_output=True, text=True, check=True, timeout=60).stdout
        want = rr.smooth(raw, rounds)
        if rounds:
            want[:rounds], want[-rounds:] = raw[:rounds], raw[-rounds:]
        np.testing.assert_allclose([float(x) for x in out.split()], want, rtol=1e-14, atol=0, err_msg=f'{npts} days')


# ---------------------------------------------------------------------------------------------
# GPU
# ---------------------------------------------------------------------------------------------
def oracle_rows(sim, batch=None, index=0):
    """The restatement applied to a finished covasim_amd Sim's tables and dates (read from the
    batch that ran it, when given)."""
    from covasim_amd import _lib
    from covasim_amd import results as cvres
    if batch is None:
        counts = sim._w['results'].cpu().numpy().view(np.uint32)
        counts_f = sim._w['results_f'].cpu().numpy()
        get = sim.people.get
    else:
        res, resf = batch.raw_results()
        counts, counts_f = res[index], resf[index]

        def get(key):
            return batch.get(key, index)
    dur = sim.pars['dur']
    return rr.finalize(counts, counts_f, _lib.R_COL, _lib.R_BYVAR, _lib.MAX_VARIANTS, int(sim.pars['n_variants']),
                       float(sim.people.n), sim.pars['pop_infected'], sim.pars['use_waning'], sim.import_schedule(),
                       get('date_infectious'), get('date_recovered'), get('date_dead'),
                       dur['exp2inf']['par1'] + dur['asym2rec']['par1']), cvres


def assert_rows_match(sim, want, cvres):
    for name in cvres.F_ROW_NAMES:
        got, exp = sim.results[name].values, np.asarray(want[name], dtype=float)
        if name == 'doubling_time':
            assert np.array_equal(np.isnan(got), np.isnan(exp)), name
            np.testing.assert_allclose(got[~np.isnan(got)], exp[~np.isnan(exp)], rtol=1e-13, err_msg=name)
        elif name == 'r_eff':
            np.testing.assert_allclose(got, exp, rtol=1e-5, atol=1e-9, err_msg=name)
        else:
            assert np.array_equal(got, exp, equal_nan=True), (name, got[:5], exp[:5])
    for name in cvres.FV_ROW_NAMES:
        assert np.array_equal(sim.results['variant'][name].values, want['variant'][name], equal_nan=True), name


@pytest.mark.gpu
@pytest.mark.parametrize('case', ['hybrid', 'variants_waning'])
def test_device_finalize_matches_restatement(case):
    import covasim_amd as cv
    from tests.helpers import copy_pop, make_population
    print(f'finalize case {case}', flush=True)
    if case == 'hybrid':
        pop = make_population(n=20000, pop_type='hybrid')
        sim = cv.Sim(pop_size=20000, pop_type='hybrid', n_days=60, rand_seed=3, beta=0.03, popdict=copy_pop(pop),
                     dynam_layer=dict(c=1))
    else:
        pop = make_population(n=20000, pop_type='random')
        sim = cv.Sim(pop_size=20000, n_days=50, rand_seed=5, beta=0.02, use_waning=True, popdict=copy_pop(pop),
                     variants=[cv.variant(dict(rel_beta=1.7), days=[10], n_imports=30)])
    sim.run()
    want, cvres = oracle_rows(sim)
    assert_rows_match(sim, want, cvres)
    assert sim.results['cum_infections'].values[-1] > 100
    assert np.isfinite(sim.results['r_eff'].values).all()


@pytest.mark.gpu
def test_batch_finalize_and_reduce():
    import torch
    import covasim_amd as cv
    from oracle import results_ref
    from tests.helpers import copy_pop, make_population
    sims = []
    for i, n in enumerate([5000, 12000, 8000, 3000]):
        pop = make_population(n=n, pop_type='hybrid', seed=i + 1)
        sims.append(cv.Sim(pop_size=n, pop_type='hybrid', n_days=40, rand_seed=10 + i, beta=0.03 + 0.005 * i,
                           popdict=copy_pop(pop), dynam_layer=dict(c=1)))
    b = cv.BatchSim(sims)
    b.run()
    for i, sim in enumerate(sims):
        want, cvres = oracle_rows(sim, batch=b, index=i)
        assert_rows_match(sim, want, cvres)
    red = b.reduce()
    med = b.reduce(quantiles=[0.25, 0.75])
    mean = b.reduce(use_mean=True, bounds=1.5)
    stack = np.stack([np.stack([s.results[k].values for k in cvres.F_ROW_NAMES]) for s in sims])
    for got, kw in [(red, {}), (med, dict(quantiles=(0.25, 0.75))), (mean, dict(use_mean=True, bounds=1.5))]:
        c, lo, hi = results_ref.reduce(stack, **kw)
        for i, k in enumerate(cvres.F_ROW_NAMES):
            assert np.array_equal(got[k].values, c[i], equal_nan=True), k
            assert np.array_equal(got[k].low, lo[i], equal_nan=True), k
            assert np.array_equal(got[k].high, hi[i], equal_nan=True), k
    torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize('S', [1, 2, 7, 256, 1000, 4096])
def test_device_reduce_matches_numpy(S):
    import torch
    from covasim_amd import results as cvres
    rng = np.random.default_rng(S)
    vals = rng.normal(size=(S, 3, 37)) * 10.0 ** rng.integers(-3, 4, size=(1, 3, 37))
    vals[:, 0, :5] = np.round(vals[:, 0, :5])  # ties
    vals[rng.integers(S), 1, 3] = np.nan
    vals[:, 2, 7] = np.inf if S > 1 else 1.0
    t = torch.as_tensor(vals, device='cuda')
    for kw in [dict(), dict(quantiles={'low': 0.05, 'high': 0.95}), dict(quantiles=[0.0, 1.0]),
               dict(use_mean=True), dict(use_mean=True, bounds=3)]:
        got = [x.cpu().numpy() for x in cvres.reduce_tables(t, **kw)]
        q = kw.get('quantiles', (0.1, 0.9))
        q = (q['low'], q['high']) if isinstance(q, dict) else tuple(q)
        with np.errstate(invalid='ignore'):
            want = rr.reduce(vals, quantiles=q, use_mean=kw.get('use_mean', False), bounds=kw.get('bounds', 2))
        for g, w in zip(got, want):
            assert np.array_equal(g, w, equal_nan=True), (kw, np.argwhere(~((g == w) | (np.isnan(g) & np.isnan(w))))[:5])


@pytest.mark.gpu
@pytest.mark.parametrize('days', [0, 1, 2, 3, 4, 11, 12, 27, 28, 59, 63, 64, 128])
def test_day_counts_around_waves_and_graph_parts(days):
    """Rows of days + 1 points against the restatement (the series are summed by waves of 64 days), from a run in
    graphs of 4, 8, 16, 32, .. days on a stream of its own, which an eager run equals."""
    import covasim_amd as cv
    import torch
    print(f'{days} days', flush=True)

    def run(graph):
        sim = cv.Sim(pop_size=3000, pop_type='hybrid', n_days=days, rand_seed=4, beta=0.03, use_waning=True,
                     dynam_layer=dict(c=1), variants=[cv.variant(dict(rel_beta=1.5), days=2, n_imports=20)],
                     interventions=[cv.test_prob(symp_prob=0.2, asymp_prob=0.01), cv.contact_tracing(trace_time=1)])
        stream = torch.cuda.Stream() if graph else torch.cuda.current_stream()
        with torch.cuda.stream(stream):
            sim.run(use_graph=graph)
        return sim
    parts, eager = run(True), run(False)
    for key, res in eager.results.items():
        if hasattr(res, 'values') and not callable(res.values):
            assert np.array_equal(res.values, parts.results[key].values, equal_nan=True), key
    want, cvres = oracle_rows(parts)
    assert_rows_match(parts, want, cvres)


@pytest.mark.gpu
@pytest.mark.parametrize('npts', [3, 64, 65, 181, 1100])
@pytest.mark.parametrize('smoothing', [0, 1, 2, 3, 40])
def test_r_eff_smoothing_matches_restatement(npts, smoothing):
    """Every count of smoothing rounds, on days within one wave, across waves and past one workgroup's threads. The
    16 agents' dates are small whole numbers, so their means are exact; a round is three roundings of positive terms
    (2^-53 each), 40 rounds and the mean stay below 2^-45."""
    import torch
    from covasim_amd import _lib
    from covasim_amd import results as cvres
    S, n = 48, 16
    rng = np.random.default_rng(npts)
    counts = np.zeros((S, npts, _lib.R_COLS), np.uint32)
    counts[:, :, _lib.R_COL['new_infections']] = rng.integers(1, 1000, (S, npts))
    counts[:, :, _lib.R_COL['n_infectious']] = rng.integers(1, 1000, (S, npts))
    counts_f = np.zeros((S, npts, _lib.RF_COLS))
    d_inf = rng.integers(0, 20, S * n).astype(np.float32)
    d_rec = d_inf + 8
    nan = np.full(S * n, np.nan, np.float32)
    period = min(npts, 12)
    dev = lambda a: torch.from_numpy(a).cuda()
    rows, _ = cvres.finalize_tables(dev(counts.view(np.int32)), dev(counts_f), npts, 1, False, np.zeros(S),
                                    np.full(S, period), np.arange(S + 1) * n, None, dev(d_inf), dev(d_rec), dev(nan),
                                    smoothing=smoothing)
    got = rows[:, cvres.F_ROW_NAMES.index('r_eff')].cpu().numpy()
    for s in range(S):
        want = rr.compute_r_eff(counts[s, :, _lib.R_COL['new_infections']].astype(float), np.zeros(npts),
                                counts[s, :, _lib.R_COL['n_infectious']].astype(float), d_inf[s * n:(s + 1) * n],
                                d_rec[s * n:(s + 1) * n], nan[:n], period, smoothing)
        np.testing.assert_allclose(got[s], want, rtol=2.0 ** -45, atol=0, err_msg=f'sim {s}')


@pytest.mark.gpu
def test_import_refused_before_a_graph_run_starts():
    """An import event that cannot be drawn (a variant the run does not have) is refused before any day has run, also
    where its day lies in a later graph than the first."""
    import ctypes as C

    import covasim_amd as cv
    import torch
    from covasim_amd import _lib
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        sim = cv.Sim(pop_size=2000, n_days=40, rand_seed=4,
                     variants=[cv.variant(dict(rel_beta=1.5), days=30, n_imports=5)])
        sim.initialize()
        torch.cuda.synchronize()
        imp = _lib.ImportsS.from_buffer_copy(sim._imports)
        assert imp.n == 1
        vars_ = (C.c_int32 * 1)(7)
        imp.variants = C.cast(vars_, C.POINTER(C.c_int32))
        before = sim.people.snapshot()
        rc = _lib.lib().cvk_run_days(sim.people.struct(), sim._layers, sim._params, sim._work, 0, sim.npts, 20,
                                     C.byref(imp), 1, C.c_void_p(stream.cuda_stream))
        torch.cuda.synchronize()
    assert rc != 0
    after = sim.people.snapshot()
    assert all(np.array_equal(before[k], after[k], equal_nan=True) for k in before)


@pytest.mark.gpu
def test_layer_refused_before_a_graph_run_starts():
    """A resampled layer whose weights the last day's close could not write (their address is no multiple of 8) is
    refused before any day has run, also where no earlier day touches them (the contacts are generated)."""
    import ctypes as C

    import covasim_amd as cv
    import torch
    from covasim_amd import _lib
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        sim = cv.Sim(pop_size=2000, pop_type='hybrid', n_days=20, rand_seed=4, dynam_layer=dict(c=1))
        sim.initialize()
        torch.cuda.synchronize()
        layers = type(sim._layers).from_buffer_copy(sim._layers)
        index = sim.layer_keys().index('c')
        assert layers[index].dynamic
        layers[index].beta += 4
        layers[index].n_edges -= 1
        before = sim.people.snapshot()
        _lib.check(_lib.lib().cvk_set_tuning(_lib.TUNE_GENERATE_DYNAMIC, 1), 'tuning')
        try:
            rc = _lib.lib().cvk_run_days(sim.people.struct(), layers, sim._params, sim._work, 0, sim.npts, 20,
                                         C.byref(sim._imports), 1, C.c_void_p(stream.cuda_stream))
        finally:
            _lib.check(_lib.lib().cvk_set_tuning(_lib.TUNE_GENERATE_DYNAMIC, 2), 'tuning')
        torch.cuda.synchronize()
    assert rc == _lib.E_ALIGN
    after = sim.people.snapshot()
    assert all(np.array_equal(before[k], after[k], equal_nan=True) for k in before)


@pytest.mark.gpu
def test_more_graph_parts_than_are_kept_at_once():
    """2100 days are 66 parts, the first 64 released while the run goes on: the results are an eager run's."""
    import covasim_amd as cv
    import torch

    def run(graph):
        sim = cv.Sim(pop_size=300, pop_type='hybrid', n_days=2100, rand_seed=4, beta=0.03, use_waning=True,
                     dynam_layer=dict(c=1))
        with torch.cuda.stream(torch.cuda.Stream() if graph else torch.cuda.current_stream()):
            sim.run(use_graph=graph)
        return sim
    parts, eager = run(True), run(False)
    for key, res in eager.results.items():
        if key != 'variant':
            assert np.array_equal(res.values, parts.results[key].values, equal_nan=True), key
    assert eager.results['cum_reinfections'].values[-1] > 0
