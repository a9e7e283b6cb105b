"""Performance cases: the work a user of covasim_amd has the GPU do, through its public entry points.

Five kinds of case:
  sim      one Sim, run from day 0 to the end (``Sim.run``): the transmission step, its transitions, imports,
           resampled contacts and, with ``trace``, testing, contact tracing and a change_beta schedule
  batch    many independent sims advanced together (``BatchSim.run`` and ``BatchSim.reduce``)
  relax    one calibration step: expected incidence and its gradient (``Relaxation.expected`` and backward)
  script   a whole program: the population built on the device, the Sim initialised and run, its results
  kernels  the reference's three numba kernels through their drop-ins (``utils.compute_*``)

A case is a dict of plain values. ``prepare`` makes what the program holds before the call, ``run`` is one pass
and returns everything it computed, ``exact`` the same in 64 bits by plain torch where that can be had.
"""

import math

import numpy as np
import torch

import covasim_amd as cv
from covasim_amd import _lib, popgen
from covasim_amd import utils as cvu
from covasim_amd.relax import Relaxation, log_incidence_loss

HYBRID_EDGES = 18.0        # stored contacts per agent of the hybrid population
HYBRID_COMMUNITY = 10.0    # of them in the community layer, the one resampled daily
RANDOM_EDGES = 10.0
STATE_ARRAYS = 30          # 4-byte arrays of agent state
PHILOX_OPS = 60            # integer operations of one 10-round draw of four words


def listed():
    return [
        # the reference's default sim: 20k agents, one random layer held for the whole run, waning immunity;
        # what a notebook or a calibration loop runs most, bound by latency and launches
        dict(name='sim_random_20k', kind='sim', n=20_000, pop='random', days=60, waning=True, variants=0,
             dynamic=False, trace=False, graph=False, beta=0.016),
        # an ordinary city study: hybrid layers held, waning immunity, a second variant imported on day 30
        dict(name='sim_hybrid_100k', kind='sim', n=100_003, pop='hybrid', days=90, waning=True, variants=1,
             dynamic=False, trace=False, graph=False, beta=0.016),
        # a policy study: daily testing and tracing of every layer, beta reduced from day 30, contacts of the
        # community layer resampled daily, on a stream of its own (the run is then one captured graph)
        dict(name='sim_traced_300k', kind='sim', n=300_007, pop='hybrid', days=120, waning=False, variants=0,
             dynamic=True, trace=True, graph=True, beta=0.016),
        # the headline workload: 1M hybrid agents, community layer resampled daily, 180 days
        dict(name='sim_hybrid_1m', kind='sim', n=1_000_000, pop='hybrid', days=180, waning=False, variants=0,
             dynamic=True, trace=False, graph=False, beta=0.016),
        # a country: 10M hybrid agents, waning immunity, two variants, 120 days
        dict(name='sim_hybrid_10m', kind='sim', n=10_000_000, pop='hybrid', days=120, waning=True, variants=1,
             dynamic=True, trace=False, graph=False, beta=0.016),
        # a parameter sweep: 64 hybrid sims of 10k to 500k agents, beta 0.010 to 0.025, and their summary
        dict(name='batch_64', kind='batch', sims=64, lo=10_000, hi=500_000, days=120, dynamic=True),
        # one gradient of a calibration in double precision: a town, every layer held
        dict(name='relax_f64_30k', kind='relax', n=30_011, days=45, precision=64, dynamic=False),
        # one gradient of a calibration at scale: 1M agents, community layer in expectation, 60 days
        dict(name='relax_f32_1m', kind='relax', n=1_000_000, days=60, precision=32, dynamic=True),
        # a whole script, as most programs are: a new hybrid population, schools and work clipped from day 15 and
        # back on day 30, community layer resampled daily, 45 days
        dict(name='script_hybrid_500k', kind='script', n=500_009, pop='hybrid', days=45, waning=False, dynamic=True,
             clip=True, beta=0.02),
        # the drop-in kernels on host arrays, as the reference's own day loop calls them
        dict(name='kernels_host_20k', kind='kernels', n=20_000, edges=200_000, host=True, prevalence=0.03),
        # the drop-in kernels on device tensors at scale
        dict(name='kernels_1m', kind='kernels', n=1_000_000, edges=10_000_000, host=False, prevalence=0.05),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['sim', 'sim', 'sim', 'batch', 'relax', 'relax', 'script', 'kernels'])
    if kind == 'sim':
        pop = rng.choice(['random', 'hybrid', 'hybrid'])
        trace = rng.random() < 0.25
        n = _log_int(rng, 2_000, 1_000_000 if trace else 4_000_000)
        return dict(kind='sim', n=n, pop=pop, days=rng.randint(20, 180 if n < 2_000_000 else 90),
                    waning=rng.random() < 0.5, variants=rng.randint(0, 2), dynamic=rng.random() < 0.6, trace=trace,
                    graph=rng.random() < 0.3, beta=round(rng.uniform(0.010, 0.025), 4))
    if kind == 'batch':
        hi = _log_int(rng, 20_000, 500_000)
        return dict(kind='batch', sims=_log_int(rng, 4, 64), lo=2_000 + hi // 50, hi=hi, days=rng.randint(20, 120),
                    dynamic=rng.random() < 0.7)
    if kind == 'relax':
        precision = rng.choice([32, 32, 64])
        return dict(kind='relax', n=_log_int(rng, 5_000, 1_000_000 if precision == 32 else 300_000),
                    days=rng.randint(15, 75), precision=precision, dynamic=rng.random() < 0.5)
    if kind == 'script':
        pop = rng.choice(['random', 'hybrid', 'hybrid'])
        return dict(kind='script', n=_log_int(rng, 2_000, 3_000_000), pop=pop, days=rng.randint(20, 90),
                    waning=rng.random() < 0.5, dynamic=rng.random() < 0.6, clip=rng.random() < 0.5,
                    beta=round(rng.uniform(0.010, 0.025), 4))
    host = rng.random() < 0.4
    n = _log_int(rng, 2_000, 200_000 if host else 2_000_000)
    return dict(kind='kernels', n=n, edges=n * rng.randint(4, 15) + rng.randint(0, 63), host=host,
                prevalence=round(rng.uniform(0.001, 0.2), 4))


# ---------------------------------------------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------------------------------------------
def _population(n, pop, seed, edges):
    """A population built on the device; its resampled layer, if any, holds exactly ``edges`` contacts."""
    pars = cv.make_pars(pop_size=n, pop_type=pop, rand_seed=seed)
    pars['prognoses'] = cv.get_prognoses()
    people = popgen.make_population(pars, households='categorical' if pop == 'hybrid' else 'poisson')
    people['age'], people['sex'] = people['age'].cpu().numpy(), people['sex'].cpu().numpy()
    if edges:
        g = torch.Generator(device='cuda').manual_seed(seed % (1 << 62))
        ends = torch.randint(0, n, (2, edges), generator=g, device='cuda', dtype=torch.int32)
        people['contacts']['c' if pop == 'hybrid' else 'a'] = dict(p1=ends[0].clone(), p2=ends[1].clone(),
                                                                   beta=torch.ones(edges, device='cuda'))
    return people


def _community_edges(n, pop):
    return int(n * (HYBRID_COMMUNITY if pop == 'hybrid' else RANDOM_EDGES)) + n % 7


def _make_sim(n, pop, days, seed, beta, waning, dynamic, variants=0, trace=False, log_capacity=None):
    layer = 'c' if pop == 'hybrid' else 'a'
    variants = [cv.variant(dict(rel_beta=1.7 + 0.2 * k), days=[min(30 + 10 * k, days)], n_imports=100)
                for k in range(variants)]
    interventions = []
    if trace:
        probs = dict(h=1.0, s=0.5, w=0.5, c=0.1) if pop == 'hybrid' else dict(a=0.4)
        times = dict(h=0, s=1, w=1, c=2) if pop == 'hybrid' else dict(a=1)
        interventions = [cv.change_beta(min(30, days), 0.8),
                         cv.test_prob(symp_prob=0.1, asymp_prob=0.001, test_delay=1),
                         cv.contact_tracing(trace_probs=probs, trace_time=times)]
    sim = cv.Sim(pop_size=n, pop_type=pop, n_days=days, rand_seed=seed, beta=beta, use_waning=waning,
                 pop_infected=20, dynam_layer={layer: 1} if dynamic else {}, variants=variants,
                 interventions=interventions, log_capacity=log_capacity,
                 popdict=_population(n, pop, seed, _community_edges(n, pop) if dynamic else 0))
    return sim.initialize()


def _prepare_sim(case, seed):
    sim = _make_sim(case['n'], case['pop'], case['days'], 1 + seed, case['beta'], case['waning'], case['dynamic'],
                    case['variants'], case['trace'])
    live = list(sim.people._d.values()) + [v for k, v in sim._w.items() if k.startswith('diag_')]
    return dict(kind='sim', sim=sim, live=live, first=[v.clone() for v in live],
                stream=torch.cuda.Stream() if case['graph'] else None)


def _prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    sizes = rng.permutation(np.geomspace(case['lo'], case['hi'], case['sims']).astype(int))
    betas = rng.uniform(0.010, 0.025, case['sims'])
    sims = [_make_sim(int(sizes[i]), 'hybrid', case['days'], 1 + seed * 4096 + i, float(betas[i]), False,
                      case['dynamic'], log_capacity=1024) for i in range(case['sims'])]
    batch = cv.BatchSim(sims)
    return dict(kind='batch', batch=batch, first=batch.snapshot_state())


def _prepare_relax(case, seed):
    sim = _make_sim(case['n'], 'hybrid', case['days'], 1 + seed, 0.016, False, case['dynamic'], log_capacity=1024)
    relax = Relaxation(sim, precision=case['precision'], w_samples=5_000, w_seed=seed)
    rng = np.random.default_rng(seed)
    theta = torch.as_tensor(relax.theta0() * rng.uniform(0.8, 1.25, relax.n_params))
    day = np.arange(relax.n_days)
    observed = torch.as_tensor(20.0 * np.exp(0.12 * day) * rng.uniform(0.7, 1.4, relax.n_days))
    return dict(kind='relax', relax=relax, theta=theta, observed=observed)


def _prepare_script(case, seed):
    return dict(kind='script', case=case, seed=1 + seed)


def _kernel_inputs(case, seed):
    """Day 40 of an epidemic: dates of the infectious and recovered, factors, flags and one layer's contacts."""
    g = torch.Generator(device='cuda').manual_seed(seed)
    n, E = case['n'], case['edges']
    day = 40

    def uniform(m=n):
        return torch.rand(m, generator=g, device='cuda')

    u = uniform()
    inf = u < case['prevalence']
    past = (u >= case['prevalence']) & (u < 0.2 + case['prevalence'])
    sus = ~(inf | past)
    nan = torch.full((n,), float('nan'), device='cuda')
    length = (5 + 12 * uniform()).round()
    start = torch.where(inf, day - (length * uniform()).floor(), torch.where(past, day - 5 - length, nan))
    dead = past & (uniform() < 0.01)
    rel_trans = (-torch.log1p(-uniform()) * 0.6 * 100).floor() / 100  # most agents infect few, some infect many
    return dict(t=day, start=start, recovered=torch.where(dead, nan, start + length),
                dead=torch.where(dead, start + length, nan), rel_trans=rel_trans,
                rel_sus=torch.tensor([0.34, 0.67, 1.0, 1.24, 1.47], device='cuda')[(5 * uniform()).long().clamp(max=4)],
                inf=inf, sus=sus, symp=inf & (uniform() < 0.6), iso=inf & (uniform() < 0.1), quar=uniform() < 0.02,
                immunity=torch.where(past, 0.8 * uniform(), torch.zeros(n, device='cuda')),
                p1=(uniform(E) * n).to(torch.int32).clamp(max=n - 1), p2=(uniform(E) * n).to(torch.int32).clamp(max=n - 1),
                betas=torch.ones(E, device='cuda'))


def _prepare_kernels(case, seed):
    x = _kernel_inputs(case, seed)
    if case['host']:
        x = {k: v.cpu().numpy() if isinstance(v, torch.Tensor) else v for k, v in x.items()}
    record = np.empty((2, case['n']), np.int32) if case['host'] else torch.empty(2, case['n'], dtype=torch.int32,
                                                                                 device='cuda')
    return dict(kind='kernels', x=x, seed=1 + seed, record=record)


def prepare(case, seed):
    return {'sim': _prepare_sim, 'batch': _prepare_batch, 'relax': _prepare_relax, 'script': _prepare_script,
            'kernels': _prepare_kernels}[case['kind']](case, seed)


# ---------------------------------------------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------------------------------------------
def _tables(results):
    flat = {k: r for k, r in results.items() if k != 'variant'}
    return dict(rows=np.stack([flat[k].values for k in sorted(flat)]),
                variants=np.stack([results['variant'][k].values for k in sorted(results['variant'])]))


def _sim_again(state):
    """Puts a finished sim back to day 0 (the agents as they were initialised) and runs it."""
    sim = state['sim']
    torch._foreach_copy_(state['live'], state['first'])
    _lib.reset_workspace(sim._w)
    sim.t, sim.complete, sim.results_ready = 0, False, False
    sim.run()
    resampled = [lay for k, lay in sim.people.contacts.items() if sim['dynam_layer'].get(k)]
    return dict(_tables(sim.results), counts=sim._w['results'], sums=sim._w['results_f'], people=sim.people._d,
                resampled=[(lay.tensor('p1'), lay.tensor('p2')) for lay in resampled])


def _run_sim(state):
    if state['stream'] is None:
        return _sim_again(state)
    with torch.cuda.stream(state['stream']):
        return _sim_again(state)


def _run_batch(state):
    batch = state['batch']
    batch.restore_state(state['first'])
    batch.run()
    R = batch.reduce()
    flat = [R[k] for k in sorted(R) if k != 'variant']
    tables = [_tables(s.results) for s in batch.sims]
    return dict(rows=np.stack([t['rows'] for t in tables]), variants=np.stack([t['variants'] for t in tables]),
                middle=np.stack([r.values for r in flat]), low=np.stack([r.low for r in flat]),
                high=np.stack([r.high for r in flat]), people=batch._d,
                resampled=[(batch._layers[k]['p1'], batch._layers[k]['p2'])
                           for i, k in enumerate(batch.layer_keys) if batch.dynamic[i]])


def _run_relax(state):
    theta = state['theta'].clone().requires_grad_(True)
    expected = state['relax'].expected(theta)
    log_incidence_loss(expected, state['observed']).backward()
    return dict(expected=expected.detach(), grad=theta.grad)


def _run_script(state):
    case, hybrid = state['case'], state['case']['pop'] == 'hybrid'
    layer, closed = ('c', ['s', 'w']) if hybrid else ('a', ['a'])
    third = case['days'] // 3
    clip = [cv.clip_edges([third, 2 * third], [0.3, 1.0], layers=closed)] if case['clip'] else []
    sim = cv.Sim(pop_size=case['n'], pop_type=case['pop'], n_days=case['days'], rand_seed=state['seed'],
                 beta=case['beta'], use_waning=case['waning'], dynam_layer={layer: 1} if case['dynamic'] else {},
                 interventions=clip, popgen='device', households='categorical' if hybrid else 'poisson')
    sim.run()
    return dict(_tables(sim.results), counts=sim._w['results'], sums=sim._w['results_f'], people=sim.people._d)


VIRAL = dict(frac_time=0.3, load_ratio=2.0, high_cap=4.0)
FACTORS = dict(beta_layer=0.6, asymp_factor=0.8, iso_factor=0.1, quar_factor=0.2)


def _run_kernels(state):
    x = state['x']
    load = cvu.compute_viral_load(x['t'], x['start'], x['recovered'], x['dead'], **VIRAL)
    trans, sus = cvu.compute_trans_sus(x['rel_trans'], x['rel_sus'], x['inf'], x['sus'], FACTORS['beta_layer'], load,
                                       x['symp'], x['iso'], x['quar'], FACTORS['asymp_factor'], FACTORS['iso_factor'],
                                       FACTORS['quar_factor'], x['immunity'])
    cvu.set_seed(state['seed'])
    source, target = cvu.compute_infections(0.016, x['p1'], x['p2'], x['betas'], trans, sus, t=x['t'])
    return dict(load=load, trans=trans, sus=sus, pairs=_infected(state, source, target))


def _infected(state, source, target):
    """Source and target columns of the day's record, which has room for an infection of every agent."""
    record = state['record']
    record[...] = -1
    record[0, :len(source)] = source
    record[1, :len(target)] = target
    return record


def run(state):
    return {'sim': _run_sim, 'batch': _run_batch, 'relax': _run_relax, 'script': _run_script,
            'kernels': _run_kernels}[state['kind']](state)


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how close another correct one comes
# ---------------------------------------------------------------------------------------------------------------
def _day_loop_work(n, days, edges, dynamic_edges):
    """Agent state in and out once, the held contacts once, the resampled contacts out once, every agent's
    state word read and written on each day; one draw per two contacts of each resample."""
    return dict(bytes=n * 4 * STATE_ARRAYS * 2 + 8 * edges + 8 * days * n,
                flops=days * dynamic_edges / 2 * PHILOX_OPS + n * 20 * PHILOX_OPS)


def work(case):
    if case['kind'] in ('sim', 'script'):
        n, hybrid = case['n'], case['pop'] == 'hybrid'
        edges = n * (HYBRID_EDGES if hybrid else RANDOM_EDGES)
        dyn = (n * (HYBRID_COMMUNITY if hybrid else RANDOM_EDGES)) if case['dynamic'] else 0
        made = _day_loop_work(n, case['days'] + 1, edges, dyn)
        if case['kind'] == 'script':  # the population is made and written first
            made = dict(bytes=made['bytes'] + n * 29 + 12 * edges, flops=made['flops'] + (edges / 4 + 3 * n) * PHILOX_OPS)
        return made
    if case['kind'] == 'batch':
        mean = (case['hi'] - case['lo']) / math.log(case['hi'] / case['lo'])
        n = case['sims'] * mean
        return _day_loop_work(n, case['days'] + 1, n * HYBRID_EDGES, n * HYBRID_COMMUNITY if case['dynamic'] else 0)
    if case['kind'] == 'relax':
        n, word = case['n'], case['precision'] // 8
        slots = n * 2 * (HYBRID_EDGES - (HYBRID_COMMUNITY if case['dynamic'] else 0))
        # the contact lists once; every day's infections written and, by the adjoint, read with its own history
        return dict(bytes=4 * slots + 3 * word * case['days'] * n, flops=case['days'] * slots * 50)
    return dict(bytes=case['n'] * (16 + 29) + 12 * case['edges'], flops=case['n'] * 30 + case['edges'] * 10)


def tolerance(case):
    if case['kind'] == 'relax':
        # measured against 64 bits over the sizes drawn: up to 9e-7 in 32 bits, 8e-16 in 64
        return {'rel': 4e-6} if case['precision'] == 32 else {'rel': 1e-13}
    if case['kind'] in ('sim', 'batch', 'script'):
        # counts and agent state are fixed by the draws; means over agents are 64-bit sums in any order
        return {'rel': 1e-9}
    return 'exact'


# ---------------------------------------------------------------------------------------------------------------
# 64 bits
# ---------------------------------------------------------------------------------------------------------------
XMAX = 0.999999  # cap of a contact's transmission probability


def _exact_relax(case, seed):
    state = _prepare_relax(case, seed)
    relax, sim = state['relax'], state['relax'].sim
    n, days = relax.n, relax.n_days
    bins = torch.as_tensor(relax.bins_np, device='cuda').long()
    rel_trans = sim.people._d['rel_trans'].double()
    w = torch.as_tensor(relax.w, device='cuda')[bins]  # [n][lag]
    slots, contacts = list(relax.dyn_slots), []
    for k, key in enumerate(relax.layer_keys):
        p1, p2 = (sim.people.contacts[key].tensor(c).long() for c in ('p1', 'p2'))
        keep = p1 != p2
        contacts.append(None if slots[k] else (torch.cat([p1[keep], p2[keep]]), torch.cat([p2[keep], p1[keep]])))
    seed_frac = relax.seed_frac
    theta = state['theta'].to('cuda').requires_grad_(True)
    sig_bin = theta[1 + relax.n_layers:]
    sigma = sig_bin[bins]
    s = torch.full((n,), 1.0 - seed_frac, dtype=torch.float64, device='cuda')
    infected, expected = [], []
    for t in range(days):
        past = infected[max(0, t - (w.shape[1] - 1)):t]
        acc = torch.zeros(n, dtype=torch.float64, device='cuda')
        for d, row in enumerate(reversed(past), start=1):
            acc = acc + row * w[:, d]
        tr = rel_trans * acc
        L = torch.zeros(n, dtype=torch.float64, device='cuda')
        for k in range(relax.n_layers):
            rate = theta[0] * theta[1 + k]
            if contacts[k] is not None:
                src, tgt = contacts[k]
                L = L.index_add(0, tgt, torch.log1p(-(rate * sigma[tgt] * tr[src]).clamp(max=XMAX)))
            else:
                total = torch.stack([torch.log1p(-(rate * b * tr).clamp(max=XMAX)).sum() for b in sig_bin])
                own = torch.log1p(-(rate * sigma * tr).clamp(max=XMAX))
                L = L + slots[k] / n * (total[bins] - own)
        new = s * -torch.expm1(L)
        s = s * torch.exp(L)
        infected.append(new + seed_frac if t == 0 else new)
        expected.append(new.sum())
    expected = torch.stack(expected)
    observed = state['observed'].to('cuda')
    torch.mean((torch.log1p(expected[1:]) - torch.log1p(observed[1:])) ** 2).backward()
    return dict(expected=expected.detach().cpu(), grad=theta.grad.cpu())


def _exact_kernels(case, seed):
    x = {k: v.double() if isinstance(v, torch.Tensor) and v.is_floating_point() else v
         for k, v in _kernel_inputs(case, seed).items()}
    stop = torch.where(torch.isnan(x['dead']), x['recovered'], x['dead'])
    total = stop - x['start']
    frac, ratio, cap = VIRAL['frac_time'], VIRAL['load_ratio'], VIRAL['high_cap']
    point = torch.where(frac * total > cap, cap / total, torch.full_like(total, frac))
    early = ((x['t'] - x['start']) / total < point).double()
    load = (ratio * early + (1 - early)) / (1 + frac * (ratio - 1))
    inf, sus, symp, iso, quar = (x[k].double() for k in ('inf', 'sus', 'symp', 'iso', 'quar'))
    f_quar = (1 - quar) + quar * FACTORS['quar_factor']
    trans = (x['rel_trans'] * inf * f_quar * (symp + (1 - symp) * FACTORS['asymp_factor'])
             * ((1 - iso) + iso * FACTORS['iso_factor']) * FACTORS['beta_layer'] * load)
    return dict(load=load.cpu(), trans=trans.cpu(), sus=(x['rel_sus'] * sus * f_quar * (1 - x['immunity'])).cpu(),
                pairs=None)


def exact(case, seed):
    """Sims and batches are fixed by their draws: 64 bits have nothing to add there."""
    if case['kind'] == 'relax':
        slots = case['n'] * 2 * (HYBRID_EDGES - (HYBRID_COMMUNITY if case['dynamic'] else 0))
        return _exact_relax(case, seed) if slots * case['days'] <= 1.2e9 else None
    if case['kind'] == 'kernels':
        return _exact_kernels(case, seed)
    return None
