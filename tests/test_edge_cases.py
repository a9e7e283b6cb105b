"""Boundary cases of whole runs, the HIP path against the oracle (sim.py:558-685): no seed infections, zero days
(the seeds and day 0 only), a population without any contact, an empty static layer beside a daily-resampled
one, and a population of seven agents. Counts and every agent array are compared exactly, in graph and eager
runs."""

import numpy as np
import pytest

from tests.helpers import copy_pop, make_population

pytestmark = pytest.mark.gpu


def _case(name):
    if name == 'no_seeds':
        return make_population(n=2000, pop_type='hybrid'), dict(n_days=20, pop_infected=0, beta=0.05,
                                                                 pop_type='hybrid')
    if name == 'zero_days':
        return make_population(n=2000, pop_type='hybrid'), dict(n_days=0, beta=0.05, pop_type='hybrid')
    if name == 'no_contacts':
        pop = make_population(n=1500, pop_type='random', contacts={'a': 0})
        assert len(pop['contacts']['a']['p1']) == 0
        return pop, dict(n_days=25, beta=0.05, pop_type='random')
    if name == 'empty_static_layer':
        pop = make_population(n=2000, pop_type='hybrid')
        for c in ('p1', 'p2'):
            pop['contacts']['s'][c] = np.zeros(0, np.int32)
        pop['contacts']['s']['beta'] = np.zeros(0, np.float32)
        return pop, dict(n_days=30, beta=0.05, pop_type='hybrid', dynam_layer=dict(c=1))
    if name == 'seven_agents':
        return make_population(n=7, pop_type='random', contacts={'a': 4}), dict(n_days=15, beta=0.5,
                                                                               pop_type='random', pop_infected=2)
    raise KeyError(name)


@pytest.mark.parametrize('use_graph', [True, False])
@pytest.mark.parametrize('name', ['no_seeds', 'zero_days', 'no_contacts', 'empty_static_layer', 'seven_agents'])
def test_boundary_run_matches_oracle(gpu, name, use_graph):
    from tests.test_gpu_parity import assert_people_equal, assert_results_equal, run_pair
    print(f'boundary case {name} graph={use_graph}', flush=True)
    pop, pars = _case(name)
    n_days = pars.pop('n_days')
    sim, osim, ores = run_pair(copy_pop(pop), n_days=n_days, seed=3, use_graph=use_graph, **pars)
    assert len(sim.results['new_infections'].values) == n_days + 1
    assert_results_equal(sim, ores)
    assert_people_equal(sim, osim)
    if name in ('no_seeds', 'no_contacts'):
        assert sim.results['new_infections'].values.sum() == 0


@pytest.mark.parametrize('n,k', [(33, 1), (33, 33), (2000, 9), (2000, 65), (200_003, 130_000), (200_003, 200_003)])
def test_infection_counts_per_wave_match_oracle(gpu, n, k):
    """Seeds only: from one target in the whole run to every agent of a wave's words (more than its log stage
    holds); outcomes, counts and the log against the oracle."""
    from tests.test_gpu_parity import assert_people_equal, assert_results_equal, run_pair
    print(f'{k} seeds among {n}', flush=True)
    pop = make_population(n=n, pop_type='random', contacts={'a': 0})
    sim, osim, ores = run_pair(copy_pop(pop), n_days=1, seed=5, pop_type='random', use_waning=True, pop_infected=k)
    assert_results_equal(sim, ores)
    assert_people_equal(sim, osim)
    log = sim.infection_log()
    assert sorted(r['target'] for r in log) == sorted(tg for (_, tg, _, _, _) in osim.people.infection_log)
    assert len(log) == k and all(r['source'] is None and r['layer'] == 'seed_infection' for r in log)


@pytest.mark.parametrize('n', [255, 257, 511, 513, 262_143, 262_145])
def test_agent_pass_block_edges_match_oracle(gpu, n):
    """One agent per thread up to 2^18 agents, two above, with the infectious map of 512-agent words (not the bitmap)
    in LDS: half-written words, and reinfections on the days whose severity immunity is not stored."""
    from covasim_amd import _lib
    from tests.test_gpu_parity import assert_people_equal, assert_results_equal, run_pair
    print(f'{n} agents', flush=True)
    pop = make_population(n=n, pop_type='random')
    days = 60 if n < 1000 else 5
    _lib.check(_lib.lib().cvk_set_tuning(_lib.TUNE_EDGE_LDS, 0), 'tuning')
    try:
        sim, osim, ores = run_pair(copy_pop(pop), n_days=days, seed=3, pop_type='random', use_waning=True,
                                   pop_infected=n // 8, beta=0.05)
    finally:
        _lib.check(_lib.lib().cvk_set_tuning(_lib.TUNE_EDGE_LDS, 1), 'tuning')
    assert_results_equal(sim, ores)
    assert_people_equal(sim, osim)
