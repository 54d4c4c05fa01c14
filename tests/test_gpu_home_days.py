"""Days whose office hours run on the home layout (most agents isolated by a lockdown) against
the CPU oracle (exact): the isolated, the essential workers that still commute, and, in a batch,
runs without a lockdown beside larger ones with one."""
import numpy as np
import pytest

import epirust_amd as G
from oracle import epicpu as O
from tests.gpu_helpers import assert_agents_equal, interventions_config, say

pytestmark = pytest.mark.gpu


def config(cfg1, n, g, lockdown_at, essential):
    cfg = interventions_config(cfg1, n=n, g=g)
    cfg["interventions"] = [{"Vaccinate": {"at_hour": 400, "percent": 0.2}}]
    if lockdown_at:
        cfg["interventions"].append({"Lockdown": {"at_number_of_infections": lockdown_at,
                                                  "essential_workers_population": essential}})
    return cfg


@pytest.mark.parametrize("essential", [0.0, 0.3, 0.6])
@pytest.mark.parametrize("calls", [(960,), (24, 7, 41, 888)])
def test_lockdown_days(cfg1, essential, calls):
    say("[home days] essential %g, calls of %s hours" % (essential, calls))
    cfg = config(cfg1, 6000, 190, 25, essential)
    gpu, cpu = G.Simulation(cfg), O.OracleSim(cfg)
    for k in calls:
        g_rows, g_stop = gpu.step(k)
        c_rows, c_stop = cpu.step(k)
        assert np.array_equal(g_rows, c_rows) and g_stop == c_stop
        assert_agents_equal(gpu.agents(), cpu.agents(), "a call of %d hours" % k)
    assert gpu.events() == cpu.events()
    assert any(kind == 1 for _, kind in gpu.events())  # the lockdown came
    gpu.close()
    cpu.close()


def test_runs_without_a_lockdown_in_such_a_batch(cfg1):
    say("[home days] batch")
    cfgs = [config(cfg1, 9000, 230, 20, 0.1), config(cfg1, 3000, 130, 0, 0), config(cfg1, 2500, 110, 100000, 0.1)]
    batch = G.Batch(cfgs, [7, 8, 9])
    rows, stopped = batch.step(600)
    for i, c in enumerate(cfgs):
        cpu = O.OracleSim(c, seed=7 + i)
        ref, stop = cpu.step(600)
        assert np.array_equal(rows[i], ref) and bool(stopped[i]) == bool(stop)
        assert_agents_equal(batch.agents(i), cpu.agents(), "run %d" % i)
        assert batch.events(i) == cpu.events()
        cpu.close()
    batch.close()


@pytest.mark.parametrize("hours", [5, 7, 8, 11, 15, 16, 24])
def test_small_handle_moves_to_the_office_layout_when_its_blocks_are_set(cfg1, hours):
    say("[home days] block size set after %d hours" % (24 + hours))
    cfg = interventions_config(cfg1, n=3500, g=150)
    gpu, cpu = G.Simulation(cfg), O.OracleSim(cfg)
    for k in (24 + hours, 2, 70):
        g_rows, _ = gpu.step(k)
        c_rows, _ = cpu.step(k)
        assert np.array_equal(g_rows, c_rows)
        gpu.set_office_block_size(128)
        assert_agents_equal(gpu.agents(), cpu.agents(), "a call of %d hours" % k)
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("n", [1, 64, 30000, 30001, 65535, 65536])
def test_both_sides_of_the_size_that_has_an_office_layout(cfg1, n):
    say("[home days] %d agents" % n)
    cfg = config(cfg1, n, max(60, int(2.2 * n ** 0.5)), 0, 0)
    cfg["starting_infections"] = {"exposed": min(n, 30), "infected_mild_asymptomatic": 0,
                                  "infected_mild_symptomatic": 0, "infected_severe": 0}
    gpu, cpu = G.Simulation(cfg), O.OracleSim(cfg)
    for k in (13, 30):
        g_rows, _ = gpu.step(k)
        c_rows, _ = cpu.step(k)
        assert np.array_equal(g_rows, c_rows)
        assert_agents_equal(gpu.agents(), cpu.agents(), "a call of %d hours" % k)
    gpu.close()
    cpu.close()
