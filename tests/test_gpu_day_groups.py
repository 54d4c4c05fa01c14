"""Hours of a day that run as one launch, decided day by day, and the sums of the per-block
counts, against the CPU oracle (exact)."""
import numpy as np
import pytest

import epirust_amd as G
from oracle import epicpu as O
from tests.gpu_helpers import assert_agents_equal, interventions_config, say

pytestmark = pytest.mark.gpu


def small(cfg1, vaccinate=(), hours=None, n=2000, g=120):
    cfg = interventions_config(cfg1, n=n, g=g)
    cfg["interventions"] = [{"Lockdown": {"at_number_of_infections": 30, "essential_workers_population": 0.3}}]
    cfg["interventions"] += [{"Vaccinate": {"at_hour": h, "percent": 0.2}} for h in vaccinate]
    if hours:
        cfg["hours"] = hours
    return cfg


# Hours of days 1 and 3 (24 d + 1 .. 24 d + 24) on both sides of each group's edges, others plain.
@pytest.mark.parametrize("hours", [(24, 96), (25, 97), (26, 101), (29, 102), (30, 95), (31, 79, 125)])
def test_vaccinations_split_only_their_own_days(cfg1, hours):
    say("[day groups] vaccinations at %s" % (hours,))
    cfg = small(cfg1, hours)
    gpu, cpu = G.Simulation(cfg), O.OracleSim(cfg)
    for k in (72, 72, 30):
        g_rows, _ = gpu.step(k)
        c_rows, _ = cpu.step(k)
        assert np.array_equal(g_rows, c_rows)
        assert_agents_equal(gpu.agents(), cpu.agents(), "after %d hours" % k)
    assert gpu.events() == cpu.events()
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("hours", [48, 49, 50, 53, 55, 56])
def test_run_that_ends_in_the_night_of_a_batch(cfg1, hours):
    """Run 0 ends at hour `hours` - 1 (hours of day 23, 0, 1, 4, 6, 7), run 1 has a vaccination
    the next night, run 2 neither."""
    say("[day groups] a run of %d hours" % hours)
    cfgs = [small(cfg1, hours=hours), small(cfg1, (74,), n=1500, g=110), small(cfg1, n=900, g=90)]
    batch = G.Batch(cfgs, [3, 4, 5])
    rows, stopped = batch.step(120)
    for i, c in enumerate(cfgs):
        cpu = O.OracleSim(c, seed=3 + i)
        ref, stop = cpu.step(120)
        assert np.array_equal(rows[i], ref) and bool(stopped[i]) == bool(stop)
        cpu.close()


# 64-agent blocks: the epilogue's 64 threads add four blocks each per pass.
@pytest.mark.parametrize("n", [64, 65, 63 * 64 + 1, 64 * 64 + 1, 255 * 64 + 63, 256 * 64 + 1, 513 * 64])
def test_counts_of_many_blocks(cfg1, n):
    say("[day groups] %d agents in blocks of 64" % n)
    cfg = small(cfg1, n=n, g=max(60, int(3 * n ** 0.5)))
    if n < 100:
        cfg["starting_infections"] = {"exposed": 3, "infected_mild_asymptomatic": 1, "infected_mild_symptomatic": 1,
                                      "infected_severe": 1}
    gpu, cpu = G.Simulation(cfg), O.OracleSim(cfg)
    gpu.set_block_size(64)
    g_rows, _ = gpu.step(33)
    c_rows, _ = cpu.step(33)
    assert np.array_equal(g_rows, c_rows)
    gpu.close()
    cpu.close()


# Graphs of one and of four days, runs that end inside one, and days of other groups between them.
@pytest.mark.parametrize("vaccinate", [(), (74,), (25, 221)])
@pytest.mark.parametrize("calls", [(95,), (96,), (97, 240), (24, 400)])
def test_calls_of_many_days(cfg1, vaccinate, calls):
    say("[day groups] calls of %s hours, vaccinations at %s" % (calls, vaccinate))
    cfg = small(cfg1, vaccinate, hours=420)
    gpu, cpu = G.Simulation(cfg), O.OracleSim(cfg)
    for k in calls:
        g_rows, g_stop = gpu.step(k)
        c_rows, c_stop = cpu.step(k)
        assert np.array_equal(g_rows, c_rows) and g_stop == c_stop
        assert_agents_equal(gpu.agents(), cpu.agents(), "a call of %d hours" % k)
    assert gpu.events() == cpu.events()
    gpu.close()
    cpu.close()
