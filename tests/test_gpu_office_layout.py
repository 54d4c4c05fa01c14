"""Small populations on the office layout. A handle of at most 30,000 agents runs office hours on the
home layout until its block size is set, so the parity tests that are written for the office layout's
launches (its moves, the claim filter, slot -> id reads) run here once more with one set, as do those
of the lockdown's switch between the layouts. All against the CPU oracle (exact)."""
import numpy as np
import pytest

import epirust_amd as G
from oracle import epicpu as O
from tests.gpu_helpers import assert_agents_equal, say
from tests.test_gpu_day_groups import (test_calls_of_many_days, test_run_that_ends_in_the_night_of_a_batch,
                                       test_vaccinations_split_only_their_own_days)
from tests.test_gpu_home_days import (config, test_lockdown_days, test_runs_without_a_lockdown_in_such_a_batch)
from tests.test_gpu_parity import (test_batch_of_mixed_replicates_matches_single_runs, test_cfg1_every_hour_bit_exact,
                                   test_csv_population_bit_exact, test_hospital_growth_and_full_hospital,
                                   test_interventions_every_hour_bit_exact,
                                   test_night_launch_in_a_batch_with_sweeps,
                                   test_partial_days_match_day_graphs_and_plain_launches,
                                   test_quiet_hours_launch_with_a_vaccination_at_hour_of_day_1,
                                   test_sparse_offices_fill_blocks_to_the_filter_limit,
                                   test_sweeps_at_sleep_hours_and_at_the_last_hour,
                                   test_whole_run_with_day_graphs_matches,
                                   test_zero_transmission_closed_forms_through_gpu)
from tests.test_gpu_stream import (test_run_writes_the_stream_when_enabled, test_stream_lines_match_oracle_every_hour,
                                   test_stream_stops_with_the_simulation)
from tests.test_gpu_windows import test_every_hour_on_grids_of_every_width

pytestmark = pytest.mark.gpu
LOCKED, UNLOCKED = 1, 2


@pytest.fixture(autouse=True)
def office_layout(monkeypatch):
    """Every handle that a test opens gets the block size that builds its office layout."""
    for handle in (G.Simulation, G.Batch):
        def open_with_blocks(self, *args, _open=handle.__init__, **kwargs):
            _open(self, *args, **kwargs)
            self.set_block_size(256)
        monkeypatch.setattr(handle, "__init__", open_with_blocks)


def lockdown_hours(cfg, seed, hours):
    """The hours of the run's lockdown and of its end."""
    cpu = O.OracleSim(cfg, seed=seed)
    cpu.step(hours)
    events = cpu.events()
    cpu.close()
    return [h for h, kind in events if kind == LOCKED][0], [h for h, kind in events if kind == UNLOCKED][0]


# 31,000 agents have an office layout by themselves. The calls: whole days up to the lockdown and past
# it, office hours of an isolated day split, and one call over the end of the lockdown.
@pytest.mark.parametrize("n,essential", [(5000, 0.0), (9000, 0.2), (31000, 0.1)])
def test_layouts_switch_with_a_lockdown(cfg1, n, essential):
    cfg = config(cfg1, n, int(2.3 * n ** 0.5), n // 40, essential)
    cfg["starting_infections"]["exposed"] = n // 200
    cfg["hours"] = 1200
    locked, unlocked = lockdown_hours(cfg, 5, 1000)
    say("[office layout] %d agents, lockdown %d..%d" % (n, locked, unlocked))
    assert 24 * 9 <= locked <= unlocked - 24 * 6  # after the first days' graphs, for some days
    gpu, cpu = G.Simulation(cfg, seed=5), O.OracleSim(cfg, seed=5)
    h = 0
    for end in (locked - 24, locked + 24 * 4 + 11, locked + 24 * 4 + 14, unlocked + 24 * 8 + 5, 1000):
        g_rows, g_stop = gpu.step(end - h)
        c_rows, c_stop = cpu.step(end - h)
        assert np.array_equal(g_rows, c_rows) and g_stop == c_stop
        assert_agents_equal(gpu.agents(), cpu.agents(), "hour %d" % end)
        h = end
    assert gpu.events() == cpu.events()
    gpu.close()
    cpu.close()


def test_layouts_switch_with_the_lockdowns_of_a_batch(cfg1):
    """Most agents are isolated from the larger runs' lockdowns on, one run has none."""
    cfgs = [config(cfg1, 20000, 330, 500, 0.1), config(cfg1, 6000, 180, 0, 0), config(cfg1, 9000, 220, 300, 0.2)]
    for c in cfgs:
        c["starting_infections"]["exposed"] = c["population"]["Auto"]["number_of_agents"] // 200
        c["hours"] = 1000
    starts = [lockdown_hours(cfgs[i], 7 + i, 900)[0] for i in (0, 2)]
    say("[office layout] batch, lockdowns at %s" % starts)
    assert max(starts) <= 504 - 24 * 5
    batch, cpus = G.Batch(cfgs, [7, 8, 9]), [O.OracleSim(c, seed=7 + i) for i, c in enumerate(cfgs)]
    h = 0
    for end in (max(starts) + 24 * 2 + 13, max(starts) + 24 * 3, 800):
        rows, stopped = batch.step(end - h)
        for i, cpu in enumerate(cpus):
            ref, stop = cpu.step(end - h)
            assert np.array_equal(rows[i], ref) and bool(stopped[i]) == bool(stop)
            assert_agents_equal(batch.agents(i), cpu.agents(), "run %d hour %d" % (i, end))
        h = end
    for i, cpu in enumerate(cpus):
        assert batch.events(i) == cpu.events()
        cpu.close()
    batch.close()
