"""The scan for the hospital's first vacant cell over many blocks: grown hospitals whose rows fill
from a few to dozens of them, against the CPU oracle every day (exact). A block takes 512 items,
the cells of a row that lie in one strip of the grid."""
import numpy as np
import pytest

import epirust_amd as G
from oracle import epicpu as O
from tests.gpu_helpers import assert_agents_equal, interventions_config, say

pytestmark = pytest.mark.gpu
BUILD_HOSPITAL = 3


def config(cfg1, n, g):
    """Many severe cases from the start, so that patients are admitted day after day once the
    hospital has grown on the first."""
    cfg = interventions_config(cfg1, n=n, g=g)
    cfg["hours"] = 24 * 30
    cfg["geography_parameters"]["hospital_beds_percentage"] = 0.0
    cfg["disease"]["percentage_severe_infected_population"] = 0.9
    cfg["starting_infections"] = {"exposed": n // 10, "infected_mild_asymptomatic": 0, "infected_mild_symptomatic": 0,
                                  "infected_severe": n // 10}
    cfg["interventions"] = [{"BuildNewHospital": {"spread_rate_threshold": 5}}]
    return cfg


def patients(agents, hospital):
    """Admitted agents in the hospital's cells; of a day's admissions one gets the first vacant cell."""
    x, y = np.asarray(agents["x"]), np.asarray(agents["y"])
    x0, y0, x1, y1 = hospital
    return int(((np.asarray(agents["flags"]) & 1 != 0) & (x >= x0) & (x <= x1) & (y >= y0) & (y <= y1)).sum())


# 2 x 301 items in 2 blocks; 5 x 1301 in 13; 11 x 3001 in 65
@pytest.mark.parametrize("n,g", [(6000, 300), (12000, 1300), (20000, 3000)])
def test_grown_hospital_of_many_scan_blocks(cfg1, n, g):
    say("[hospital blocks] %d agents on %d x %d" % (n, g, g))
    cfg = config(cfg1, n, g)
    gpu, cpu = G.Simulation(cfg), O.OracleSim(cfg)
    most = 0
    for day in range(1, 25):
        g_rows, g_stop = gpu.step(24)
        c_rows, c_stop = cpu.step(24)
        assert np.array_equal(g_rows, c_rows) and g_stop == c_stop, "day %d" % day
        agents = cpu.agents()
        assert_agents_equal(gpu.agents(), agents, "day %d" % day)
        most = max(most, patients(agents, cpu.geometry()[0][4]))
        if c_stop:
            break
    assert gpu.events() == cpu.events() and (24, BUILD_HOSPITAL) in gpu.events()
    assert most >= 3
    gpu.close()
    cpu.close()


def test_grown_hospitals_of_a_batch(cfg1):
    """The blocks of later simulations start after earlier ones' have published their cells."""
    sizes = [(6000, 300), (9000, 1300), (4000, 700), (12000, 2000)]
    say("[hospital blocks] batch of %s" % (sizes,))
    cfgs = [config(cfg1, n, g) for n, g in sizes]
    batch = G.Batch(cfgs, [3, 4, 5, 6])
    cpus = [O.OracleSim(c, seed=3 + i) for i, c in enumerate(cfgs)]
    for day in range(1, 25):
        rows, stopped = batch.step(24)
        for i, cpu in enumerate(cpus):
            ref, stop = cpu.step(24)
            assert np.array_equal(rows[i], ref) and bool(stopped[i]) == bool(stop)
            assert_agents_equal(batch.agents(i), cpu.agents(), "run %d, day %d" % (i, day))
    for i, cpu in enumerate(cpus):
        assert batch.events(i) == cpu.events() and (24, BUILD_HOSPITAL) in batch.events(i)
        cpu.close()
    batch.close()
