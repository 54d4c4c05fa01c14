"""The step's neighbourhood windows on grids of every width modulo 4, with areas that end on
the last row or past it, against the CPU oracle after every hour (exact)."""
import numpy as np
import pytest

import epirust_amd as G
from oracle import epicpu as O
from tests.gpu_helpers import assert_agents_equal, interventions_config, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", [60, 61, 62, 63, 64, 65, 66, 67, 131])
def test_every_hour_on_grids_of_every_width(cfg1, g):
    n = g * g // 8
    say("[windows] %d agents on %d x %d" % (n, g, g))
    cfg = interventions_config(cfg1, n=n, g=g)
    cfg["disease"]["percentage_severe_infected_population"] = 0.9
    cfg["interventions"] = [{"BuildNewHospital": {"spread_rate_threshold": 5}}]
    gpu, cpu = G.Simulation(cfg), O.OracleSim(cfg)
    for h in range(1, 241):
        g_rows, _ = gpu.step(1)
        c_rows, stop = cpu.step(1)
        assert np.array_equal(g_rows, c_rows), "hour %d" % h
        if h <= 48 or h % 24 in (0, 1, 9, 18):
            assert_agents_equal(gpu.agents(), cpu.agents(), "hour %d" % h)
        if stop:
            break
    assert gpu.events() == cpu.events()
    gpu.close()
    cpu.close()
