"""The population of every simulation of one batch, built together on the device, against the
CPU oracle (exact): sizes around the launch blocks, starting infections of every mix, among them
none, one kind only, and every agent."""
import copy

import pytest

import epirust_amd as G
from oracle import epicpu as O
from tests.gpu_helpers import assert_agents_equal, say

pytestmark = pytest.mark.gpu


def config(cfg1, n, exposed, asymptomatic, mild, severe, working=0.7, transport=0.2):
    cfg = copy.deepcopy(cfg1)
    cfg["population"]["Auto"].update(number_of_agents=n, working_percentage=working,
                                     public_transport_percentage=transport)
    cfg["geography_parameters"]["grid_size"] = max(60, int(2.5 * n ** 0.5))
    cfg["hours"] = 60
    cfg["starting_infections"] = {"exposed": exposed, "infected_mild_asymptomatic": asymptomatic,
                                  "infected_mild_symptomatic": mild, "infected_severe": severe}
    return cfg


MIX = [(1, 1, 0, 0, 0), (2, 0, 1, 0, 1), (255, 0, 0, 0, 0), (256, 3, 0, 0, 0), (257, 0, 4, 3, 2), (1023, 1, 1, 1, 1),
       (1025, 0, 0, 0, 9), (5000, 0, 0, 7, 0), (4097, 4097, 0, 0, 0), (3000, 1000, 900, 800, 300), (140000, 5, 0, 3, 2)]


def check(cfgs, seeds):
    batch = G.Batch(cfgs, seeds)
    for i, c in enumerate(cfgs):
        cpu = O.OracleSim(c, seed=seeds[i])
        assert_agents_equal(batch.agents(i), cpu.agents(), "run %d" % i)
        cpu.close()
    rows, _ = batch.step(26)
    for i, c in enumerate(cfgs):
        cpu = O.OracleSim(c, seed=seeds[i])
        ref, _ = cpu.step(26)
        assert (rows[i] == ref).all()
        assert_agents_equal(batch.agents(i), cpu.agents(), "run %d after a day" % i)
        cpu.close()
    batch.close()


def test_mixed_batch(cfg1):
    say("[init batch] %d populations" % len(MIX))
    check([config(cfg1, *m) for m in MIX], [11 + i for i in range(len(MIX))])


@pytest.mark.parametrize("working,transport", [(0.0, 0.0), (1.0, 1.0), (0.7, 0.0)])
def test_work_and_transport_extremes(cfg1, working, transport):
    say("[init batch] working %g transport %g" % (working, transport))
    check([config(cfg1, n, 2, 0, 1, 0, working, transport) for n in (300, 2500)], [5, 6])


@pytest.mark.parametrize("mix", MIX)
def test_alone(cfg1, mix):
    say("[init batch] alone %s" % (mix,))
    check([config(cfg1, *mix)], [77])
