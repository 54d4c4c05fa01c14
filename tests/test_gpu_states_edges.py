"""The citizen-state formatter at the edges of its blocks (256 records, 16 blocks a group) and of
its numbers (ids and coordinates that gain a digit inside a block), byte for byte against
the records of epi_citizen_states formatted on the host."""
import copy

import pytest

import epirust_amd as G
from tests.gpu_helpers import say
from tests.test_zz_no_alloc import DeviceBuffer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,g", [(1, 60), (9, 60), (11, 60), (255, 60), (256, 60), (257, 60), (4096, 160), (4097, 160),
                                 (10001, 250), (100100, 1100), (1000300, 2001)])
@pytest.mark.parametrize("shift", [0, 1, 15])
def test_text_equals_the_records(cfg1, n, g, shift):
    say("[states] %d agents, text at +%d" % (n, shift))
    c = copy.deepcopy(cfg1)
    c["population"]["Auto"]["number_of_agents"] = n
    c["geography_parameters"]["grid_size"] = g
    c["starting_infections"]["exposed"] = min(n, 5)
    sim = G.Simulation(c)
    sim.step(20)
    _, rec = sim.citizen_states()
    want = b",".join(b'{"citizen_id":"%d","state":"%s","location":{"x":%d,"y":%d}}' %
                     (r["citizen_id"], r["state"], r["x"], r["y"]) for r in rec)
    room = n * 80 + 64
    text, length = DeviceBuffer(room), DeviceBuffer(8)
    text.write(b"\xa5" * room)
    rc = G.lib().epi_citizen_states_text_noalloc(sim._h, text.p.value + shift, room - 64, length.p)
    assert rc == 0, G.lib().epi_last_error()
    got = text.read(room)
    k = int.from_bytes(length.read(8), "little")
    assert k == len(want) and got[shift:shift + k] == want
    assert got[:shift] == b"\xa5" * shift and got[shift + k:shift + k + 16] == b"\xa5" * 16  # nothing around it
    sim.close()
    text.free()
    length.free()
