"""The launch-shape autotuner's choice from its timings (epirust_amd/autotune.py), and the committed table."""
from epirust_amd import autotune


def tune(monkeypatch, tmp_path, times):
    monkeypatch.setattr(autotune, "_time", lambda configs, seeds, hours, repeats, block, office: times[(block, office)])
    cfg = {"population": {"Auto": {"number_of_agents": 1000}}, "seed": 1}
    block, office, _ = autotune.tune([cfg], path=str(tmp_path / "t.json"), candidates=(256, 512), verbose=False)
    assert autotune.tuned_shape([cfg], str(tmp_path / "t.json")) == (block, office)
    return block, office


def test_an_office_size_of_its_own_has_to_gain_more_than_the_repeats_differ(monkeypatch, tmp_path):
    same = {(256, 256): [1.20, 1.21], (512, 512): [1.00, 1.01]}
    assert tune(monkeypatch, tmp_path, {**same, (512, 256): [0.995, 0.998]}) == (512, 512)
    assert tune(monkeypatch, tmp_path, {**same, (512, 256): [0.97, 1.02]}) == (512, 512)
    assert tune(monkeypatch, tmp_path, {**same, (512, 256): [0.97, 0.98]}) == (512, 256)


def test_the_table_was_measured_over_twenty_days():
    for key, entry in autotune.load_table().items():
        assert entry["hours"] >= 480, key
        ms, office = entry["ms_per_hour"], entry["office_ms_per_hour"]
        assert ms[str(entry["block"])] == min(ms.values()), key
        if entry["office_block"] != entry["block"]:
            assert office[str(entry["office_block"])] < office[str(entry["block"])], key
