"""The autotuner's choice (host logic; the timings are made up): tile shapes
are written only where they beat the bands that are picked without an entry."""
import json

import pytest

from cudaprotoplanetarydisks_amd import autotune, ensemble


class Batch:
    """Stands for an Ensemble: its substeps take `picked` until tile shapes are
    set, then what `tuned` gives for them."""
    n = 2

    def __init__(self, decks, tiles=None):
        self.shape = None

    def __enter__(self):
        return self

    def __exit__(self, *a):
        pass

    def set_tiles(self, k, rows, band):
        self.shape = (rows, band)

    def substep(self, t_end):
        Clock.now += Clock.picked if self.shape is None else Clock.tuned(*self.shape)


class Clock:
    now = 0.0

    @classmethod
    def perf_counter(cls):
        return cls.now


@pytest.fixture
def timings(monkeypatch):
    def make(picked, tuned):
        Clock.picked, Clock.tuned = picked, staticmethod(tuned)
        monkeypatch.setattr(autotune, "Ensemble", Batch)
        monkeypatch.setattr(autotune, "time", Clock)
    return make


def tune(path):
    assert autotune.main(["--grids", "128x384", "--out", str(path), "--steps", "3"]) == 0
    return json.loads(path.read_text())


def test_no_entry_where_the_picked_bands_are_faster(timings, tmp_path):
    timings(1e-3, lambda rows, band: 1.5e-3)
    path = tmp_path / "tiles.json"
    path.write_text(json.dumps({"128x384": {"src_rows": 8, "trad_band": 8}, "64x192": {"src_rows": 8, "trad_band": 16}}))
    assert tune(path) == {"64x192": {"src_rows": 8, "trad_band": 16}}


def test_entry_where_a_shape_is_faster(timings, tmp_path):
    timings(1e-3, lambda rows, band: 0.5e-3 if (rows, band) == (16, 32) else 2e-3)
    e = tune(tmp_path / "tiles.json")["128x384"]
    assert (e["src_rows"], e["trad_band"]) == (16, 32)
    assert e["ms_picked"] == pytest.approx(1.0) and e["ms_per_substep"] == pytest.approx(0.5)


def test_written_entries_are_read_back(timings, tmp_path):
    timings(1e-3, lambda rows, band: 1e-4 * rows + 1e-6 * band)
    entries = tune(tmp_path / "tiles.json")
    assert ensemble.load_tiles(str(tmp_path / "tiles.json")) == entries
    assert entries["128x384"]["src_rows"] == 8
