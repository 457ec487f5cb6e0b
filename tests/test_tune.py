"""The tuning table (no GPU): entries set, read back, removed and cleared
through the C ABI; candidate shapes; JSON tables."""
import pytest

from tbfsolver_amd import tune as Tu
from tbfsolver_amd._lib import TbfgError


def test_table_round_trip():
    Tu.clear()
    assert Tu.get_entry("sweep", (256, 192, 256), "mixed") == (0, 0, 0)
    Tu.set_entry("sweep", (256, 192, 256), "mixed", (32, 16, 256))
    Tu.set_entry("op", (256, 192, 256), "fp64", (-1, 0, 0))
    assert Tu.get_entry("sweep", (256, 192, 256), "mixed") == (32, 16, 256)
    assert Tu.get_entry("sweep", (256, 192, 256), "fp64") == (0, 0, 0)        # precision is part of the key
    assert Tu.get_entry("sweep_edge", (256, 192, 256), "mixed") == (0, 0, 0)  # and the family
    assert Tu.get_entry("op", (256, 192, 256), "fp64") == (-1, 0, 0)
    Tu.set_entry("sweep", (256, 192, 256), "mixed", (0, 0, 0))                # removes
    assert Tu.get_entry("sweep", (256, 192, 256), "mixed") == (0, 0, 0)
    Tu.clear()
    assert Tu.get_entry("op", (256, 192, 256), "fp64") == (0, 0, 0)
    with pytest.raises(TbfgError):
        Tu.check(Tu.lib().tbfg_tune_set(7, Tu._i3((1, 1, 1)), 4, Tu._i3((1, 1, 1))))  # no such family


def test_candidates_tile_the_level():
    assert Tu.candidates("sweep", (256, 192, 256), "mixed") == Tu.SWEEP_F
    assert Tu.candidates("sweep", (96, 32, 96), "mixed") == []              # below the plane-march size
    assert Tu.candidates("sweep", (192, 96, 128), "mixed") == [(64, 8, 256), (32, 16, 256), (64, 16, 512),
                                                                (32, 8, 128)]
    assert (64, 4, 128) in Tu.candidates("sweep", (256, 192, 256), "fp64")
    ops = Tu.candidates("op", (96, 40, 64), "mixed")
    assert (-1, 0, 0) in ops and (128, 512, 0) not in ops and (32, 256, 0) in ops


def test_json_tables(tmp_path):
    Tu.clear()
    table = {"precision": "mixed", "entries": {"128,96,128": {"op": {"shape": [64, 512, 0], "ms": 1.0, "tried": {}},
                                                             "sweep": {"shape": [32, 16, 256], "ms": 1.0,
                                                                       "tried": {}}}}}
    p = str(tmp_path / "t.json")
    Tu.save(table, p)
    assert Tu.load(p) == table
    assert Tu.get_entry("op", (128, 96, 128), "mixed") == (64, 512, 0)
    assert Tu.get_entry("sweep", (128, 96, 128), "mixed") == (32, 16, 256)
    Tu.clear()


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("wins", [False, True], ids=["built-in", "shapes"])
def test_tuner_enters_what_beats_the_built_in_choice(monkeypatch, tmp_path, precision, wins):
    """With every shape 5 % slower than the built-in choice nothing is entered; with the 32-cell tiles 5 % faster
    they are, the operator's under the FP64 key that handles of every precision look up, also from a saved table."""
    dims = (192, 96, 128)
    monkeypatch.setattr(Tu, "_case", lambda d: (None, None, None))
    families = (("op", "fp64"), ("sweep", precision), ("sweep_edge", precision))

    def time_solves(*_):
        ms = 1.0
        for kind, key in families:
            shape = Tu.get_entry(kind, dims, key)
            if shape != Tu.BUILT_IN:
                ms += -0.05 if wins and shape[0] == 32 else 0.05
        return ms

    monkeypatch.setattr(Tu, "_time_solves", time_solves)
    Tu.clear()
    try:
        table = Tu.autotune([dims], precision)
        got = {kind: Tu.get_entry(kind, dims, key) for kind, key in families}
        assert set(table["entries"]["192,96,128"]) == {"op", "sweep", "sweep_edge"}
        for shape in got.values():
            assert (shape[0] == 32) if wins else shape == Tu.BUILT_IN
        path = str(tmp_path / "t.json")
        Tu.save(table, path)
        Tu.clear()
        Tu.load(path)
        assert {kind: Tu.get_entry(kind, dims, key) for kind, key in families} == got
    finally:
        Tu.clear()


def test_tuner_does_not_enter_noise(monkeypatch):
    """A shape ahead by less than 1 %, or by less than the built-in choice differs from itself, is noise."""
    dims = (192, 96, 128)
    monkeypatch.setattr(Tu, "_case", lambda d: (None, None, None))
    Tu.clear()
    try:
        for base, other in ((lambda n: 1.0, 0.995), (lambda n: 1.0 + 0.04 * (n % 2), 0.97)):
            calls = [0]

            def time_solves(*_):
                if all(Tu.get_entry(k, dims, p) == Tu.BUILT_IN for k in Tu.KINDS for p in ("mixed", "fp64")):
                    calls[0] += 1
                    return base(calls[0])
                return other

            monkeypatch.setattr(Tu, "_time_solves", time_solves)
            Tu.tune_instance(dims, "mixed")
            assert all(Tu.get_entry(k, dims, p) == Tu.BUILT_IN for k in Tu.KINDS for p in ("mixed", "fp64"))
    finally:
        Tu.clear()
