"""The launch shapes of the tuner, on a stand-in for a handle (no GPU)."""
import numpy as np
import pytest

from tbplas_amd import _lib, tune


class Handle:
    """What a handle keeps of a shape."""

    def __init__(self):
        self.state = {}

    def set_tuning(self, blocks, stage):
        self.state.update(blocks=blocks, stage=bool(stage))

    def set_blocking(self, enable=True, max_rows=0, terms=3):
        assert terms in (3, 4, 5)
        self.state.update(terms=terms if enable else 0, rows=max_rows, resident=False)

    def set_resident(self, enable=True):
        self.state["resident"] = bool(enable)


class Ham:
    def __init__(self, precision, n=1000):
        self.handle, self.precision, self.n = Handle(), precision, n


@pytest.mark.parametrize("precision", [_lib.TBG_FP64, _lib.TBG_FP32])
@pytest.mark.parametrize("K", [1, 8, 12, 64])
@pytest.mark.parametrize("batch", [False, True])
def test_the_untuned_shape_is_the_one_set(precision, K, batch):
    """Setting the returned shape again leaves the handle as apply did."""
    H = Ham(precision)
    shape = tune.apply([H, Ham(precision)] if batch else H, K, np.ones(5), enabled=False)
    assert H.handle.state["resident"]
    again = Handle()
    tune._set(again, shape)
    assert again.state == H.handle.state


@pytest.mark.parametrize("terms,state", [(1, (0, False)), (3, (3, False)), (5, (5, False)),
                                         (32, (5, True)), (36, (4, True))])
def test_shapes(terms, state):
    """32 alone is what saved shapes hold."""
    h = Handle()
    tune._set(h, (8, False, terms))
    assert (h.state["terms"], h.state["resident"]) == state
    assert (h.state["blocks"], h.state["stage"]) == (8, False)


@pytest.mark.parametrize("n,K,steps,resident", [
    (8000, 1, 64, False), (8000, 1, 99, False), (8000, 1, 100, True), (8000, 2, 64, False),
    (8000, 4, 40, True), (8000, 4, 39, False), (69999, 1, 1, False), (70000, 1, 1, True),
    (8000, 1, None, True), (2_000_000, 8, 1, True)])
@pytest.mark.parametrize("tuned", [False, True])
def test_few_steps_on_a_small_sample_take_tile_passes(n, K, steps, resident, tuned, monkeypatch):
    """The tables of resident passes take longer than such a run gains, with
    a shape from the tuner as well; a batch counts as a whole."""
    monkeypatch.setattr(tune, "autotune", lambda H, K, bes: ((8, True, tune.RESIDENT), None))
    for hams in (Ham(_lib.TBG_FP64, n), [Ham(_lib.TBG_FP64, n // 2), Ham(_lib.TBG_FP64, n - n // 2)]):
        H0 = hams[0] if isinstance(hams, list) else hams
        shape = tune.apply(hams, K, np.ones(5), tuned, steps)
        assert H0.handle.state["resident"] == resident
        assert H0.handle.state["terms"] == 5
        assert (shape[2] >= tune.RESIDENT) == resident


def test_a_shape_without_resident_passes_stays(monkeypatch):
    monkeypatch.setattr(tune, "autotune", lambda H, K, bes: ((8, True, 1), None))
    H = Ham(_lib.TBG_FP64)
    assert tune.apply(H, 1, np.ones(5), True, 3) == (8, True, 1)
    assert H.handle.state["terms"] == 0
