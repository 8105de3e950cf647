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
    def __init__(self, precision):
        self.handle, self.precision = Handle(), precision


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
