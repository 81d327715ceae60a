"""The learned engine's choice for a level (gz_selector_choose): the model's
choice within the trust band and the near-tie margin of a search's large
levels.  CPU only; bars: the rule's own edges, exact.
"""
import ctypes as C

import numpy as np
import pytest

PULL, PUSH = 1, 2


@pytest.fixture()
def choose(gz):
    lib = gz.lib
    fn = lib.gz_selector_choose
    fn.argtypes, fn.restype = [C.c_int, C.c_uint64, C.c_uint64, C.c_int, C.POINTER(C.c_float)], C.c_int
    lib.gz_selector_set_trust(C.c_double(gz.TRUST_ABOVE), C.c_double(gz.TRUST_BELOW))
    lib.gz_selector_set_tie(C.c_double(gz.TIE))

    def call(bfs, vote, threshold, pull_minus_push):
        """The choice of a model that predicts the push cheaper by that much (log times)."""
        y = np.array([pull_minus_push, 0.0], np.float32)
        return fn(bfs, vote, threshold, PULL if y[0] < y[1] else PUSH, y.ctypes.data_as(C.POINTER(C.c_float)))

    yield call
    lib.gz_selector_set_trust(C.c_double(gz.TRUST_ABOVE), C.c_double(gz.TRUST_BELOW))
    lib.gz_selector_set_tie(C.c_double(gz.TIE))


@pytest.mark.parametrize("threshold", [4000, 4003, 1 << 40])
def test_near_ties_of_searches_only(gz, choose, threshold):
    quarter = threshold // 4
    for vote in (quarter, threshold):
        assert choose(1, vote, threshold, 0.25) == 1  # a near tie: pull
        assert choose(1, vote, threshold, 0.5) == 0   # at the margin: the model's push
        assert choose(1, vote, threshold, 4.0) == 0
        assert choose(0, vote, threshold, 0.25) == 0  # CC: the model's push
    assert choose(1, quarter - 1, threshold, 0.25) == 0
    for bfs in (0, 1):
        assert choose(bfs, threshold + 1, threshold, 4.0) == 1      # above the band: pull
        assert choose(bfs, threshold // 32 - 1, threshold, -4.0) == 0  # below it: push
        assert choose(bfs, quarter, threshold, -0.25) == 1          # the model's pull


def test_margin_is_settable(gz, choose):
    gz.lib.gz_selector_set_tie(C.c_double(1.0))
    assert choose(1, 1000, 4000, 0.75) == 1 and choose(1, 1000, 4000, 1.0) == 0
    for off in (0.0, -1.0):
        gz.lib.gz_selector_set_tie(C.c_double(off))
        assert choose(1, 4000, 4000, 0.01) == 0
        assert choose(1, 4000, 4000, -0.01) == 1
    # without the band the margin still goes by the threshold
    gz.lib.gz_selector_set_trust(C.c_double(0.0), C.c_double(0.0))
    gz.lib.gz_selector_set_tie(C.c_double(gz.TIE))
    assert choose(1, 8000, 4000, 0.25) == 1 and choose(1, 8000, 4000, 0.75) == 0
    assert choose(1, 1, 4000, -0.25) == 1
