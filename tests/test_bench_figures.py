"""bench.py's figures of the row update from an instrumented run's phases."""
from types import SimpleNamespace

import pytest

import bench


def result(phases, **kw):
    return SimpleNamespace(ms_phase=phases, steps=4, unique_rows=4000, short_rows=2400, **kw)


def test_short_rows_with_a_phase_of_their_own():
    name, nbytes, ms = bench.update_figures(result([0.1, 1, 0, 1, 0.2, 0.5, 0.25, 0.125]), 64, 4)
    assert name == "k_seg_update" and ms == 0.5
    assert nbytes == 600 * 64 * (2 * 4 + 16)


def test_rows_in_one_launch():
    name, nbytes, ms = bench.update_figures(result([0.1, 1, 0, 1, 0.2, 0.5, 0.0, 0.125]), 64, 2, master=True)
    assert name == "k_rows + k_long_combine" and ms == pytest.approx(0.625)
    assert nbytes == 1000 * 64 * (2 + 24)
