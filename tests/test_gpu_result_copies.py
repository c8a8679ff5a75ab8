"""Large results on their way to the caller's array: into ordinary memory they go through a
pinned ring that a few helper threads empty, into page-locked memory (which the copy engine
writes itself) they go without either."""
import os
import threading

import numpy as np
import pytest
import torch

from cloverleaf_amd import _native as N

pytestmark = pytest.mark.gpu


def threads_during(call):
    """The call's result, and the threads that the process gained at most while it ran."""
    before, most, done = len(os.listdir("/proc/self/task")) + 1, 0, threading.Event()

    def watch():
        nonlocal most
        while not done.is_set():
            most = max(most, len(os.listdir("/proc/self/task")))

    w = threading.Thread(target=watch)
    w.start()
    try:
        out = call()
    finally:
        done.set()
        w.join()
    return out, most - before


def open_table(rows, dims=128):
    table = np.random.default_rng(rows).standard_normal((rows, dims), dtype=np.float32)
    cfg = N.default_config()
    cfg.dims = dims
    ctx = N.Context(cfg)
    ctx.set_features(np.array([0, 1], np.uint64), np.array([0], np.uint32), rows)
    ctx.set_table(table)
    return ctx, table


@pytest.mark.parametrize("locked", [False, True])
def test_page_locked_results_take_no_threads(locked):
    ctx, table = open_table(1_000_000)
    with ctx:
        host = torch.empty(table.shape, dtype=torch.float32, pin_memory=locked)
        out = host.numpy()

        def read():
            return N.load().ep_get_table(ctx.handle, N.ptr(out, N.c_float))

        assert read() == 0  # the runtime's own threads are there from here on
        out[:] = 0
        rc, gained = threads_during(read)
        assert rc == 0 and np.array_equal(out, table)
        assert gained == 0 if locked else gained >= 1
