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


# Rows of 100 and 256 values: less than a 1 MiB chunk, a chunk to the row, one row past the small
# ring of 2 chunks and past one of 8, either side of 12 MiB (helper threads), many rounds of the
# ring and a last partial chunk.
ROWS = [(100, 1), (100, 2621), (100, 2622), (100, 2 * 2621 + 1), (100, 8 * 2621 + 1), (256, 1024), (256, 8 * 1024), (256, 12 * 1024 - 1),
        (256, 12 * 1024), (256, 12 * 1024 + 1), (256, 40_007)]


@pytest.mark.parametrize("dims,rows", ROWS)
def test_master_rows_and_moments_read_back(dims, rows):
    """Tables and moments that lie in one record per row."""
    rng = np.random.default_rng(dims + rows)
    table = rng.standard_normal((rows, dims), dtype=np.float32)
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.precision = dims, 32, 2, N.EP_PREC_BF16_MASTER
    cfg.max_nodes_kind, cfg.max_nodes = N.EP_SAMPLE_FIXED, 2
    nodes = 64
    with N.Context(cfg) as ctx:
        ctx.set_graph(np.arange(nodes + 1, dtype=np.uint64), np.roll(np.arange(nodes, dtype=np.uint32), 1))
        # features at both ends of the table and between
        ids = np.linspace(0, rows - 1, nodes).astype(np.uint32)
        ctx.set_features(np.arange(nodes + 1, dtype=np.uint64), ids, rows)
        ctx.set_table(table)
        assert np.array_equal(ctx.get_table(), table)
        anchors = np.arange(32, dtype=np.uint32)
        out = ctx.step_explicit(anchors, *ctx.sample_batch(anchors, 1), 1, 0.01)
        m, v = ctx.get_adam()
        after = ctx.get_table()
    g = np.zeros_like(m)
    g[out["feat"]] = out["grad"]
    b1, b2 = np.float32(1.0) - np.float32(0.9), np.float32(1.0) - np.float32(0.999)
    # one FP32 product for m, two for v: 2 and 3 roundings of 2^-24
    assert np.all(np.abs(m - b1.astype(np.float64) * g) <= 2 * 2.0**-24 * np.abs(m))
    assert np.all(np.abs(v - b2.astype(np.float64) * g.astype(np.float64) ** 2) <= 3 * 2.0**-24 * np.abs(v) + 1e-44)
    still = ~g.any(axis=1)
    assert np.array_equal(after[still], table[still])
    assert rows < 3 or np.any(after != table)


@pytest.mark.parametrize("rows", [12 * 2048 - 1, 12 * 2048, 12 * 2048 + 1, 12 * 2048 + 2047])
def test_results_around_the_ring_bound(rows):
    """FP32 tables and node embeddings of 128 values either side of 12 MiB."""
    ctx, table = open_table(rows)
    with ctx:
        assert np.array_equal(ctx.get_table(), table)
        ip = np.arange(rows + 1, dtype=np.uint64)
        ids = np.random.default_rng(1).permutation(rows).astype(np.uint32)
        assert np.array_equal(ctx.embed_averaged(ip, ids), table[ids])  # one feature a node: its row


def test_a_small_ring_grows():
    """A small read of rows, a large result, the small read again."""
    rows, nodes = 3000, 30_000
    table = np.random.default_rng(4).standard_normal((rows, 128), dtype=np.float32)
    cfg = N.default_config()
    cfg.dims, cfg.precision = 128, N.EP_PREC_BF16_MASTER
    with N.Context(cfg) as ctx:
        ctx.set_features(np.array([0, 1], np.uint64), np.array([0], np.uint32), rows)
        ctx.set_table(table)
        assert np.array_equal(ctx.get_table(), table)
        bf16 = (ctx.get_table_bf16().astype(np.uint32) << 16).view(np.float32)
        ids = np.random.default_rng(5).integers(0, rows, size=nodes).astype(np.uint32)
        assert np.array_equal(ctx.embed_averaged(np.arange(nodes + 1, dtype=np.uint64), ids), bf16[ids])
        assert np.array_equal(ctx.get_table(), table)


@pytest.mark.parametrize("prec", [N.EP_PREC_FP32, N.EP_PREC_BF16, N.EP_PREC_BF16_MASTER])
def test_two_readers_of_one_context(prec):
    """One of them has the ring; the other takes the runtime's copy or waits for its turn."""
    rows = 70_001
    table = np.random.default_rng(3).standard_normal((rows, 128), dtype=np.float32)
    cfg = N.default_config()
    cfg.dims, cfg.precision = 128, prec
    with N.Context(cfg) as ctx:
        ctx.set_features(np.array([0, 1], np.uint64), np.array([0], np.uint32), rows)
        ctx.set_table(table)
        want = table
        if prec == N.EP_PREC_BF16:
            want = (ctx.get_table_bf16().astype(np.uint32) << 16).view(np.float32)
        good = [0, 0]

        def read(k):
            for _ in range(6):
                m, v = ctx.get_adam()
                good[k] += np.array_equal(ctx.get_table(), want) and not m.any() and not v.any()

        threads = [threading.Thread(target=read, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert good == [6, 6]


@pytest.mark.parametrize("prec", [N.EP_PREC_FP32, N.EP_PREC_BF16, N.EP_PREC_BF16_MASTER])
def test_reads_take_no_device_memory(prec):
    rows = 500_000
    cfg = N.default_config()
    cfg.dims, cfg.precision = 128, prec
    with N.Context(cfg) as ctx:
        ctx.set_features(np.array([0, 1], np.uint64), np.array([0], np.uint32), rows)
        ctx.set_table(None)
        torch.cuda.synchronize()
        free, done = [torch.cuda.mem_get_info(0)[0]], threading.Event()

        def watch():
            while not done.is_set():
                free.append(torch.cuda.mem_get_info(0)[0])

        w = threading.Thread(target=watch)
        w.start()
        try:
            table, (m, v) = ctx.get_table(), ctx.get_adam()
        finally:
            done.set()
            w.join()
    assert table.any() and not m.any() and not v.any()
    assert len(free) > 5 and free[0] - min(free) < 1 << 20
