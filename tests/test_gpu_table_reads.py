"""Table and moment reads (ep_get_table, ep_get_adam) that stage on the device: tables larger
than one 64 MiB staging chunk with a ragged last chunk, widths whose rows are not a power of
two, tables on both sides of the BF16 widening threshold (2^23 values), and a few rows.
Every comparison is exact except the moments, which are held to the one product that makes
them from the merged gradient."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N
from tests.problems import make_problem

pytestmark = pytest.mark.gpu

# (dims, rows): 68 MB of FP32 rows (two chunks), 2^23 values less / more one row, one row
SIZES = [(100, 170_003), (256, 32_767), (256, 32_769), (8, 3), (64, 1)]


@pytest.mark.parametrize("dims,rows", SIZES)
@pytest.mark.parametrize("prec", [N.EP_PREC_FP32, N.EP_PREC_BF16, N.EP_PREC_BF16_MASTER])
def test_table_reads_back(dims, rows, prec):
    table = np.random.default_rng(dims + rows).standard_normal((rows, dims)).astype(np.float32)
    table[0, :3] = (np.inf, -0.0, np.nan)
    cfg = N.default_config()
    cfg.dims, cfg.precision = dims, prec
    with N.Context(cfg) as ctx:
        ctx.set_features(np.array([0, 1], np.uint64), np.array([0], np.uint32), rows)
        ctx.set_table(table)
        got = ctx.get_table()
        if prec == N.EP_PREC_BF16:  # the parameter is the rounded row
            want = (ctx.get_table_bf16().astype(np.uint32) << 16).view(np.float32)
        else:
            want = table
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        m, v = ctx.get_adam()
        assert not m.any() and not v.any()


@pytest.mark.parametrize("prec", [N.EP_PREC_FP32, N.EP_PREC_BF16_MASTER])
def test_moments_after_a_step(prec):
    prob = make_problem(seed=77, n=200, V=500, D=100, fmax=6)
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.precision = 100, 32, 3, prec
    cfg.max_nodes_kind, cfg.max_nodes = N.EP_SAMPLE_FIXED, 4
    with N.Context(cfg) as ctx:
        ctx.set_graph(prob.indptr, prob.indices)
        ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
        ctx.set_table(prob.table)
        anchors = np.arange(32, dtype=np.uint32)
        out = ctx.step_explicit(anchors, *ctx.sample_batch(anchors, 1), 1, 0.01)
        m, v = ctx.get_adam()
    g = np.zeros_like(m)
    g[out["feat"]] = out["grad"]
    b1, b2 = np.float32(1.0) - np.float32(0.9), np.float32(1.0) - np.float32(0.999)
    # one FP32 product for m, two for v: 2 and 3 roundings of 2^-24
    assert np.all(np.abs(m - b1.astype(np.float64) * g) <= 2 * 2.0**-24 * np.abs(m))
    assert np.all(np.abs(v - b2.astype(np.float64) * g.astype(np.float64) ** 2) <= 3 * 2.0**-24 * np.abs(v) + 1e-44)


def test_large_reads_from_two_threads():
    """Copies of 8 MiB and more go through a pinned ring and helper threads of their own."""
    import threading

    tables = [np.random.default_rng(k).standard_normal((150_001 + k, 64)).astype(np.float32) for k in range(2)]
    got = [[], []]

    def work(k):
        cfg = N.default_config()
        cfg.dims = 64
        with N.Context(cfg) as ctx:
            ctx.set_features(np.array([0, 1], np.uint64), np.array([0], np.uint32), len(tables[k]))
            ctx.set_table(tables[k])
            got[k] = [np.array_equal(ctx.get_table(), tables[k]) for _ in range(5)]

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got == [[True] * 5] * 2


@pytest.mark.parametrize("nodes", [32_767, 32_768, 40_000])  # either side of 8 MiB of output rows
def test_embedding_large_node_sets(nodes):
    rng = np.random.default_rng(nodes)
    table = rng.standard_normal((500, 64)).astype(np.float32)
    counts = rng.integers(0, 4, size=nodes)
    ip = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint64)
    ids = rng.integers(0, 500, size=int(ip[-1])).astype(np.uint32)
    cfg = N.default_config()
    cfg.dims = 64
    with N.Context(cfg) as ctx:
        ctx.set_features(np.array([0, 1], np.uint64), np.array([0], np.uint32), 500)
        ctx.set_table(table)
        out = ctx.embed_averaged(ip, ids)
        for bad in (0, 4095, 4096, len(ids) - 1):  # the id check's blocks of 4096
            wrong = ids.copy()
            wrong[bad] = 500
            with pytest.raises(N.NativeError, match="feature id out of range"):
                ctx.embed_averaged(ip, wrong)
    want = np.zeros((nodes, 64))
    np.add.at(want, np.repeat(np.arange(nodes), counts), table[ids].astype(np.float64))
    want[counts > 0] /= counts[counts > 0, None]
    # at most 3 rows added and one division: 3 roundings of 2^-24 of sums below 3 max |row|
    assert np.max(np.abs(out - want)) <= 4 * 3 * 2.0**-24 * np.abs(table).max()
