"""Steps that exceed the capacity of their context: with every neighbour (or a share of them)
the step buffers are sized for distinct anchors, and a split that names a hub again and again
asks for more.  Such a step is refused (EP_ECAPACITY), updates nothing and leaves the buffers'
neighbours alone; other contexts go on."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N

pytestmark = pytest.mark.gpu

LEAVES, K = 400, 3


def learn(form, train, most):
    """Learns on a star graph (node 0 is the hub) where one node has `most` features and the
    others one; returns whether that was refused, left the table alone, and left it finite."""
    n = LEAVES + 1
    ip = np.concatenate([[0, LEAVES], LEAVES + np.arange(1, n)]).astype(np.uint64)
    ix = np.concatenate([np.arange(1, n), np.zeros(LEAVES)]).astype(np.uint32)
    counts = np.ones(n, np.int64)
    counts[5] = most
    fp = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint64)
    ids = (np.arange(int(fp[-1])) % 90).astype(np.uint32)
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.passes, cfg.valid_pct, cfg.alpha = 32, 64, K, 2, 0.0, 0.01
    cfg.grad_mode = N.EP_GRAD_EXACT
    if form == "atomic":
        cfg.scatter = N.EP_SCATTER_ATOMIC
    if form == "weighted":
        cfg.weighted_neighbor_averaging = 1
    if form == "probability":
        cfg.max_nodes_kind, cfg.max_nodes_p = N.EP_SAMPLE_PROBABILITY, 0.9
    table = np.random.default_rng(1).uniform(-1, 1, size=(90, 32)).astype(np.float32)
    with N.Context(cfg) as ctx:
        ctx.set_graph(ip, ix)
        if form == "weighted":
            deg = np.diff(ip.astype(np.int64))
            ctx.set_edge_weights(np.concatenate([np.arange(1, d + 1) / d for d in deg]).astype(np.float32))
        ctx.set_features(fp, ids, 90)
        ctx.set_table(table)
        ctx.set_split(train, train[:0])
        refused = False
        try:
            ctx.learn()
        except N.NativeError as e:
            assert "EP_ECAPACITY" in str(e)
            refused = True
        return refused, np.array_equal(ctx.get_table(), table), np.isfinite(ctx.get_table()).all()


HUB, ALL = np.zeros(64, np.uint32), np.arange(LEAVES + 1, dtype=np.uint32)


@pytest.mark.parametrize("form", ["sort", "atomic", "weighted", "probability"])
def test_too_many_keys(form):
    """Room for 400 + 63 + 64 (1 + K) keys; 64 hubs ask for 64 (400 + 1 + K), or 0.9 of it."""
    assert learn(form, HUB, 1) == (True, True, True)
    assert learn(form, ALL, 1) == (False, False, True)


def test_too_many_neighbour_rows():
    """Lists of up to 60 features leave room for all the keys, but not for the rows: 400 + 63 of
    them, 64 hubs ask for 64 * 400."""
    assert 60 * (LEAVES + 63 + 64 * (1 + K)) > 64 * (LEAVES + 1 + K + 59)
    assert learn("weighted", HUB, 60) == (True, True, True)
    assert learn("weighted", ALL, 60) == (False, False, True)
    assert learn("sort", HUB, 60) == (False, False, True)  # no rows of their own: it all fits
