"""The radix sort's scatter blocks add up their digit bases from the totals of groups of
blocks: 16 groups of up to 16 blocks (steps of up to 2M keys at capacity) and 32 larger
groups, at every digit width class: one pass (up to 11 bits), two passes of 8 to 11 bits,
three passes.  The same batch on contexts of either capacity updates the table, moments and
loss alike, bit for bit, and the merged gradient matches the FP64 oracle's feature set."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N
from tests.problems import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [2, 1500, 60_000, 1_000_000, 3_000_000, 5_000_000])
def test_group_bases_equal_scan_bases(vocab):
    base = make_problem(seed=9, n=700, V=min(vocab, 2000), D=8, fmax=10, zipf=0.8)
    # spread the ids over the vocabulary, both ends included
    ids = (base.f_ids.astype(np.int64) * (vocab - 1) // max(min(vocab, 2000) - 1, 1)).astype(np.uint32)
    table = np.random.default_rng(1).uniform(-1, 1, size=(vocab, 8)).astype(np.float32)
    anchors = np.random.default_rng(2).permutation(700)[:400].astype(np.uint32)
    got, samples = [], None
    for capacity in (400, 120_000):
        cfg = N.default_config()
        cfg.dims, cfg.batch_size, cfg.negatives, cfg.gamma, cfg.valid_pct = 8, capacity, 5, 0.5, 0.0
        cfg.max_nodes_kind, cfg.max_nodes = N.EP_SAMPLE_FIXED, 6
        with N.Context(cfg) as ctx:
            ctx.set_graph(base.indptr, base.indices)
            ctx.set_features(base.f_indptr, ids, vocab)
            ctx.set_table(table)
            samples = samples or ctx.sample_batch(anchors, 1)
            out = ctx.step_explicit(anchors, *samples, 1, 0.01)
            order = np.argsort(out["feat"])
            m, v = ctx.get_adam()
            got.append([out["loss"], out["feat"][order], out["grad"][order], ctx.get_table(), m, v])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    feats = got[0][1]
    assert len(np.unique(feats)) == len(feats) and np.isin(feats, ids).all()
    assert (vocab == 2) or len(feats) > 200
