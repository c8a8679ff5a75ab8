"""A batch whose step buffers no GPU can hold is refused; the context then places buffers anew
for the batches that fit."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N
from tests.problems import make_problem

pytestmark = pytest.mark.gpu


def test_a_context_after_a_batch_too_large_for_the_device():
    prob = make_problem(seed=71, n=300, V=400, D=8, fmax=60)
    cfg = N.default_config()
    cfg.dims, cfg.attention_heads, cfg.attention_dk = 128, 4, 32  # rows of 768
    cfg.batch_size, cfg.negatives, cfg.passes, cfg.valid_pct, cfg.alpha = 32, 5, 2, 0.0, 0.01
    cfg.max_nodes_kind, cfg.max_nodes = N.EP_SAMPLE_FIXED, 20
    table = np.random.default_rng(2).uniform(-1, 1, size=(400, 768)).astype(np.float32)
    every = np.arange(prob.n, dtype=np.uint32)

    def learn(ctx):
        ctx.set_table(table)
        ctx.set_split(every, every[:0])
        ctx.learn()
        return ctx.get_table()

    with N.Context(cfg) as ctx:
        ctx.set_graph(prob.indptr, prob.indices)
        ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
        first = learn(ctx)
        # 300,000 anchors of up to 60 * 26 occurrences: 1.4 TB of gradient rows
        with pytest.raises(N.NativeError, match="EP_ENOMEM"):
            ctx.sample_batch(np.zeros(300_000, np.uint32), 1)
        assert np.array_equal(learn(ctx), first)
    assert not np.array_equal(first, table)
