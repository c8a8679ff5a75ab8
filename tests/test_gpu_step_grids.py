"""The row kernels' grids and work units follow the step's key capacity.  The same explicit
batch runs on a context sized for it (a wave and a region per chunk of keys, regions dealt to
up to 16 units), on one sized for a far larger batch (the full grid) and on one large enough
for eight regions per wave (the region queue): table, moments and loss must agree bit for
bit, whatever the grid."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N
from tests.problems import make_problem

pytestmark = pytest.mark.gpu


def run(prob, dims, capacity, anchors, samples, steps, precision=N.EP_PREC_FP32):
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.gamma, cfg.precision = dims, capacity, 3, 0.5, precision
    cfg.max_nodes_kind, cfg.max_nodes, cfg.valid_pct = N.EP_SAMPLE_FIXED, 4, 0.0
    with N.Context(cfg) as ctx:
        ctx.set_graph(prob.indptr, prob.indices)
        ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
        ctx.set_table(prob.table)
        losses = [ctx.step_explicit(anchors, *samples, p + 1, 0.01)["loss"] for p in range(steps)]
        m, v = ctx.get_adam()
        return [np.concatenate(losses), ctx.get_table(), m, v]


# vocab 40: every row hot (medium and long rows); 3000: short rows only
@pytest.mark.parametrize("vocab", [40, 3000])
@pytest.mark.parametrize("dims", [8, 64, 100, 256])
@pytest.mark.parametrize("n", [1, 2, 65, 500])
def test_capacity_does_not_change_results(n, dims, vocab):
    prob = make_problem(seed=n + dims, n=600, V=vocab, D=dims, fmax=8, zipf=0.7)
    anchors = np.random.default_rng(n).permutation(600)[:n].astype(np.uint32)
    cfg = N.default_config()
    cfg.dims, cfg.negatives, cfg.max_nodes_kind, cfg.max_nodes = dims, 3, N.EP_SAMPLE_FIXED, 4
    with N.Context(cfg) as ctx:
        ctx.set_graph(prob.indptr, prob.indices)
        ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
        samples = ctx.sample_batch(anchors, 1)
    small = run(prob, dims, n, anchors, samples, 2)
    for capacity in (20_000, 270_000) if dims == 64 else (20_000,):
        large = run(prob, dims, capacity, anchors, samples, 2)
        for a, b in zip(small, large):
            assert np.array_equal(a, b), capacity
    assert np.isfinite(small[1]).all() and small[0].any()
