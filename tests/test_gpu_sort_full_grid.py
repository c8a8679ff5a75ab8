"""The radix sort over a grid of more than 256 blocks that nearly all hold keys (32 groups of
blocks, bases from every group), at one, two and three passes: the merged gradient of a batch
of over a million keys against the FP64 oracle, within the parity tests' bars."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N
from tests.problems import make_problem, oracle_step

pytestmark = pytest.mark.gpu

S, K, FMAX, B, D = 10, 5, 60, 3300, 8


def case(vocab):
    prob = make_problem(seed=19, n=1500, V=1500, D=D, fmax=FMAX, avg_deg=14, zipf=0.8)
    # the ids spread over the vocabulary, both ends included
    prob.f_ids = (prob.f_ids.astype(np.int64) * (vocab - 1) // (prob.V - 1)).astype(np.uint32)
    prob.V = vocab
    prob.table = np.random.default_rng(1).uniform(-1, 1, size=(vocab, D)).astype(np.float32)
    anchors = np.random.default_rng(2).integers(0, prob.n, size=B).astype(np.uint32)
    return prob, anchors


@pytest.mark.parametrize("vocab", [1500, 1_000_000, 5_000_000])  # 11, 20 and 23 bits
def test_merged_gradient_matches_oracle(vocab):
    prob, anchors = case(vocab)
    assert B * FMAX * (1 + S + K) > 256 * 8192  # capacity of more than 256 blocks
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.gamma, cfg.valid_pct = D, B, K, 0.5, 0.0
    cfg.max_nodes_kind, cfg.max_nodes, cfg.grad_mode = N.EP_SAMPLE_FIXED, S, N.EP_GRAD_EXACT
    with N.Context(cfg) as ctx:
        ctx.set_graph(prob.indptr, prob.indices)
        ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
        ctx.set_table(prob.table)
        cnt, nbr, neg = ctx.sample_batch(anchors, 1)
        out = ctx.step_explicit(anchors, cnt, nbr, neg, 1, 0.01)
    lens = np.diff(prob.f_indptr.astype(np.int64))
    keys = lens[anchors].sum() + lens[neg].sum() + sum(lens[nbr[i, :c]].sum() for i, c in enumerate(cnt))
    assert keys > 1_400_000  # over 10 rounds of 256 keys for each of the 512 blocks
    res, merged, *_ = oracle_step(prob, anchors, cnt, nbr, neg, 0.5, 0.01, 1, "exact")
    want = np.array([r.loss if (r is not None and r.contributes) else 0.0 for r in res])
    assert np.max(np.abs(out["loss"] - want)) <= 1e-5 * np.max(want)
    assert np.array_equal(np.sort(out["feat"]), np.array(sorted(merged), np.uint32))
    g = np.stack([merged[int(f)] for f in out["feat"]])
    assert np.max(np.abs(out["grad"] - g)) <= 1e-5 * np.max(np.abs(g))
