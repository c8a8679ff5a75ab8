"""Attention blocks at the edges of the 32-item score tiles: nodes of exactly 2, 31, 32, 33, 63
and 64 distinct features, in the step (loss, constructions, merged gradient) and in inference,
against the FP64 oracle.  The probabilities of a tile are turned over through the LDS for the
key side (column sums, dK): one tile, one full tile, a second tile of one item, two full tiles,
and d_k below the tile's 32 columns.  Bars as in test_gpu_attention: FP32 arithmetic on the
rows the kernels read, 1e-5 of the largest value."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N
from oracle import ep_oracle as O
from tests.problems import Problem, dense_grad, make_problem, oracle_step
from tests.test_gpu_attention import TOL, att_ctx, rel

pytestmark = pytest.mark.gpu


def tile_problem(items, heads, dk, dm, bf16):
    p = make_problem(seed=items + dk, n=40, V=100, D=heads * (2 * dk + dm), fmax=2, avg_deg=6, table_scale=0.6)
    rng = np.random.default_rng(items)
    ids = np.concatenate([rng.choice(p.V, size=items, replace=False) for _ in range(p.n)]).astype(np.uint32)
    table = p.table
    if bf16:
        u = table.view(np.uint32)
        table = ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).view(np.float32)
    return Problem(p.indptr, p.indices, (np.arange(p.n + 1) * items).astype(np.uint64), ids, p.V, p.D, table)


@pytest.mark.parametrize("heads,dk,dm,window", [(4, 32, 128, 0), (2, 16, 32, 0), (2, 32, 64, 5)])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("items", [2, 31, 32, 33, 63, 64])
def test_step_and_embedding_at_tile_edges(items, bf16, heads, dk, dm, window):
    prob = tile_problem(items, heads, dk, dm, bf16)
    ctx = att_ctx(prob, heads, dk, dm, S=3, K=3, B=10, window=window,
                  precision=N.EP_PREC_BF16 if bf16 else N.EP_PREC_FP32)
    att = (heads, dk, window) if window else (heads, dk)
    emb = ctx.embed_attention(prob.f_indptr, prob.f_ids)
    for i in range(0, prob.n, 5):
        ref = O.attention_embed(prob.table, prob.f_ids[i * items:(i + 1) * items], heads, dk, window or None)
        assert rel(emb[i], ref) <= TOL
    anchors = np.arange(0, 40, 4, dtype=np.uint32)
    samples = ctx.sample_batch(anchors, 1)
    out = ctx.step_explicit(anchors, *samples, pass_=1, lr=0.01, apply_update=False, want_cons=True)
    res, merged, *_ = oracle_step(prob, anchors, *samples, 0.5, 0.01, 1, "first_leaf", attention=att)
    assert sum(r is not None and r.contributes for r in res) >= 5
    for i, r in enumerate(res):
        if r is not None:
            assert rel(out["cons"][i], np.stack(r.vectors)) <= TOL
    want = dense_grad(merged, prob.V, prob.D)
    got = np.zeros_like(want)
    assert set(out["feat"].tolist()) == set(merged.keys())
    got[out["feat"]] = out["grad"]
    assert rel(got, want) <= TOL
    ctx.close()
