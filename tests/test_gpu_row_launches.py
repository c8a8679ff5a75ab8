"""Short rows, medium rows and pieces in one launch (an unnamed tile, steps of up to 2M keys)
against the separate kernels (the same tile, named): loss, merged gradient, tables and moments
bit for bit, at every width, precision and batch count, with rows of every kind: up to 32
entries, up to 128 (a medium row's batch runs straddle its lane 64), and more, in runs both
short and cut into pieces."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N
from tests.problems import make_problem

pytestmark = pytest.mark.gpu

FORMS = {"fp32": (N.EP_PREC_FP32, 0), "bf16": (N.EP_PREC_BF16, 0), "bf16-fp16": (N.EP_PREC_BF16, 1),
         "master": (N.EP_PREC_BF16_MASTER, 0), "master-fp16": (N.EP_PREC_BF16_MASTER, 1)}
S, K = 6, 4


def run(prob, form, concurrent, tile, anchors, samples):
    cfg = N.default_config()
    cfg.precision, cfg.fp16_adjoints = FORMS[form]
    cfg.dims, cfg.negatives, cfg.gamma, cfg.valid_pct = prob.D, K, 3.0, 0.0
    cfg.batch_size, cfg.concurrent_batches = len(anchors) // concurrent, concurrent
    cfg.max_nodes_kind, cfg.max_nodes, cfg.grad_mode = N.EP_SAMPLE_FIXED, S, N.EP_GRAD_EXACT
    cfg.seg_vpl, cfg.seg_unroll = tile
    with N.Context(cfg) as ctx:
        ctx.set_graph(prob.indptr, prob.indices)
        ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
        ctx.set_table(prob.table)
        got = []
        for p in range(2):
            samples = samples or ctx.sample_batch(anchors, 1)
            out = ctx.step_explicit(anchors, *samples, p + 1, 0.01)
            order = np.lexsort((out["grad"][:, 0], out["feat"]))
            got += [out["loss"], out["feat"][order], out["grad"][order]]
        got += [ctx.get_table(), *ctx.get_adam()]
        if form != "fp32":
            got.append(ctx.get_table_bf16())
        return samples, got


@pytest.mark.parametrize("concurrent", [1, 2, 8])
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("dims", [8, 16, 32, 64, 100, 128, 256])
def test_one_launch_equals_separate_kernels(dims, form, concurrent):
    prob = make_problem(seed=dims, n=500, V=1200, D=dims, fmax=8, zipf=1.0)
    anchors = np.random.default_rng(dims).permutation(500)[:400].astype(np.uint32)
    samples, one = run(prob, form, concurrent, (0, 0), anchors, None)
    _, separate = run(prob, form, concurrent, (4, 8), anchors, samples)
    # the rows' entries: occurrences of each feature over the examples' nodes
    cnt, nbr, neg = samples
    nodes = np.concatenate([anchors, neg.ravel(), *(nbr[i, :c] for i, c in enumerate(cnt))]).astype(np.int64)
    ip = prob.f_indptr.astype(np.int64)
    rows = np.bincount(np.concatenate([prob.f_ids[ip[u]:ip[u + 1]] for u in nodes]), minlength=prob.V)
    assert np.count_nonzero(one[0]) > 380  # nearly every example counts
    for lo, hi, least in ((1, 32, 100), (33, 64, 10), (65, 128, 10), (129, 10**6, 10)):
        assert np.count_nonzero((rows >= lo) & (rows <= hi)) >= least
    for a, b in zip(one, separate):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dims,form", [(64, "fp32"), (64, "master-fp16"), (256, "fp32"), (256, "bf16")])
def test_more_regions_than_waves(dims, form):
    """Several regions for some of the one launch's waves: between 5120 (its short-row waves)
    and 8192 regions of 64 keys."""
    prob = make_problem(seed=dims + 1, n=3000, V=30_000, D=dims, fmax=16, zipf=0.7)
    anchors = np.random.default_rng(3).integers(0, prob.n, size=4800).astype(np.uint32)
    samples, one = run(prob, form, 1, (0, 0), anchors, None)
    _, separate = run(prob, form, 1, (4, 8), anchors, samples)
    cnt, nbr, neg = samples
    lens = np.diff(prob.f_indptr.astype(np.int64))
    keys = lens[anchors].sum() + lens[neg].sum() + sum(lens[nbr[i, :c]].sum() for i, c in enumerate(cnt))
    assert 5200 * 64 < keys < 8192 * 64 and np.count_nonzero(one[0]) > 4700
    for a, b in zip(one, separate):
        assert np.array_equal(a, b)


def test_one_launch_is_no_slower_with_more_regions_than_waves():
    """0.45M keys: the row kernels' time of one launch against that of the separate ones.  With
    the regions past its waves taken from a queue its short rows took 134 us where they take 38 now."""
    prob = make_problem(seed=8, n=4800, V=3000, D=64, fmax=16, zipf=0.9)
    ms = []
    for tile in ((0, 0), (4, 8)):
        cfg = N.default_config()
        cfg.dims, cfg.batch_size, cfg.negatives, cfg.gamma, cfg.valid_pct = 64, 4800, K, 3.0, 0.0
        cfg.alpha = 1e-3  # the examples stay active
        cfg.max_nodes_kind, cfg.max_nodes, cfg.grad_mode = N.EP_SAMPLE_FIXED, S, N.EP_GRAD_EXACT
        cfg.seg_vpl, cfg.seg_unroll = tile
        with N.Context(cfg) as ctx:
            ctx.set_graph(prob.indptr, prob.indices)
            ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
            ctx.set_table(prob.table)
            runs = [ctx.bench_steps(2, 10, instrument=True) for _ in range(5)]
        ms.append(np.median([sum(r.ms_phase[5:8]) for r in runs]))
    print(f"one launch {ms[0]:.4f} ms, separate {ms[1]:.4f}", flush=True)
    assert ms[0] < 1.25 * ms[1]


def test_wide_fp16_tiles_keep_their_loads_in_flight():
    """FP16 adjoint rows of 256 with 16 values a lane, short rows alone, against 4 values.  With
    each row's load waited for inside its own branch they took 2.7 times as long."""
    prob = make_problem(seed=9, n=3000, V=200_000, D=256, fmax=32, zipf=0.5)
    ms = []
    for tile in ((4, 8), (16, 2)):
        cfg = N.default_config()
        cfg.precision, cfg.fp16_adjoints = N.EP_PREC_BF16, 1
        cfg.dims, cfg.batch_size, cfg.negatives, cfg.gamma, cfg.valid_pct = 256, 3000, K, 3.0, 0.0
        cfg.alpha = 1e-3
        cfg.max_nodes_kind, cfg.max_nodes, cfg.grad_mode = N.EP_SAMPLE_FIXED, S, N.EP_GRAD_EXACT
        cfg.seg_vpl, cfg.seg_unroll = tile
        with N.Context(cfg) as ctx:
            ctx.set_graph(prob.indptr, prob.indices)
            ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
            ctx.set_table(prob.table)
            ms.append(np.median([ctx.bench_steps(2, 10, instrument=True).ms_phase[5] for _ in range(5)]))
    print(f"4 values {ms[0]:.4f} ms, 16 values {ms[1]:.4f}", flush=True)
    assert ms[1] < 1.8 * ms[0]
