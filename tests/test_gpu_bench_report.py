"""What ep_bench_steps reports about the row kernels: the segment tile in use and the phases."""
import numpy as np
import pytest

from cloverleaf_amd import _native as N
from tests.problems import make_problem

pytestmark = pytest.mark.gpu


def bench(dims, tile=(0, 0), batch=64, prec=N.EP_PREC_FP32, noise=0.0):
    prob = make_problem(seed=dims, n=300, V=700, D=dims, fmax=8)
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.precision, cfg.noise = dims, batch, 3, prec, noise
    cfg.max_nodes_kind, cfg.max_nodes, cfg.valid_pct = N.EP_SAMPLE_FIXED, 4, 0.0
    cfg.seg_vpl, cfg.seg_unroll = tile
    with N.Context(cfg) as ctx:
        ctx.set_graph(prob.indptr, prob.indices)
        ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
        ctx.set_table(prob.table)
        return ctx.bench_steps(2, 6, instrument=True)


@pytest.mark.parametrize("prec", [N.EP_PREC_FP32, N.EP_PREC_BF16])
@pytest.mark.parametrize("dims", [16, 64, 100, 128, 256])
def test_tile_of_small_steps(dims, prec):
    """Steps whose rows take one launch have one tile, whatever the width."""
    r = bench(dims, prec=prec)
    assert (r.seg_vpl, r.seg_unroll) == (4, 8)
    assert r.fwd_x in (1, 2) and r.unique_rows > 0


def test_tile_asked_for_by_name():
    r = bench(64, tile=(8, 4))
    assert (r.seg_vpl, r.seg_unroll) == (8, 4)


def test_phases_of_one_launch():
    """Short rows, medium rows and pieces in one launch: its time is the short rows' phase."""
    r = bench(64)
    assert r.ms_phase[5] > 0 and r.ms_phase[6] == 0 and r.ms_phase[7] > 0
    assert r.ms_scatter_avg == pytest.approx(sum(r.ms_phase[3:8]))


@pytest.mark.parametrize("kw", [dict(tile=(8, 4)), dict(noise=0.1), dict(batch=40_000)])
def test_phases_of_separate_kernels(kw):
    r = bench(64, **kw)
    assert r.ms_phase[5] > 0 and r.ms_phase[6] > 0 and r.ms_phase[7] > 0


def test_a_context_that_grows_tunes_the_tile():
    """Small steps first, then, on features with longer lists, steps of more than 2M keys at
    capacity: the same table as a context that starts there with the reported tile named."""
    small = make_problem(seed=4, n=300, V=900, D=64, fmax=2)
    large = make_problem(seed=5, n=300, V=900, D=64, fmax=40)
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.valid_pct = 64, 8192, 3, 0.0
    cfg.max_nodes_kind, cfg.max_nodes = N.EP_SAMPLE_FIXED, 4
    every = np.arange(small.n, dtype=np.uint32)
    with N.Context(cfg) as ctx:
        ctx.set_graph(small.indptr, small.indices)
        ctx.set_features(small.f_indptr, small.f_ids, small.V)
        assert ctx.bench_steps(1, 2, instrument=False).seg_vpl == 4
        ctx.set_features(large.f_indptr, large.f_ids, large.V)
        ctx.set_table(large.table)
        r = ctx.bench_steps(1, 40, instrument=False)
        assert r.seg_vpl in (4, 8, 16) and r.seg_unroll > 0
        ctx.set_table(large.table)
        ctx.set_split(every, every[:0])  # the steps above have shuffled theirs
        ctx.learn()
        got = ctx.get_table()
    cfg.seg_vpl, cfg.seg_unroll = r.seg_vpl, r.seg_unroll
    with N.Context(cfg) as ctx:
        ctx.set_graph(small.indptr, small.indices)
        ctx.set_features(large.f_indptr, large.f_ids, large.V)
        ctx.set_table(large.table)
        ctx.set_split(every, every[:0])  # the steps above have shuffled theirs
        ctx.learn()
        assert np.array_equal(ctx.get_table(), got)
