"""The limit of ep_step_explicit_noalloc: a step whose arrays take up to 64 MiB runs, a larger
one is refused with its size.  The arrays' sizes are restated here, one line per array; the
sort's totals have a place of their own beside them and don't count."""
import re

import numpy as np
import pytest

from cloverleaf_amd import _native as N
from tests.problems import make_problem

pytestmark = pytest.mark.gpu

D, K, S, FMAX = 64, 5, 10, 8
LIMIT = 64 << 20


def needed(n):
    """Bytes of the arrays of an FP32 step of n anchors (Fixed(S) neighbours), in order."""
    nc, ent = K + 2, 1 + S + K
    keys = n * FMAX * ent
    long_cap, piece_cap = keys // 65 + 1, keys // 16 + 1
    sort_grid = min(2048, max(256, (keys // 8192 + 255) // 256 * 256))
    chunks, regions = (keys + 63) // 64, 2048 * 4
    assert chunks < 32 * regions
    per_region = (chunks + regions - 1) // regions
    sizes = [4 * n, 4 * n, 4 * n * S, 4 * n * K, 4 * n, 8 * n * ent, 4 * n * ent, 4 * (n + 1),  # anchors .. keyoff
             4 * n * nc * D, 4 * n * nc, n * nc, 4 * n]  # adj, coef, elig, loss
    sizes += [4 * keys] * 4 + [4 * 2048 * sort_grid]  # two key and slot buffers, block counts
    sizes += [4 * long_cap] * 3 + [4 * 8 * long_cap] * 2
    sizes += [16 * regions * per_region * 64, 8 * regions * per_region * 2, 4 * regions, 4 * regions]
    sizes += [4 * piece_cap, 4 * piece_cap, 4 * piece_cap * D]
    at = 0
    for x in sizes:
        at = (at + 255) // 256 * 256 + max(x, 16)
    return at


@pytest.fixture(scope="module")
def prob():
    p = make_problem(seed=52, n=4000, V=900, D=D, avg_deg=12, fmax=FMAX, zipf=0.9)
    assert np.diff(p.f_indptr.astype(np.int64)).max() == FMAX
    return p


def open_ctx(prob):
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.gamma, cfg.valid_pct = D, 64, K, 0.5, 0.0
    cfg.max_nodes_kind, cfg.max_nodes = N.EP_SAMPLE_FIXED, S
    ctx = N.Context(cfg)
    ctx.set_graph(prob.indptr, prob.indices)
    ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
    ctx.set_table(prob.table)
    return ctx


def refuse(ctx, n):
    z = np.zeros(n, np.uint32)
    with pytest.raises(N.NativeError, match="EP_ECAPACITY") as e:
        ctx.step_explicit_noalloc(z, z, np.zeros((n, S), np.uint32), np.zeros((n, K), np.uint32), 1, 0.01)
    return int(re.search(r"needs (\d+) bytes of scratch", str(e.value)).group(1))


def test_size_of_a_refused_step(prob):
    with open_ctx(prob) as ctx:
        for n in (20_000, 33_333):
            assert refuse(ctx, n) == needed(n)


def test_steps_up_to_the_limit_run(prob):
    n = max(n for n in range(1, 12_000) if needed(n) <= LIMIT)
    assert needed(n) > LIMIT - (1 << 19)
    anchors = np.random.default_rng(5).integers(0, prob.n, size=n).astype(np.uint32)
    with open_ctx(prob) as ref, open_ctx(prob) as ctx:
        samples = ref.sample_batch(anchors, 1)
        out = ref.step_explicit(anchors, *samples, 1, 0.01)
        loss = ctx.step_explicit_noalloc(anchors, *samples, 1, 0.01)
        assert np.count_nonzero(loss) > n // 4 and np.array_equal(loss, out["loss"])
        for a, b in zip([ref.get_table(), *ref.get_adam()], [ctx.get_table(), *ctx.get_adam()]):
            assert np.array_equal(a, b)
        refuse(ctx, n + 1)
