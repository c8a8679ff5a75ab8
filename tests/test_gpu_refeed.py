"""A resident context that is given graphs and features again and again: the step buffers are
placed anew each time, and the device memory that the context holds stays the same."""
import numpy as np
import pytest
import torch

from cloverleaf_amd import _native as N
from tests.problems import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("refeed", ["graph", "features"])
def test_refeeding_holds_no_more_memory(refeed):
    prob = make_problem(seed=31, n=200, V=400, D=64, fmax=4)
    cfg = N.default_config()
    cfg.dims, cfg.batch_size, cfg.negatives, cfg.valid_pct, cfg.passes = 64, 64, 3, 0.0, 1
    cfg.max_nodes_kind, cfg.max_nodes = N.EP_SAMPLE_FIXED, 4
    free = []
    with N.Context(cfg) as ctx:
        ctx.set_graph(prob.indptr, prob.indices)
        ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
        ctx.set_table(prob.table)
        for k in range(45):
            if refeed == "graph":
                ctx.set_graph(prob.indptr, prob.indices)
            else:
                ctx.set_features(prob.f_indptr, prob.f_ids, prob.V)
            ctx.learn()
            if k in (4, 44):
                torch.cuda.synchronize()
                free.append(torch.cuda.mem_get_info(0)[0])
    # one array of half a megabyte left behind by each of the 40 rounds would be 20 MiB
    assert free[0] - free[1] < 4 << 20
