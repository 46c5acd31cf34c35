"""The wide mode in launches with more queries than run at once (rows of 128
floats are read one pass at a time with the pool of 1024 then): every copy of a
query as in a small launch."""
import pytest
import torch

from common import Problem
from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ef', [129, 256])
def test_full_launches(ef, device):
    print('wide full', ef, flush=True)
    B, times = 24, 180     # 4320 queries, at most 4096 of this pool at once
    p = Problem(n=5000, d=128, deg=40, sample_ratio=0.6, seed=81, n_query=B)
    I, D = p.entries(24, seed=ef)
    graph = kernels.prepare_graph(p.sub_indptr.to(device), p.sub_indices.to(device),
                                  p.mapping.to(device), len(p.nodelist), p.deg)
    rows = kernels.PreparedRows(p.x[p.nodelist].contiguous().to(device))

    def search(n):
        out_I = torch.empty(n * B, 4, ef, dtype=torch.long, device=device)
        out_D = torch.empty(n * B, 4, ef, device=device)
        kernels.traverse_wide_prepared(out_I, out_D, graph, rows,
                                       p.query.repeat(n, 1).to(device),
                                       I.repeat(n, 1).to(device), D.repeat(n, 1).to(device))
        return out_I.view(n, B, -1), out_D.view(n, B, -1)
    few_I, few_D = search(1)
    many_I, many_D = search(times)
    assert torch.equal(many_D, few_D.expand_as(many_D))
    assert torch.equal(many_I, few_I.expand_as(many_I))
