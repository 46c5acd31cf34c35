"""Every size of the search's lists (the deepest level of the open list whole, in
part, or of one node; in registers, LDS or device memory), traversal and refine,
against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from common import Problem, assert_same_search
from pilotann_amd import kernels
from test_gpu_refine import run_both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def problem():
    return Problem(n=6000, d=128, deg=48, sample_ratio=0.5, seed=71, n_query=40)


@pytest.mark.parametrize('dp', [32, 128])
@pytest.mark.parametrize('ef', [3, 8, 12, 16, 24, 32, 48, 64, 96, 128, 256, 512])
def test_list_sizes(ef, dp, problem, device):
    print('list size', 4 * ef, dp, flush=True)
    p, B = problem, 40
    I, D = p.entries(32, seed=ef, dp=dp)
    out_I = torch.empty(B, 4, ef, dtype=torch.long, device=device)
    out_D = torch.empty(B, 4, ef, dtype=torch.float, device=device)
    x = p.x[:, :dp].contiguous()
    query = p.query[:, :dp].contiguous()
    kernels.traverse_cuda(out_I, out_D, p.sub_indptr.to(device), p.sub_indices.to(device),
                          p.mapping.to(device), x[p.nodelist].contiguous().to(device),
                          query.to(device), I.to(device), D.to(device), p.deg)
    ref_I = np.empty((B, 4 * ef), np.int64)
    ref_D = np.empty((B, 4 * ef), np.float32)
    oracle.traverse_cpu(ref_I, ref_D, I.numpy().copy(), D.numpy().copy(),
                        p.sub_indptr.numpy(), p.sub_indices.numpy(), x.numpy(),
                        query.numpy(), 4 * ef)
    cand_I, cand_D = out_I.flatten(1).contiguous(), out_D.flatten(1).contiguous()
    assert_same_search(cand_I.cpu(), cand_D.cpu(), ref_I, ref_D)
    k = min(10, 4 * ef)
    # the refine's lists are as long: 4 * ef cells
    got, ref = run_both(p, dp, 4 * ef, k, cand_I, cand_D, device)
    assert_same_search(got['buf_I'], got['buf_D'], ref['buf_I'], ref['buf_D'])
    assert_same_search(got['out_I'], got['out_D'], ref['out_I'], ref['out_D'])
