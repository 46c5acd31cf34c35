"""The same queries in a small launch and in one of more queries than run at once,
whose wavefronts take one query after the other on the same lists and bits: the
same rows, bit for bit.  (Both have the visited bits in LDS where these are few,
as here; test_gpu_full_launches.py compares the two forms.)"""
import pytest
import torch

from common import Problem
from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('d', [32, 40, 128])
@pytest.mark.parametrize('ef', [4, 48, 256])
def test_batch_size_does_not_matter(d, ef, device):
    print('near bits', d, ef, flush=True)
    p = Problem(n=5000, d=d, deg=32, sample_ratio=0.6, seed=81, n_query=48)
    I, D = p.entries(32, seed=3)
    I[:, 5] = -1
    args = [p.sub_indptr.to(device), p.sub_indices.to(device), p.mapping.to(device),
            p.x[p.nodelist].contiguous().to(device)]

    def search(times):
        B = 48 * times
        out_I = torch.full((B, 4, ef), -7, dtype=torch.long, device=device)
        out_D = torch.full((B, 4, ef), -7.0, device=device)
        counters = torch.zeros(5, dtype=torch.long, device=device)
        kernels.traverse_cuda(out_I, out_D, *args, p.query.repeat(times, 1).to(device),
                              I.repeat(times, 1).to(device), D.repeat(times, 1).to(device),
                              p.deg, counters=counters)
        return out_I, out_D, counters

    few_I, few_D, few = search(1)
    # more queries than any launch runs at once (20 wavefronts a compute unit)
    times = 5400 // 48
    many_I, many_D, many = search(times)
    assert torch.equal(many_I, few_I.repeat(times, 1, 1))
    assert torch.equal(many_D, few_D.repeat(times, 1, 1))
    assert torch.equal(many, few * times)
