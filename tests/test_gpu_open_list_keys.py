"""Keys at the ends of their range in every size of the open list: entries at
negative, tied and infinite distances in no order, on rows whose distances tie
throughout, so that left and right children compare equal on every level."""
import numpy as np
import pytest
import torch

import oracle
from common import assert_same_search
from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ef', [3, 8, 12, 16, 24, 32, 48, 64, 96, 128, 256, 512])
def test_tied_and_extreme_keys(ef, device):
    print('keys', 4 * ef, flush=True)
    n, deg, dp, B, n_init = 4000, 40, 32, 24, 70
    g = torch.Generator().manual_seed(ef)
    x = torch.randint(-2, 3, (n, dp), generator=g).float()
    query = torch.randint(-2, 3, (B, dp), generator=g).float()
    indices = torch.randint(n, (n, deg), generator=g)
    indptr = torch.arange(0, n * deg + 1, deg)
    nodes = torch.arange(n)
    I = torch.stack([torch.randperm(n, generator=g)[:n_init] for _ in range(B)]).contiguous()
    D = torch.randint(-40, 400, (B, n_init), generator=g).float()
    D[:, ::9] = float('inf')
    D[1::3] = D[1::3].sort(-1).values
    D[2::3] = D[2::3].sort(-1, descending=True).values
    D = D.contiguous()
    out_I = torch.empty(B, 4, ef, dtype=torch.long, device=device)
    out_D = torch.empty(B, 4, ef, dtype=torch.float, device=device)
    kernels.traverse_cuda(out_I, out_D, indptr.to(device), indices.flatten().to(device),
                          nodes.to(device), x.to(device), query.to(device), I.to(device),
                          D.to(device), deg)
    ref_I = np.empty((B, 4 * ef), np.int64)
    ref_D = np.empty((B, 4 * ef), np.float32)
    oracle.traverse_cpu(ref_I, ref_D, I.numpy().copy(), D.numpy().copy(), indptr.numpy(),
                        indices.flatten().numpy(), x.numpy(), query.numpy(), 4 * ef)
    given = [dict(zip(I[b].tolist(), D[b].tolist())) for b in range(B)]

    def worst_tie(b, ids, dist):
        # another member of the tie: each at that distance, as an entry or a row
        for i in ids:
            assert dist in (given[b].get(int(i)), float((x[int(i)] - query[b]).square().sum()))

    assert_same_search(out_I.flatten(1).cpu(), out_D.flatten(1).cpu(), ref_I, ref_D, worst_tie)
