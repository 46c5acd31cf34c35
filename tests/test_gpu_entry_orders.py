"""Entries pushed on the open list in every order they can come in: the walk is
taken again only after an entry that got in, which must leave the list, cell
for cell, what one push after the other leaves (oracle)."""
import numpy as np
import pytest
import torch

import oracle
from common import Problem, assert_same_search
from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def problem():
    return Problem(n=3000, d=32, deg=32, sample_ratio=0.4, seed=61, n_query=32)


@pytest.mark.parametrize('order', ['as drawn', 'ascending', 'descending', 'coarse'])
@pytest.mark.parametrize('ef,n_init', [(1, 1), (4, 65), (32, 200), (128, 128), (512, 300)])
def test_entry_orders(order, ef, n_init, problem, device):
    print('entries', order, ef, n_init, flush=True)
    p, B = problem, 32
    I, D = p.entries(n_init, seed=ef)
    if order in ('ascending', 'descending'):
        D, place = torch.sort(D, dim=1, descending=order == 'descending')
        I = torch.gather(I, 1, place)
    elif order == 'coarse':       # many entries at one distance, some unused places
        D = (D / 8).round() * 8
        I[:, ::7] = -1
    I, D = I.contiguous(), D.contiguous()
    out_I = torch.empty(B, 4, ef, dtype=torch.long, device=device)
    out_D = torch.empty(B, 4, ef, dtype=torch.float, device=device)
    kernels.traverse_cuda(out_I, out_D, p.sub_indptr.to(device), p.sub_indices.to(device),
                          p.mapping.to(device), p.x[p.nodelist].contiguous().to(device),
                          p.query.contiguous().to(device), I.to(device), D.to(device), p.deg)
    ref_I = np.empty((B, 4 * ef), np.int64)
    ref_D = np.empty((B, 4 * ef), np.float32)
    oracle.traverse_cpu(ref_I, ref_D, I.numpy().copy(), D.numpy().copy(),
                        p.sub_indptr.numpy(), p.sub_indices.numpy(), p.x.numpy(),
                        p.query.numpy(), 4 * ef)
    x, query = p.x.numpy(), p.query.numpy()

    def at_that_distance(b, ids, dist):
        # an entry that was named with that distance, or a row at it
        named = I[b][D[b] == dist].tolist()
        rows = oracle.square_dist(query[b].copy(), x, ids.copy())
        for node, row in zip(ids.tolist(), rows):
            assert node in named or (int(p.mapping[node]) >= 0 and row == dist)
    # with rounded distances, entries at exactly the worst distance kept may be
    # others of that distance
    assert_same_search(out_I.flatten(1).cpu(), out_D.flatten(1).cpu(), ref_I, ref_D,
                       worst_tie=at_that_distance if order == 'coarse' else None)
