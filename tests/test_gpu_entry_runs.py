"""Entries pushed on the open list: every order in which some stay out and later ones
get in again, against the oracle's list (whose array the expansions' order shows)."""
import numpy as np
import pytest
import torch

import oracle
from common import Problem, assert_same_search
from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('order', ['ascending', 'descending', 'saw', 'any', 'equal'])
@pytest.mark.parametrize('ef,n_init', [(4, 100), (8, 64), (16, 130), (64, 200), (250, 300)])
def test_entries_in_any_order(ef, n_init, order, device):
    p = Problem(n=3000, d=32, deg=24, sample_ratio=0.6, seed=ef, n_query=24)
    I, D = p.entries(n_init, seed=7)
    at = torch.argsort(D, 1)
    if order == 'descending':
        at = at.flip(1)
    if order == 'saw':       # rising runs, each begun lower than the one before ended
        at = at.view(24, -1, 5 if n_init % 5 == 0 else 4).transpose(1, 2).flip(1).reshape(24, -1)
    if order != 'any':
        I, D = torch.gather(I, 1, at), torch.gather(D, 1, at)
    if order == 'equal':     # many at the same distance as the one before
        D = (D * 2).round() / 2
    I, D = I.contiguous(), D.contiguous()
    ref_I = np.empty((24, 4 * ef), np.int64)
    ref_D = np.empty((24, 4 * ef), np.float32)
    oracle.traverse_cpu(ref_I, ref_D, I.numpy().copy(), D.numpy().copy(),
                        p.sub_indptr.numpy(), p.sub_indices.numpy(), p.x.numpy(),
                        p.query.numpy(), 4 * ef)
    sub = kernels.prepare_graph(p.sub_indptr.to(device), p.sub_indices.to(device),
                                p.mapping.to(device), p.nodelist.numel(), p.deg)
    rows = kernels.prepare_rows(p.x[p.nodelist].contiguous().to(device))
    for beside in (0, 1 << 40):
        out_I = torch.empty(24, 4, ef, dtype=torch.long, device=device)
        out_D = torch.empty(24, 4, ef, device=device)
        kernels.traverse_prepared(out_I, out_D, sub, rows, p.query.to(device), I.to(device),
                                  D.to(device), beside=beside)
        got_I, got_D = out_I.flatten(1).cpu().numpy(), out_D.flatten(1).cpu().numpy()
        if order == 'equal':   # members of a tie may differ, distances not
            assert np.array_equal(got_D, ref_D)
        else:
            assert_same_search(got_I, got_D, ref_I, ref_D)
