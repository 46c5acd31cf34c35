"""Searches whose wavefront has helpers that read rows ahead of it, against the
oracle and, bit for bit and counter for counter, against the form without."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from common import Problem, assert_same_search
from pilotann_amd import _lib, kernels

pytestmark = pytest.mark.gpu

# dp, degree, ef, entries, queries: one new row a step and up to 64; the lists of
# every storage form (registers, LDS, device memory); one, a few, many queries
CASES = [
    (8, 1, 4, 1, 1),
    (8, 8, 4, 2, 1024),   # (as many as run at once: four workgroups a compute unit)
    (32, 32, 16, 32, 65),
    (40, 17, 24, 64, 128),
    (64, 64, 48, 0, 3),
    (96, 33, 64, 7, 40),
    (128, 64, 8, 64, 300),
    (128, 64, 128, 64, 33),
    (128, 48, 250, 16, 9),
    (64, 32, 512, 32, 5),
]


def wavefronts(n_storage, batch, beside, dp, ef_total):
    form = ctypes.c_int(-1)
    _lib.check(_lib.lib().pa_traverse_wavefronts(n_storage, batch, beside, dp, ef_total,
                                                 ctypes.byref(form)), 'pa_traverse_wavefronts')
    return form.value


@pytest.mark.parametrize('dp,deg,ef,n_init,n_query', CASES)
def test_same_as_without_helpers(dp, deg, ef, n_init, n_query, device):
    p = Problem(n=5000, d=dp, deg=deg, sample_ratio=0.5, seed=dp + deg, n_query=n_query)
    I, D = p.entries(max(n_init, 1), seed=5)
    I, D = I[:, :n_init].contiguous(), D[:, :n_init].contiguous()
    if n_init > 4:
        I[:, 3], D[:, 3] = I[:, 1], D[:, 1]   # an entry twice
        I[:, 2] = -1                          # an unused one
    sub = kernels.prepare_graph(p.sub_indptr.to(device), p.sub_indices.to(device),
                                p.mapping.to(device), p.nodelist.numel(), deg)
    rows = kernels.prepare_rows(p.x[p.nodelist].contiguous().to(device))
    query, dI, dD = p.query.to(device), I.to(device), D.to(device)
    assert [wavefronts(p.nodelist.numel(), n_query, beside, dp, 4 * ef)
            for beside in (0, 1 << 40)] == [4, 1]
    results = []
    for beside in (0, 1 << 40):
        out_I = torch.empty(n_query, 4, ef, dtype=torch.long, device=device)
        out_D = torch.empty(n_query, 4, ef, device=device)
        tally = torch.zeros(5, dtype=torch.long, device=device)
        kernels.traverse_prepared(out_I, out_D, sub, rows, query, dI, dD, tally, beside=beside)
        results.append((out_I.flatten(1).cpu(), out_D.flatten(1).cpu(), tally.cpu()))
    for with_helpers, without in zip(*results):
        assert torch.equal(with_helpers, without)
    ref_I = np.empty((n_query, 4 * ef), np.int64)
    ref_D = np.empty((n_query, 4 * ef), np.float32)
    oracle.traverse_cpu(ref_I, ref_D, I.numpy().copy(), D.numpy().copy(),
                        p.sub_indptr.numpy(), p.sub_indices.numpy(), p.x.numpy(),
                        p.query.numpy(), 4 * ef)
    assert_same_search(results[0][0].numpy(), results[0][1].numpy(), ref_I, ref_D)
