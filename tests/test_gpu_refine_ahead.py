"""The refine's three forms (eight, four and one wavefront a query) on the random cases
of the sweep: the same in every bit.  Cases with more candidates than a wavefront has
lanes, with and without coordinates to complete, one query and some dozens."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from pilotann_amd import _lib, kernels
from test_gpu_refine_fuzz import make_case

pytestmark = pytest.mark.gpu


def wavefronts(c, beside):
    form = ctypes.c_int(-1)
    _lib.check(_lib.lib().pa_refine_wavefronts(c['n'], c['B'], beside, c['d'], c['ef_search'],
                                               ctypes.byref(form)), 'pa_refine_wavefronts')
    return form.value


@pytest.mark.parametrize('seed', range(24))
def test_three_forms_agree(seed, device):
    c = make_case(9000 + seed)
    print('refine forms', seed, c['n'], c['d'], c['dp'], c['ef_search'], c['B'], flush=True)
    xn, qn = c['x'][:, :c['dp']].contiguous().numpy(), c['query'][:, :c['dp']].contiguous().numpy()
    cand_D = torch.from_numpy(np.stack([
        oracle.square_dist(qn[b].copy(), xn, c['cand'][b].clamp(min=0).numpy().copy())
        for b in range(c['B'])])).to(device)
    sub = kernels.prepare_graph(c['sub_indptr'].to(device), c['sub_indices'].to(device),
                                c['mapping'].to(device), c['n_sub'], c['deg_sub'])
    full = kernels.prepare_full_graph(c['full_indptr'].to(device),
                                      c['full_indices'].to(device), c['deg_full'])
    rows = kernels.PreparedRows(c['x'].to(device))
    query = c['query'].to(device)
    besides = [next(b for b in range(0, 1 << 13, 16) if wavefronts(c, b) == form)
               for form in (8, 4, 1)]
    results = []
    for beside in besides:
        init_I, init_D = c['cand'].to(device), cand_D.clone()
        buf_I = torch.empty(c['B'], c['n_buffers'], dtype=torch.long, device=device)
        buf_D = torch.empty(c['B'], c['n_buffers'], device=device)
        out_I = torch.empty(c['B'], c['k'], dtype=torch.long, device=device)
        out_D = torch.empty(c['B'], c['k'], device=device)
        counters = torch.zeros(6, dtype=torch.long, device=device)
        kernels.traverse_refine_cuda(out_I, out_D, buf_I, buf_D, init_I, init_D, sub, full, rows,
                                     query, c['ef_search'], c['dp'], counters, beside=beside)
        results.append([t.cpu().numpy() for t in (out_I, out_D, buf_I, buf_D, init_D, counters)])
    for ahead, helped, single in zip(*results):
        assert np.array_equal(ahead, single, equal_nan=ahead.dtype == np.float32)
        assert np.array_equal(helped, single, equal_nan=helped.dtype == np.float32)
