"""The refine with four wavefronts per query and with one, over the random cases of
the sweep against the oracle (which runs the first form): the same in every bit."""
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
    _lib.check(_lib.lib().pa_refine_form(c['n'], c['B'], beside, c['d'], c['ef_search'],
                                         ctypes.byref(form)), 'pa_refine_form')
    return form.value


@pytest.mark.parametrize('seed', range(80))
def test_forms_agree(seed, device):
    c = make_case(5000 + seed)
    print('refine forms', seed, c['n'], c['d'], c['dp'], c['ef_search'], c['B'], flush=True)
    assert (wavefronts(c, 0), wavefronts(c, 1 << 40)) == (4, 1)
    x, query = c['x'].to(device), c['query'].to(device)
    xn, qn = c['x'][:, :c['dp']].contiguous().numpy(), c['query'][:, :c['dp']].contiguous().numpy()
    cand_D = torch.from_numpy(np.stack([
        oracle.square_dist(qn[b].copy(), xn, c['cand'][b].clamp(min=0).numpy().copy())
        for b in range(c['B'])])).to(device)
    sub = kernels.prepare_graph(c['sub_indptr'].to(device), c['sub_indices'].to(device),
                                c['mapping'].to(device), c['n_sub'], c['deg_sub'])
    full = kernels.prepare_full_graph(c['full_indptr'].to(device),
                                      c['full_indices'].to(device), c['deg_full'])
    rows = kernels.PreparedRows(x)
    results = []
    for beside in (0, 1 << 40):
        init_I, init_D = c['cand'].to(device), cand_D.clone()
        buf_I = torch.empty(c['B'], c['n_buffers'], dtype=torch.long, device=device)
        buf_D = torch.empty(c['B'], c['n_buffers'], device=device)
        out_I = torch.empty(c['B'], c['k'], dtype=torch.long, device=device)
        out_D = torch.empty(c['B'], c['k'], device=device)
        counters = torch.zeros(6, dtype=torch.long, device=device)
        kernels.traverse_refine_cuda(out_I, out_D, buf_I, buf_D, init_I, init_D, sub, full, rows,
                                     query, c['ef_search'], c['dp'], counters, beside=beside)
        results.append([t.cpu().numpy() for t in (out_I, out_D, buf_I, buf_D, init_D, counters)])
    for few, many in zip(*results):
        assert np.array_equal(few, many, equal_nan=few.dtype == np.float32)


@pytest.mark.parametrize('ef_search,batch', [(16, 1024), (64, 1024), (512, 1024), (513, 768),
                                             (1024, 768), (1025, 512), (2048, 512)])
def test_batches_that_have_four_wavefronts(ef_search, batch, device):
    """The registers of each size of the lists leave room for so many queries at once."""
    for d in (96, 768):
        case = dict(n=1_000_000, B=batch, d=d, ef_search=ef_search)
        assert wavefronts(case, 0) == 4
