"""Launches that share the device: the forms for launches that have it to
themselves (four wavefronts a query in the refine, visited bits in LDS in the
traversal) count the queries of the others, and a search in two halves says how
many there are."""
import ctypes

import pytest
import torch

from common import Problem
from pilotann_amd import IndexStaged, _lib, kernels, utils

pytestmark = pytest.mark.gpu


def near_bits(n_storage, batch, beside, dp, ef_total):
    form = ctypes.c_int(-1)
    _lib.check(_lib.lib().pa_traverse_form(n_storage, batch, beside, dp, ef_total,
                                           ctypes.byref(form)), 'pa_traverse_form')
    return form.value


def wavefronts(n_nodes, batch, beside, d, ef_search):
    form = ctypes.c_int(-1)
    _lib.check(_lib.lib().pa_refine_form(n_nodes, batch, beside, d, ef_search,
                                         ctypes.byref(form)), 'pa_refine_form')
    return form.value


@pytest.mark.parametrize('n,dp,ef', [(250_000, 128, 128), (100_000, 64, 512), (75_000, 40, 128)])
def test_near_bits_for_what_runs_at_once(n, dp, ef, device):
    alone = max(b for b in range(0, 8192, 128) if near_bits(n, b, 0, dp, ef))
    assert near_bits(n, alone + 128, 0, dp, ef) == 0
    half = alone // 2
    assert near_bits(n, half, alone - half, dp, ef) == 1
    assert near_bits(n, half, alone - half + 256, dp, ef) == 0
    assert near_bits(n, alone, 128, dp, ef) == 0
    assert near_bits(n, 1, alone, dp, ef) == 0


@pytest.mark.parametrize('d,ef', [(768, 32), (96, 64), (200, 1024), (128, 2048)])
def test_helping_wavefronts_for_what_runs_at_once(d, ef, device):
    n = 1_000_000
    alone = max(b for b in range(0, 2048, 64) if wavefronts(n, b, 0, d, ef) == 4)
    assert 0 < alone <= 1024
    assert wavefronts(n, alone + 64, 0, d, ef) == 1
    assert wavefronts(n, alone // 2, alone - alone // 2, d, ef) == 4
    assert wavefronts(n, alone, 64, d, ef) == 1
    assert wavefronts(n, 1, alone, d, ef) == 1


def test_results_do_not_depend_on_it(device):
    ef, k, dp = 16, 10, 32
    p = Problem(n=4000, d=64, deg=32, sample_ratio=0.4, seed=91, n_query=64)
    I, D = p.entries(32, seed=3, dp=dp)
    I, D = I.to(device), D.to(device)
    sub = kernels.prepare_graph(p.sub_indptr.to(device), p.sub_indices.to(device),
                                p.mapping.to(device), p.nodelist.numel(), p.deg)
    full = kernels.prepare_full_graph(p.indptr.to(device), p.indices.to(device))
    x, query = p.x.to(device), p.query.to(device)
    rows = kernels.prepare_rows(x)
    low = kernels.prepare_rows(x[p.nodelist.to(device), :dp].contiguous())
    results = []
    for beside in (0, 1, 5000, 1 << 40):
        cand_I = torch.empty(64, 4, ef, dtype=torch.long, device=device)
        cand_D = torch.empty(64, 4, ef, device=device)
        kernels.traverse_prepared(cand_I, cand_D, sub, low, query[:, :dp].contiguous(), I, D,
                                  beside=beside)
        out = [cand_I.clone(), cand_D.clone(), torch.empty(64, k, dtype=torch.long, device=device),
               torch.empty(64, k, device=device)]
        i, d = cand_I.flatten(1), cand_D.flatten(1)
        kernels.traverse_refine_cuda(out[2], out[3], i, d, i, d, sub, full, rows, query, 24, dp,
                                     beside=beside)
        results.append(out + [i, d])
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    with pytest.raises(RuntimeError):
        kernels.traverse_prepared(cand_I, cand_D, sub, low, query[:, :dp].contiguous(), I, D,
                                  beside=-1)
    with pytest.raises(RuntimeError):
        kernels.traverse_refine_cuda(out[2], out[3], i, d, i, d, sub, full, rows, query, 24, dp,
                                     beside=-1)


@pytest.mark.parametrize('batch', [2047, 2048, 2049, 2051])
@pytest.mark.parametrize('traversal', ['exact', 'wide'])
def test_a_search_in_halves_says_so(batch, traversal, device, monkeypatch):
    """Up to 2047 queries are one launch; of more, each half names the other."""
    x = utils.gaussian_mixture(6000, 64, 8, 0.6, seed=1)
    index = IndexStaged(d_model=64, d_principle=32, sample_ratio=0.4, graph_method='nsw32',
                        entry_method='random32', seed=3, build_device=device)
    index.train(x)
    index.to(device)
    query = utils.gaussian_mixture(batch, 64, 8, 0.6, seed=2, center_seed=1)
    calls = []
    for name in ('traverse_prepared', 'traverse_refine_cuda'):
        def watched(*args, real=getattr(kernels, name), name=name, **kw):
            rows = args[4].size(0) if name == 'traverse_prepared' else args[9].size(0)
            calls.append((name, rows, kw.get('beside', 0)))
            return real(*args, **kw)
        monkeypatch.setattr(kernels, name, watched)
    I, D = index.search(query, k=10, ef_search=16, refine='device', traversal=traversal)
    half = (batch + 1) // 2
    launches = [(batch, 0)] if batch < 2048 else [(half, batch - half), (batch - half, half)]
    for name in ('traverse_prepared', 'traverse_refine_cuda'):
        want = [] if name == 'traverse_prepared' and traversal == 'wide' else launches
        assert [c[1:] for c in calls if c[0] == name] == want
    # the same rows as one query after the other finds
    few_I, few_D = index.search(query[:50], k=10, ef_search=16, refine='device',
                                traversal=traversal)
    assert torch.equal(I[:50], few_I) and torch.equal(D[:50], few_D)
