"""Row lengths at the edges of how a row is read (chunks of 16 groups of eight in
the traversal and in the refine with one wavefront per query, of 32 in the one
with four; the rest in pieces of 16, 8, 4 and 2 groups, a last odd group; a tail
that starts at an odd group): the traversal on reduced rows without a kernel of
their own and both forms of the refine, bit for bit the oracle's."""
import numpy as np
import pytest
import torch

import oracle
from common import Problem, assert_same_search
from pilotann_amd import kernels
from test_gpu_refine import candidates, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('d,dp', [
    (8, 8), (16, 8), (24, 16), (40, 24), (56, 40), (96, 96), (104, 72),
    (120, 104), (136, 8), (200, 120), (248, 136), (256, 248), (264, 40),
    (384, 136), (504, 248), (520, 8), (632, 104), (760, 392), (768, 40), (768, 128),
])
def test_row_lengths(d, dp, device):
    print('row lengths', d, dp, flush=True)
    ef = 8
    p = Problem(n=2500, d=d, deg=32, sample_ratio=0.3, seed=51, n_query=24)
    init_I, init_D = p.entries(32, seed=9, dp=dp)
    cand_I, cand_D = candidates(p, dp, ef, 32, device)
    B = p.query.size(0)
    ref_I = np.empty((B, 4 * ef), np.int64)
    ref_D = np.empty((B, 4 * ef), np.float32)
    oracle.traverse_cpu(ref_I, ref_D, init_I.numpy().copy(), init_D.numpy().copy(),
                        p.sub_indptr.numpy(), p.sub_indices.numpy(),
                        np.ascontiguousarray(p.x[:, :dp].numpy()),
                        np.ascontiguousarray(p.query[:, :dp].numpy()), 4 * ef)
    assert_same_search(cand_I.cpu(), cand_D.cpu(), ref_I, ref_D)
    got, ref = run_both(p, dp, 24, 10, cand_I, cand_D, device)
    assert_same_search(got['buf_I'], got['buf_D'], ref['buf_I'], ref['buf_D'])
    assert_same_search(got['out_I'], got['out_D'], ref['out_I'], ref['out_D'])
