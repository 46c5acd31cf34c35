"""Candidates for no rows: an empty table, whatever its width; what does not fit
together is refused all the same."""
import pytest
import torch

from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('keep', [1, 64, 100, 512, 1000])
def test_no_rows(keep, device):
    base = torch.randn(300, 64, device=device)
    got = kernels.knn_candidates(base[:0], base, keep)
    assert got.shape == (0, keep) and got.dtype == torch.long and got.device == base.device


@pytest.mark.parametrize('n,d,m,keep', [(300, 64, 0, 64), (0, 32, 0, 64), (300, 32, 5, 100)])
def test_refused(n, d, m, keep, device):
    with pytest.raises(RuntimeError):
        kernels.knn_candidates(torch.randn(m, 32, device=device),
                               torch.randn(n, d, device=device), keep)
