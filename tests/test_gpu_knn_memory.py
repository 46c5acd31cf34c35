"""Memory of a call of kernels.knn_candidates: a row of a large set has a list of
scores and ids and a row of the table, and little beside them at any moment."""
import pytest
import torch

from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


def test_memory_of_a_pass(device):
    n, keep = 1 << 17, 256
    rows = kernels.HalfRows(torch.randn(n, 64, device=device))
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    table = kernels.knn_candidates(rows, rows, keep)
    torch.cuda.synchronize()
    peak = (torch.cuda.max_memory_allocated() - before) / n
    # ids of the lists, then twice the table (as it is made and as it is
    # returned) and its mask: less than the 11.5 KB that the whole call took
    # with lists of 640 places
    assert table.shape == (n, keep) and int(table.min()) >= 0
    assert peak < 11.5 * 1024, peak
