"""Rows at equal distances: the neighbour lists name them in the order of the rows,
whatever order the lists were filled in."""
import pytest
import torch

from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,keep', [
    (64, 64), (250, 256),            # one tile, one segment
    (480, 512), (512, 512),          # two segments, merged
])
@pytest.mark.parametrize('copies', [1, 2, 60])
def test_equal_distances_come_in_row_order(n, keep, copies, device):
    print('equal distances', n, keep, copies, flush=True)
    g = torch.Generator().manual_seed(n + copies)
    # whole numbers: every distance and score is exact, and many are equal
    x = torch.randint(-2, 3, (-(-n // copies), 8), generator=g).repeat(copies, 1)[:n]
    x = x[torch.randperm(n, generator=g)].float().to(device)
    rows = kernels.HalfRows(x, scale=1.0)
    d2 = torch.cdist(x.double(), x.double()).square().round().long()
    d2.fill_diagonal_(1 << 20)       # the row itself comes last
    want = torch.sort(d2 * n + torch.arange(n, device=device), dim=1).values
    for _ in range(3):
        ids, dist = kernels.knn_nearest(x, rows, rows, keep, n)
        assert torch.equal(ids, want % n)
        assert torch.equal(dist[:, :-1].long(), (want // n)[:, :-1])
        assert bool(torch.isinf(dist[:, -1]).all())
