"""The reverse edges made on the device against those made with torch on the host:
the same rows, place for place."""
import pytest
import torch

from pilotann_amd import kernels
from pilotann_amd.utils import graphs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,m,degree,edges', [
    (1, 1, 1, 'any'), (2, 1, 2, 'any'), (65, 64, 64, 'any'), (300, 7, 5, 'any'),
    (5000, 16, 32, 'any'), (5000, 48, 48, 'any'), (4097, 24, 64, 'holes'),
    (3000, 8, 40, 'hub'), (3000, 1, 64, 'hub'), (700, 5, 9, 'none'),
])
def test_same_rows_as_on_the_host(n, m, degree, edges, device):
    g = torch.Generator().manual_seed(n + m)
    forward = torch.stack([torch.randperm(max(n, m), generator=g)[:m] for _ in range(n)])
    forward[forward >= n] = -1
    if edges == 'hub':      # nodes that thousands point at, from every place
        hubs = torch.randint(0, 3, (n,), generator=g)
        place = torch.randint(0, m, (n,), generator=g)
        forward[forward < 3] = -1
        forward[torch.arange(n), place] = hubs
    if edges == 'holes':
        forward[torch.rand(n, m, generator=g) < 0.4] = -1
    if edges == 'none':
        forward[:] = -1
    want = graphs._add_reverse(forward, degree)
    got = graphs._add_reverse(forward.to(device), degree)
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize('n,m,degree', [(1, 1, 1), (65, 9, 12), (3000, 48, 48), (3000, 64, 20)])
def test_a_number_beyond_the_nodes_is_no_edge(n, m, degree, device):
    g = torch.Generator().manual_seed(n + m)
    forward = torch.randint(-1, n, (n, m), generator=g)
    none = torch.rand(n, m, generator=g) < 0.3
    beyond = torch.tensor([n, n + 1, (1 << 31) - 1, 1 << 31, 1 << 40])
    beyond = beyond[torch.randint(5, (n, m), generator=g)]
    got = kernels.graph_add_reverse(torch.where(none, beyond, forward).to(device), degree)
    want = graphs._add_reverse(forward.masked_fill(none, -1), degree)
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize('n', [0, 1, 1000, 1001, 2999, 3000, 10_007])
def test_ids_reach_the_host_whole(n, device):
    g = torch.Generator().manual_seed(n)
    ids = torch.randint(-1, max(n, 1), (n,), generator=g)
    assert torch.equal(graphs._ids_to_host(ids.to(device), piece=1000), ids)
