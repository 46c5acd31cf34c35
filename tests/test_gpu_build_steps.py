"""Steps of the graph build that are kernels of their own: rows in two
half-precision parts, and the walk along a graph's edges."""
import pytest
import torch

from pilotann_amd import kernels, utils

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,d', [(1, 1), (5, 3), (256, 64), (257, 66), (300, 260), (40, 100)])
def test_rows_in_two_parts(n, d, device):
    print('two parts', n, d, flush=True)
    g = torch.Generator().manual_seed(n + d)
    x = torch.randn(n, d, generator=g)
    x[0, 0] = 1e9                        # clamped to the half range
    if d > 2:
        x[-1, 2] = float('nan')          # stays what it is
    x = x.to(device)
    rows = kernels.HalfRows(x, scale=0.75)
    low = rows.low(x)
    want = (x * 0.75).clamp(-60000.0, 60000.0)
    tile = rows.tile
    assert rows.half.shape == low.shape == (-(-n // tile) * tile, -(-d // 64) * 64)
    half = want.half()
    assert torch.equal(rows.half[:n, :d].nan_to_num(7), half.nan_to_num(7))
    assert torch.equal(low[:n, :d].nan_to_num(7), (want - half.float()).half().nan_to_num(7))
    for part in (rows.half, low):
        assert not bool(part[n:].any()) and not bool(part[:, d:].any())
    exact = want.double().square().sum(-1)
    ok = ~exact.isnan()
    # a float32 sum of d squares, in any order
    assert torch.allclose(rows.norm[:n][ok].double(), exact[ok], rtol=(d + 2) * 2.0 ** -24)
    assert not bool(rows.norm[n:].any())


@pytest.mark.parametrize('n,deg,edges', [
    (1, 1, 0.0), (700, 3, 0.35), (5000, 2, 0.5), (900, 70, 0.02), (3000, 48, 0.02)])
def test_walk_reaches_what_the_host_reaches(n, deg, edges, device):
    print('walk', n, deg, edges, flush=True)
    g = torch.Generator().manual_seed(n + deg)
    adj = torch.randint(0, n, (n, deg), generator=g)
    adj[torch.rand(n, deg, generator=g) >= edges] = -1
    sources = torch.randint(0, n, (min(n, 3),), generator=g)
    for reverse in (False, True):
        want = utils.reachable(adj, sources, reverse=reverse)
        got = utils.reachable(adj.to(device), sources.to(device), reverse=reverse)
        assert got.dtype == torch.bool and torch.equal(got.cpu(), want)


@pytest.mark.parametrize('reverse', [False, True])
def test_walk_along_a_chain(reverse, device):
    """Far more steps than one call makes, in either direction of the numbers."""
    n = 400
    adj = torch.full((n, 2), -1, dtype=torch.long)
    adj[1:, 1] = torch.arange(n - 1)     # node i -> i - 1
    start = torch.tensor([n // 2])
    got = utils.reachable(adj.to(device), start.to(device), reverse=reverse).cpu()
    want = torch.arange(n) >= n // 2 if reverse else torch.arange(n) <= n // 2
    assert torch.equal(got, want)
