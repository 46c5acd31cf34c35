"""The neighbour lists at the edges of their forms: one tile and part of one, the
last short walk and the first long one, one segment and many merged, lists that
stay short; ranked in one call against a float64 ranking."""
import pytest
import torch

from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


def nearest(x, lo, hi, n_base, k):
    d2 = torch.cdist(x[lo:hi].double(), x[:n_base].double()).square()
    own = torch.arange(lo, hi, device=x.device)
    inside = own < n_base
    d2[torch.nonzero(inside).flatten(), own[inside]] = float('inf')
    return torch.sort(d2, dim=1)


@pytest.mark.parametrize('n_base,lo,hi,d,keep,k', [
    (40, 0, 40, 8, 64, 45),           # lists shorter than k
    (256, 0, 256, 64, 256, 240),      # one tile
    (300, 256, 300, 100, 64, 1),
    (1500, 0, 1500, 96, 512, 490),
    (4096, 2048, 4096, 64, 256, 240),    # 16 segments of one tile
    (8448, 8192, 8448, 72, 128, 100),    # 33 tiles dealt to 33 segments
])
def test_ranked_lists(n_base, lo, hi, d, keep, k, device):
    print('ranked lists', n_base, lo, hi, d, keep, k, flush=True)
    g = torch.Generator().manual_seed(n_base + d)
    x = torch.randn(max(n_base, hi), d, generator=g).to(device)
    rows = kernels.HalfRows(x)
    base = rows if n_base == rows.n else rows.rows(0, n_base)
    ids, dist = kernels.knn_nearest(x, rows.rows(lo, hi), base, keep, k, lo, hide_inf=True)
    want_d, want_i = nearest(x, lo, hi, n_base, min(k, n_base))
    there = min(k, n_base - 1)        # the row itself is not among them
    assert ids.shape == dist.shape == (hi - lo, k)
    # float32 sums of d squares, in any order
    assert torch.allclose(dist[:, :there].double(), want_d[:, :there], rtol=d * 2.0 ** -24)
    # halves rank the candidates: with `keep` well above k none of the k is missed
    if keep >= k + 16 or keep >= n_base:
        assert float((ids[:, :there] == want_i[:, :there]).float().mean()) > 0.999
    assert bool((ids[:, there:] == -1).all()) and bool(torch.isinf(dist[:, there:]).all())


@pytest.mark.parametrize('tiles', [1, 2, 32, 33])
@pytest.mark.parametrize('keep', [64, 256, 512])
def test_short_and_long_walks(tiles, keep, device):
    """One segment whose walk is `tiles` tiles and a bit less: the kept set is
    that of the same products ranked by torch."""
    print('walk', tiles, keep, flush=True)
    n, m, d = tiles * 256 - 3, 130, 64
    g = torch.Generator().manual_seed(tiles + keep)
    # whole numbers: every product is exact, and so is the ranking, up to ties
    x = torch.randint(-4, 5, (n, d), generator=g).float().to(device)
    q = torch.randint(-4, 5, (m, d), generator=g).float().to(device)
    base, query = kernels.HalfRows(x, scale=1.0), kernels.HalfRows(q, scale=1.0)
    got = kernels.knn_candidates(query, base, keep, n_seg=1)
    score = x.square().sum(-1) - 2.0 * (q @ x.T)
    kept = min(keep, n)
    worst = torch.sort(score, dim=1).values[:, kept - 1:kept]
    assert got.shape == (m, keep)
    assert bool(((got >= 0).sum(1) == kept).all())
    mine = torch.gather(score, 1, got.clamp(min=0))
    assert bool(((mine <= worst) | (got < 0)).all())
    for i in range(0, m, 17):
        row = got[i][got[i] >= 0]
        assert row.unique().numel() == kept
        assert int((score[i] < worst[i]).sum()) == int((mine[i][got[i] >= 0] < worst[i]).sum())
