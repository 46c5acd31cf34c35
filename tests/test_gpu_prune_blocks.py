"""Occlusion pruning straight from the rows at the edges of its blocks: 64
candidates at a time, 32 kept ones multiplied with them at a time, against the
rule written out on float64 distances."""
import pytest
import torch

from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('fill', [True, False])
@pytest.mark.parametrize('k,m_keep', [
    (1, 1), (63, 40), (64, 64), (65, 7), (128, 33), (129, 100), (192, 31), (256, 1),
    (256, 96), (256, 256), (200, 300),
])
def test_blocks(k, m_keep, fill, device):
    print('prune blocks', k, m_keep, fill, flush=True)
    g = torch.Generator().manual_seed(k)
    n, d, nodes = 700, 72, 24
    rows = torch.randn(n, d, generator=g)
    # a node between the centre of the rows (all candidates are kept: they are
    # farther from each other than from it) and one of them (few are)
    share = torch.linspace(0, 0.9, nodes).unsqueeze(-1)
    at = (share * rows[:nodes]).double()
    own = torch.cdist(at, rows.double()).square()
    d2 = torch.cdist(rows.double(), rows.double()).square()
    own[torch.arange(nodes), torch.arange(nodes)] = float('inf')
    cand = torch.argsort(own, dim=1)[:, :k].contiguous()
    cand_d = torch.gather(own, 1, cand)
    if k > 10:                       # some lists end early
        cand[::5, k - 6:] = -1
        cand_d[::5, k - 6:] = float('inf')
    got = kernels.graph_prune_rows(rows.to(device), cand.to(device),
                                   cand_d.float().to(device), m_keep, fill).cpu()
    assert got.shape == (nodes, m_keep)
    compared = 0
    for i in range(nodes):
        valid = int((cand[i] >= 0).sum())
        kept, rejected, near_tie = [], [], False
        for j in range(valid):
            if len(kept) >= m_keep:
                rejected.append(j)
                continue
            pair = d2[cand[i, j]][cand[i, kept]]
            # products of two parts hold about 22 bits of |a|^2 + |b|^2 ~ 2 d
            near_tie |= bool(((pair - cand_d[i, j]).abs() < 4 * d * 2.0 ** -21).any())
            (rejected if bool((pair < cand_d[i, j]).any()) else kept).append(j)
        want = (kept + (rejected if fill else []))[:m_keep]
        want += [-1] * (m_keep - len(want))
        if not near_tie:
            compared += 1
            assert got[i].tolist() == want, i
    assert compared >= nodes * 3 // 4
