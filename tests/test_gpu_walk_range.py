"""A walk on the device refuses what a walk on the host refuses: an edge to a
node that is not there, in a row that the walk looks at."""
import pytest
import torch

from pilotann_amd import utils

pytestmark = pytest.mark.gpu


def outcome(adj, start, reverse):
    try:
        return utils.reachable(adj, start, reverse=reverse).cpu()
    except IndexError:
        return None


@pytest.mark.parametrize('reverse', [False, True])
@pytest.mark.parametrize('node', [0, 4, 30, 31, 39])
@pytest.mark.parametrize('number', [40, 41, 1 << 40, -1, -2])
def test_edge_to_no_node(number, node, reverse, device):
    """A chain 0 -> 1 -> .. -> 30 and nodes that nothing leads to."""
    n = 40
    adj = torch.full((n, 70), -1, dtype=torch.long)
    adj[:30, 69] = torch.arange(1, 31)
    adj[node, 65] = number
    start = torch.tensor([4])
    want = outcome(adj, start, reverse)
    assert (want is None) == (number >= n and (reverse or 4 <= node <= 30))
    got = outcome(adj.to(device), start.to(device), reverse)
    assert (got is None) == (want is None)
    if want is not None:
        assert torch.equal(got, want)
