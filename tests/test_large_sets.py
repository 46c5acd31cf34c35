"""Sets of more rows than one launch has work-items for: the builder's kernels
with a wavefront per row take them in several launches."""
import pytest
import torch

from pilotann_amd import _lib, utils

WORK_ITEMS = 1 << 32
ROWS = WORK_ITEMS // 64      # rows of a wavefront each that no launch holds


def test_rows_in_two_parts_take_any_number_of_rows():
    """The number is no reason to refuse: what is reported is the missing
    array."""
    lib = _lib.lib()
    assert lib.pa_rows_low(None, None, ROWS, ROWS, 4, 4, 1.0, 6e4, None) == -1
    assert lib.pa_rows_low(None, None, ROWS, ROWS - 1, 4, 4, 1.0, 6e4, None) == -2


@pytest.mark.gpu
@pytest.mark.parametrize('n,pad', [(1 << 22, 0), ((1 << 22) + 1, 2), (ROWS + 5, 3)])
def test_rows_in_two_parts_over_several_launches(n, pad, device):
    print('two parts of', n, flush=True)
    g = torch.Generator(device=device).manual_seed(n)
    x = torch.randn(n, 3, device=device, generator=g)
    low = torch.full((n + pad, 4), 7.0, dtype=torch.float16, device=device)
    _lib.check(_lib.lib().pa_rows_low(
        low.data_ptr(), x.data_ptr(), n, n + pad, 3, 4, 0.75, 60000.0,
        torch.cuda.current_stream().cuda_stream), 'pa_rows_low')
    want = x * 0.75
    assert torch.equal(low[:n, :3], (want - want.half().float()).half())
    assert not bool(low[n:].any()) and not bool(low[:, 3].any())


def test_walk_takes_any_number_of_nodes():
    lib = _lib.lib()
    assert lib.pa_graph_reach(None, None, None, ROWS, 8, 0, 6, None) == -1
    assert lib.pa_graph_reach(None, None, None, ROWS, 0, 0, 6, None) == -2


@pytest.mark.gpu
@pytest.mark.parametrize('n', [(1 << 22) + 1, ROWS + 5])
@pytest.mark.parametrize('reverse', [False, True])
def test_walk_over_several_launches(n, reverse, device):
    """A chain that jumps between the nodes of the first launch and those of the
    last, in either direction."""
    print('walk over', n, reverse, flush=True)
    chain = torch.tensor([3, n - 1, 0, n - 2, 1 << 21, 7, n - 3, (1 << 21) - 1])
    adj = torch.full((n, 1), -1, dtype=torch.long, device=device)
    adj[chain[:-1].to(device), 0] = chain[1:].to(device)
    start = 3
    got = utils.reachable(adj, chain[start:start + 1].to(device), reverse=reverse)
    want = chain[:start + 1] if reverse else chain[start:]
    assert torch.equal(torch.nonzero(got).flatten().cpu(), want.sort().values)
