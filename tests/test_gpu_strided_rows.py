"""Rows that are not laid out one after the other: a set of half-precision rows
takes their second part from any view of them."""
import pytest
import torch

from pilotann_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('form', ['columns', 'transposed', 'every other', 'double', 'more rows'])
@pytest.mark.parametrize('n', [0, 300, (1 << 20) + 3])
def test_second_part_of_views(form, n, device):
    print('second part', form, n, flush=True)
    d = 8
    g = torch.Generator(device=device).manual_seed(n + 1)
    x = torch.randn(n, d, device=device, generator=g)
    rows = kernels.HalfRows(x)
    want = rows.low(x)
    scaled = x * rows.scale
    assert torch.equal(want[:n, :d], (scaled - scaled.half().float()).half())
    view = {'columns': lambda: torch.cat([x, x + 1], 1)[:, :d],
            'transposed': lambda: x.T.contiguous().T,
            'every other': lambda: torch.stack([x, x + 1], 1).flatten(0, 1)[::2],
            'double': lambda: x.double(),
            'more rows': lambda: torch.cat([x, x.new_ones(5, d)])}[form]()
    assert torch.equal(rows.low(view), want)
    assert not bool(want[n:].any()) and not bool(want[:, d:].any())


def test_refused(device):
    x = torch.randn(300, 8, device=device)
    rows = kernels.HalfRows(x)
    for wrong in (x[:200], x[:, :4], x.cpu(), x[0]):
        with pytest.raises(RuntimeError):
            rows.low(wrong)
