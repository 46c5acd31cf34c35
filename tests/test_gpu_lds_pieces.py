"""Visited bits in LDS are for launches whose queries all run at once, as the
hardware counts: LDS comes in pieces of 1280 bytes.  And the wavefronts a SIMD that
long lists keep on rows of a length without a kernel of its own."""
import ctypes

import pytest

from pilotann_amd import _lib

pytestmark = pytest.mark.gpu

PIECE, LDS, CUS = 1280, 160 * 1024, 256


@pytest.mark.parametrize('n,dp,ef_total,own', [
    # own: bytes of LDS of the kernel itself (lists, candidates, query)
    (50_000, 64, 512, 7008), (75_000, 64, 256, 2912), (90_000, 64, 256, 2912),
    (100_000, 64, 256, 2912), (200_000, 128, 32, 1616), (60_000, 32, 1024, 15_072),
    (250_000, 128, 128, 2128), (1_000_000, 64, 256, 2912),
])
def test_queries_at_once(n, dp, ef_total, own, device):
    form = ctypes.c_int()

    def near(batch):
        _lib.check(_lib.lib().pa_traverse_form(n, batch, 0, dp, ef_total, ctypes.byref(form)),
                   'pa_traverse_form')
        return form.value
    bits = -(-n // (32 * 256)) * 256 * 4
    fit = LDS // (-(-(bits + own) // PIECE) * PIECE)
    assert near(fit * CUS) == 1
    assert near(fit * CUS + 1) == 0


# (lists of 4096 cells: LDS, 14 640 bytes and the query, holds 9 with 200 floats and 10
# with fewer)
@pytest.mark.parametrize('dp', [8, 40, 96, 200])
@pytest.mark.parametrize('ef_total,per_cu', [(384, 16), (512, 16), (2048, 9)])
def test_queries_of_other_row_lengths_at_once(ef_total, per_cu, dp, device):
    slots = ctypes.c_int()
    _lib.check(_lib.lib().pa_traverse_plan(1_000_000, 1 << 20, dp, ef_total,
                                           ctypes.byref(slots), None), 'pa_traverse_plan')
    assert slots.value >= per_cu * CUS
