"""The refine on rows whose query takes nearly all of a compute unit's LDS: a few
queries, for which the form with slots for helpers (4 KB more) does not fit and the
ones without do, against the oracle."""
import pytest

from common import Problem, assert_same_search
from test_gpu_refine import candidates, run_both

pytestmark = pytest.mark.gpu

LDS = 160 * 1024


# own: bytes of LDS of the forms without helpers, and of the one with
@pytest.mark.parametrize('ef_search,d,own,own_ahead', [
    (8, 38_128, 9232, 13_392), (128, 38_000, 9744, 13_904), (2048, 31_080, 37_408, 41_568)])
def test_rows_that_fit_without_helpers(ef_search, d, own, own_ahead, device):
    groups = d // 8
    query = 32 * (groups + 2 + groups % 2)
    assert query + own <= LDS < query + own_ahead
    print('longest rows', ef_search, d, flush=True)
    dp, k = 32, 10
    p = Problem(n=300, d=d, deg=16, sample_ratio=0.5, seed=ef_search, n_query=5)
    cand_I, cand_D = candidates(p, dp, min(ef_search, 64), 16, device)
    got, ref = run_both(p, dp, ef_search, k, cand_I, cand_D, device)
    assert_same_search(got['buf_I'], got['buf_D'], ref['buf_I'], ref['buf_D'])
    assert_same_search(got['out_I'], got['out_D'], ref['out_I'], ref['out_D'])
