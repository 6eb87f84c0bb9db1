"""Chained steps whose last tables are read from global memory, whole tables into registers: both
directions of the recurrence, single operators, 8 and 16 rows per lane, and more pairs than one
sweep of the grid."""
import pytest

from test_chain_gpu import run_chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jw", [0, 1, 2])
@pytest.mark.parametrize("ub", [0, 1])
@pytest.mark.parametrize("N,K", [(300, 12), (490, 16), (900, 6), (1000, 16)])
def test_operators_past_the_limit(N, K, ub, jw):
    run_chain(N, K, jw, ub, rt=1, multi=True, B=5, izp=(1, N - 1), ozp=(2, N - K))


@pytest.mark.parametrize("N,K,B", [(400, 11, 4099), (700, 5, 2049)])
def test_several_sweeps(N, K, B):
    run_chain(N, K, 0, 1, rt=0, multi=True, B=B)
