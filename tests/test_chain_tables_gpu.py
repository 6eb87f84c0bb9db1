"""Chained steps on both sides of the LDS limit of their tables: every table in LDS (up to
9 iterations of 512 rows, 4 of 1024), some of them in global memory, and more passes than
one sweep of the grid; against the chained __float128 oracle (the bar of test_chain_gpu.py)."""
import pytest

from test_chain_gpu import run_chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ub", [1, 0])
@pytest.mark.parametrize("N,K", [(128, 16), (200, 16), (496, 9), (496, 10), (496, 16), (1000, 4), (1000, 5), (1000, 16)])
def test_chain_table_limit(N, K, ub):
    run_chain(N, K, 0, ub, rt=0, multi=True, B=3)


@pytest.mark.parametrize("jw", [1, 2])
def test_chain_single_operators_past_the_limit(jw):
    run_chain(500, 12, jw, 1, rt=1, multi=True, B=3, izp=(1, 499), ozp=(3, 486))


def test_chain_many_systems():
    run_chain(20, 2, 0, 1, rt=0, multi=True, B=16391)
