"""Threshold partial pivoting at the edges of its kernel: batches of candidates,
pivot columns in LDS or not, deferred row swaps in one, two and four columns a
wave or none, fronts of narrow levels."""
import numpy as np
import pytest

from oracle.oracle_py import OracleFactor
from spral_amd import matrices, ssids
from helpers import analyse, brute_inertia, rhs
from test_gpu_app_parity import node_factors
from test_gpu_pivot_block import block
from test_oracle_app import dense_lower

pytestmark = pytest.mark.gpu


def check(m, **kw):
    """Inertia by eigenvalues; a refined solve reaches 1e-14 (refinement would
    not converge on factors with a misplaced row)."""
    ak, inf = analyse(m, use_gpu=True, **kw)
    assert inf.flag >= 0
    opts = ssids.SSIDSOptions(**kw)
    fk, finf = ssids.ssids_factor(False, m.val, ak, opts)
    assert finf.flag >= 0
    assert finf.num_neg == brute_inertia(m)[0]
    _, b = rhs(m, 1, 4)
    x = b.copy()
    inf, bwd, its = ssids.ssids_solve_refine(x, ak, fk, opts)
    assert inf.flag >= 0 and bwd.max() <= 1e-14, (bwd, its)
    return ak, fk, finf


@pytest.mark.parametrize("kind", ["ties", "offdiag"])
@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 18, 64, 65, 129, 300])
def test_whole_front(lib, oracle_lib, n, kind):
    """The pivot sequence of a front pivoted by TPP throughout is the oracle's."""
    print(f"tpp n={n} kind={kind}", flush=True)
    m = dense_lower(block(n, kind))
    ak, _ = analyse(m, use_gpu=True, pivot_method=3)
    fk, inf = ssids.ssids_factor(False, m.val, ak, ssids.SSIDSOptions(pivot_method=3))
    of = OracleFactor(ak, m.val)
    g, o = node_factors(fk, 0), of.node_factors(0)
    assert g["nelim"] == o["nelim"]
    assert np.array_equal(g["perm"], o["perm"])
    ssids.ssids_free(ak, fk)


@pytest.mark.parametrize("n", [1030, 2100])
def test_long_columns(lib, n):
    """More columns than the deferred swaps hold, and more rows than LDS does."""
    print(f"tpp long n={n}", flush=True)
    ak, fk, _ = check(dense_lower(block(n, "offdiag")), pivot_method=3)
    ssids.ssids_free(ak, fk)


@pytest.mark.parametrize("n", [200, 500, 900, 1400])
def test_remainders(lib, n):
    """Columns that blocks of 64 left at u = 0.5 behind eliminated ones: up to
    256, 512 and 1,024 of them."""
    print(f"tpp remainder n={n}", flush=True)
    ak, fk, inf = check(dense_lower(block(n, "offdiag")), u=0.5)
    print(f"  left by the blocks: {inf.not_first_pass} of {n}", flush=True)
    assert inf.not_first_pass > n // 4
    ssids.ssids_free(ak, fk)


def test_narrow_workgroups(lib):
    """A level of more than 256 fronts (four waves each)."""
    m = matrices.kkt_laplace(grid=12, m_con=200)
    ak, fk, _ = check(m, pivot_method=3)
    ssids.ssids_free(ak, fk)
