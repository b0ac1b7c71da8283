"""The pivot block on its own: dense fronts of at most one or two 64-column
blocks against the oracle's restatement, at the widths where the block's
split (16 columns a wave, 16 x 16 blocks of its inverse) can go wrong, with
values that reach every branch of the search.

Within one block every product is an explicit fma, so the pivot order equals
the oracle's even where exact ties decide it; L and D agree to 1e-12 of the
largest entry (they differ at most by the rounding of the reciprocals)."""
import numpy as np
import pytest

from oracle.oracle_py import OracleFactor
from spral_amd import matrices, ssids
from helpers import analyse, rhs
from test_gpu_app_parity import node_factors
from test_oracle_app import dense_lower

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def block(n, kind, seed=7):
    rng = np.random.default_rng(seed + n)
    a = np.tril(rng.uniform(-1, 1, (n, n)))
    if kind == "ties":          # equal magnitudes decide by column, then row
        a = np.tril(rng.integers(-2, 3, (n, n)).astype(float))
        a[np.arange(n), np.arange(n)] += np.where(np.arange(n) % 3 == 0, 0.0, 4.0)
    elif kind == "offdiag":     # zero diagonal: every pivot off the diagonal
        a[np.arange(n), np.arange(n)] = 0.0
    elif kind == "dominant":
        a[np.arange(n), np.arange(n)] += n + 2.0
    elif kind == "highword":    # maxima that differ in the low word only
        a[np.arange(n), np.arange(n)] = 8.0 * n * (1 + 2.0 ** -40 * rng.integers(0, 9, n))
    return a + np.tril(a, -1).T


@pytest.mark.parametrize("kind", ["ties", "offdiag", "dominant", "highword"])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 48, 49, 63, 64])
def test_block_matches_oracle(lib, oracle_lib, n, kind):
    print(f"pivot block n={n} kind={kind}", flush=True)
    m = dense_lower(block(n, kind))
    ak, inf = analyse(m, use_gpu=True)
    assert inf.flag >= 0 and ak.nnodes == 1
    fk, finf = ssids.ssids_factor(False, m.val, ak, ssids.SSIDSOptions())
    of = OracleFactor(ak, m.val, app=True)
    g, o = node_factors(fk, 0), of.node_factors(0)
    assert g["nelim"] == o["nelim"]
    ne = g["nelim"]
    assert np.array_equal(g["perm"], o["perm"])
    Lg, Lo = np.tril(g["L"][:, :ne]), np.tril(o["L"][:, :ne])
    assert np.abs(Lg - Lo).max(initial=0) <= RTOL * max(1.0, np.abs(Lo).max(initial=0))
    Dg, Do = g["D"][:2 * ne], o["D"][:2 * ne]
    f = np.isfinite(Do)
    assert np.array_equal(f, np.isfinite(Dg))
    assert np.allclose(Dg[f], Do[f], rtol=RTOL, atol=0)
    for k in ("num_neg", "num_two", "matrix_rank"):
        assert getattr(finf, k) == of.stats[k], k
    ssids.ssids_free(ak, fk)


@pytest.mark.parametrize("n", [3, 40, 100])
def test_block_below_small_is_zero_pivots(lib, n):
    """Subnormal values (and values below `small`) end the block: every
    remaining index a zero pivot, rank 0."""
    for scale in (1e-312, 1e-30):
        m = dense_lower(block(n, "offdiag") * scale)
        ak, _ = analyse(m, use_gpu=True)
        fk, inf = ssids.ssids_factor(False, m.val, ak, ssids.SSIDSOptions())
        assert inf.flag == 7 and inf.matrix_rank == 0
        ssids.ssids_free(ak, fk)


@pytest.mark.parametrize("n", [1, 16, 33, 64, 65, 130])
def test_inverse_blocks_solve(lib, n):
    """Rows below the block go through its inverse: solves of dense fronts
    wider and narrower than a block reach the kernel tests' 1e-13."""
    m = dense_lower(block(2 * n + 1, "dominant"))
    ak, _ = analyse(m, use_gpu=True)
    for posdef in (False, True):
        fk, inf = ssids.ssids_factor(posdef, m.val, ak, ssids.SSIDSOptions())
        assert inf.flag >= 0
        _, b = rhs(m, 1, 3)
        x = b.copy()
        assert ssids.ssids_solve(x, ak, fk, ssids.SSIDSOptions()).flag >= 0
        assert matrices.bwd_error(m.full, x, b).max() <= 1e-13
        ssids.ssids_free(None, fk)
    ssids.ssids_free(ak)
