"""Edges of the front kernels' splits: the trailing update's runs of tiles and
the big fronts' groups of 16 right-hand sides with the solution as its flag."""
import numpy as np
import pytest

from spral_amd import matrices, ssids
from helpers import analyse, rhs
from test_gpu_parity import gpu_factor, gpu_solve
from test_gpu_pivot_block import block
from test_oracle_app import dense_lower

pytestmark = pytest.mark.gpu

RAW_TOL = 1e-13


@pytest.mark.parametrize("n", [127, 128, 129, 191, 193, 320, 2200])
def test_update_runs(lib, n):
    """Trailing panels of one tile, of whole and ragged tiles, and of more
    tiles than a front's 512 workgroups (2,200 columns: 595)."""
    print(f"update runs n={n}", flush=True)
    m = dense_lower(block(n, "dominant"))
    ak, _ = analyse(m, use_gpu=True)
    _, b = rhs(m, 1, 5)
    for posdef in (False, True):
        fk, inf = ssids.ssids_factor(posdef, m.val, ak, ssids.SSIDSOptions())
        assert inf.flag >= 0
        x = b.copy()
        assert ssids.ssids_solve(x, ak, fk, ssids.SSIDSOptions()).flag >= 0
        assert matrices.bwd_error(m.full, x, b).max() <= RAW_TOL
        ssids.ssids_free(None, fk)
    ssids.ssids_free(ak)


@pytest.mark.parametrize("n,nrhs", [(257, 4), (300, 5), (320, 16), (321, 17), (700, 64),
                                    (700, 70)])
def test_big_front_groups(lib, n, nrhs):
    """Every group's columns equal the single-right-hand-side solve's bit for
    bit; a column holding NaNs (among them the bits that mark an entry as not
    yet published) ends as NaN and changes no other column."""
    print(f"big front groups n={n} nrhs={nrhs}", flush=True)
    m = dense_lower(block(n, "dominant"))
    ak, fk, _, opts = gpu_factor(m)
    _, b = rhs(m, nrhs, 6)
    x = gpu_solve(ak, fk, opts, b)
    assert matrices.bwd_error(m.full, x, b).max() <= RAW_TOL
    for k in range(0, nrhs, 7):
        assert np.array_equal(gpu_solve(ak, fk, opts, b[:, k]), x[:, k]), k
    bad = b.copy()
    bad[:, 1] = np.uint64(0x7ff85e7b19c3d24a).view(np.float64)
    bad[::3, 2] = np.inf
    y = gpu_solve(ak, fk, opts, bad)
    assert np.isnan(y[:, 1]).all() and not np.isfinite(y[:, 2]).any()
    keep = [k for k in range(nrhs) if k not in (1, 2)]
    assert np.array_equal(y[:, keep], x[:, keep])
    ssids.ssids_free(ak, fk)
