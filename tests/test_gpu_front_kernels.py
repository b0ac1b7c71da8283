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


@pytest.mark.parametrize("n", [1, 63, 64, 65, 130, 256])
def test_front_groups(lib, n):
    """Triangles of up to 256 columns: one right-hand side, groups of four and
    of 16 give the same columns bit for bit."""
    m = dense_lower(block(n, "dominant"))
    ak, fk, _, opts = gpu_factor(m)
    _, b = rhs(m, 2100, 7)
    ref = np.stack([gpu_solve(ak, fk, opts, b[:, k]) for k in range(17)], axis=1)
    assert matrices.bwd_error(m.full, ref, b[:, :17]).max() <= RAW_TOL
    for nrhs in (2, 4, 5, 16, 17, 2100):    # past 2,048 one front's groups are of 16
        x = gpu_solve(ak, fk, opts, b[:, :nrhs])
        k = min(nrhs, 17)
        assert np.array_equal(x[:, :k], ref[:, :k]), nrhs
        if nrhs == 2100:
            assert matrices.bwd_error(m.full, x, b).max() <= RAW_TOL
    ssids.ssids_free(ak, fk)


@pytest.mark.parametrize("nrhs", [2, 5, 33])
def test_grid_groups(lib, nrhs):
    """A 14 x 13 x 11 stencil and a KKT system with delayed pivots (columns
    between the eliminated ones and the rows): every level's kernels, whole and
    ragged row blocks, against single-right-hand-side solves and jobs."""
    for m in (matrices.laplace3d(14, 13, 11, diag=5.7), matrices.kkt_laplace(grid=8, m_con=100)):
        ak, fk, _, opts = gpu_factor(m)
        _, b = rhs(m, nrhs, 8)
        x = gpu_solve(ak, fk, opts, b)
        assert matrices.bwd_error(m.full, x, b).max() <= RAW_TOL
        for k in (0, nrhs - 1):
            assert np.array_equal(gpu_solve(ak, fk, opts, b[:, k]), x[:, k]), k
        y = gpu_solve(ak, fk, opts, b, job=ssids.SSIDS_SOLVE_JOB_FWD)
        y = gpu_solve(ak, fk, opts, y, job=ssids.SSIDS_SOLVE_JOB_DIAG_BWD)
        assert np.allclose(y, x, rtol=1e-12, atol=1e-12)
        ssids.ssids_free(ak, fk)


@pytest.mark.parametrize("n,weak", [(2944, ()), (2945, (0, 192)), (3001, (0, 1, 2, 704))])
def test_update_beside_pivot_block(lib, monkeypatch, n, weak):
    """Trailing updates split around the next pivot block (over 1,024 tiles at
    the first steps) give the level-by-level path's bits, with whole blocks and
    with blocks whose columns fail (a diagonal block of 1e-6 entries)."""
    print(f"update beside pivot block n={n} weak={weak}", flush=True)
    rng = np.random.default_rng(n)
    a = rng.uniform(-1.0, 1.0, (n, n))
    a = np.tril(a) + np.tril(a, -1).T + np.diag(rng.choice([-80.0, 80.0], n))
    for k in weak:
        a[k:k + 64, k:k + 64] *= 1e-6
    m = dense_lower(a)
    ak, _ = analyse(m, use_gpu=True)
    _, b = rhs(m, 1, 8)
    got = []
    for env in ("0", "1"):
        monkeypatch.setenv("SPRAL_SSIDS_HIP_NO_PLAN", env)
        fk, inf = ssids.ssids_factor(False, m.val, ak, ssids.SSIDSOptions())
        assert inf.flag >= 0
        x = b.copy()
        assert ssids.ssids_solve(x, ak, fk, ssids.SSIDSOptions()).flag >= 0
        got.append((x, inf.num_neg, inf.num_two, inf.not_first_pass, inf.not_second_pass))
        ssids.ssids_free(None, fk)
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1:] == got[1][1:]
    assert matrices.bwd_error(m.full, got[0][0], b).max() <= 1e-12
    assert (got[0][3] > 0) == bool(weak)
    ssids.ssids_free(ak)
