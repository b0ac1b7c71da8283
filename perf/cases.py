"""The work that users of this package have it do, as measurable cases.

A case is a sparse symmetric system and what is asked of it:

* ``refactor``: new values on a resident pattern (host arrays), then a solve;
* ``fresh``: a factorization on a new handle, a solve, and the handle freed
  (a loop of single calls on an analysed pattern);
* ``device``: the resident path: values and right-hand sides in HBM,
  refactor and a solve refined to a backward error of 1e-14;
* ``solve``: a refined solve on resident factors, buffers in HBM;
* ``jobs``: the forward and the diagonal + backward solve as separate calls
  on host arrays (SSIDS jobs 1 and 4), on resident factors;
* ``batch``: many independent systems factored and solved in one call.

Systems: ``lap`` a 7-point stencil with varying couplings on an nx*ny*nz grid
(nested dissection), shifted to be indefinite or, with ``posdef``, positive
definite; ``kkt`` a saddle-point system with a 7-point H; ``kkt27`` one with a
27-point H; ``kktr`` one with a random sparse H (the batched systems).
``barrier`` adds log-uniform terms of that many decades either way to H's
diagonal, as an interior-point method does between factorizations.
Right-hand sides are A x_true with x_true uniform in [-1, 1].
"""
import ctypes as C
import math

import numpy as np
import torch

from spral_amd import _lib, batch, matrices, ssids


# --------------------------------------------------------------------------
# cases
# --------------------------------------------------------------------------
def _case(do, matrix, nx, ny=0, nz=0, nrhs=1, ordering=4, scaling=0, refine=True,
          posdef=False, mixed=False, barrier=0, count=1):
    return {"do": do, "matrix": matrix, "nx": nx, "ny": ny, "nz": nz, "nrhs": nrhs,
            "ordering": ordering, "scaling": scaling, "refine": refine, "posdef": posdef,
            "mixed": mixed, "barrier": barrier, "count": count}


def listed():
    cases = [
        # the smallest system of the batched workload on its own: an
        # optimisation loop that refactors a tiny KKT system; latency
        ("tiny_kkt_200", _case("refactor", "kktr", 200, refine=False)),
        # one ordinary system a call, new handle each time
        ("fresh_kkt_1500", _case("fresh", "kktr", 1500, ordering=2, scaling=3)),
        # a saddle-point system of 5,120 unknowns (H indefinite itself)
        ("kkt16_refactor", _case("refactor", "kkt", 16, 16, 16, nrhs=4)),
        # an interior-point step of a solver service: barrier terms far from
        # the values the order was computed from (failed and delayed pivots),
        # the matching scaling of the new values
        ("kkt20_barrier", _case("refactor", "kkt", 20, 20, 20, ordering=2, scaling=1,
                                barrier=3)),
        # a ragged grid, several right-hand sides, norm equilibration
        ("lap_37x29x23", _case("refactor", "lap", 37, 29, 23, nrhs=3, ordering=3, scaling=4,
                               refine=False)),
        # Cholesky-like factorization and its diagonal (a log-determinant)
        ("posdef_40", _case("refactor", "lap", 40, 40, 40, ordering=3, posdef=True,
                            refine=False)),
        # the headline: 64^3 stencil resident in HBM
        ("lap64_device", _case("device", "lap", 64, 64, 64, ordering=3)),
        # mixed precision on the densest fronts: 27-point KKT
        ("kkt27_32_mixed", _case("device", "kkt27", 32, 32, 32, ordering=2, scaling=3,
                                 mixed=True)),
        # solves on resident factors: one right-hand side and a full block
        ("solve64_k1", _case("solve", "lap", 64, 64, 64, ordering=3)),
        ("solve48_k64", _case("solve", "lap", 48, 48, 48, nrhs=64, ordering=3)),
        # forward and backward solves as separate jobs
        ("jobs_kkt16_k16", _case("jobs", "kkt", 16, 16, 16, nrhs=16)),
        # many systems of 200 to 5,000 unknowns at once
        ("batch_96", _case("batch", "kktr", 200, 5000, ordering=2, scaling=3, refine=False,
                           count=96)),
    ]
    return [dict(c, name=name) for name, c in cases]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    do = rng.choice(["refactor", "refactor", "fresh", "device", "solve", "jobs", "batch"])
    nrhs = rng.choice([1, 1, 2, 4, 7, 16, 33, 64]) if do in ("solve", "jobs") \
        else rng.choice([1, 1, 1, 2, 4, 5])
    if do == "batch":
        return _case("batch", "kktr", 200, _log_int(rng, 400, 5000),
                     ordering=rng.choice([2, 4]), scaling=0, refine=False,
                     count=_log_int(rng, 4, 80))
    matrix = rng.choice(["lap", "lap", "kkt", "kkt27", "kktr"])
    if do == "fresh":
        matrix = rng.choice(["lap", "kktr"])
    if matrix == "kktr":
        return _case(do, "kktr", _log_int(rng, 200, 5000), nrhs=nrhs,
                     ordering=rng.choice([2, 4]), refine=rng.random() < 0.5)
    hi = {"lap": 52, "kkt": 24, "kkt27": 24}[matrix]
    if do == "fresh":
        hi = 32
    nx, ny, nz = (_log_int(rng, 6, hi) for _ in range(3))
    if matrix == "lap":
        posdef = do in ("refactor", "device") and rng.random() < 0.3
        return _case(do, "lap", nx, ny, nz, nrhs=nrhs, ordering=3, posdef=posdef,
                     scaling=4 if do == "refactor" and rng.random() < 0.3 else 0,
                     mixed=do == "device" and not posdef and rng.random() < 0.3,
                     refine=rng.random() < 0.5)
    ordering = rng.choice([2, 4])
    return _case(do, matrix, nx, nx, nx, nrhs=nrhs, ordering=ordering,
                 scaling=3 if ordering == 2 else 0,
                 mixed=do == "device" and rng.random() < 0.3,
                 barrier=2 if do == "refactor" and matrix == "kkt" else 0)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
class _Matrix:
    """Lower-triangle CSC (1-based) with the values to factor, and the values
    the pattern was analysed with."""

    def __init__(self, n, ptr, row, val):
        self.n = n
        self.ptr = np.ascontiguousarray(ptr, np.int64)
        self.row = np.ascontiguousarray(row, np.int32)
        self.val = np.ascontiguousarray(val, np.float64)
        self.col = np.repeat(np.arange(n), np.diff(self.ptr))
        self.analysed = self.val

    def times(self, x):
        """A x for x (n, k)."""
        r, c = self.row - 1, self.col
        off = r != c
        y = np.empty_like(x)
        for j in range(x.shape[1]):
            y[:, j] = np.bincount(r, self.val * x[c, j], self.n) + \
                np.bincount(c[off], self.val[off] * x[r[off], j], self.n)
        return y


def _system(case, rng, seed):
    """One system of the case's kind (not "batch")."""
    kind, nx, ny, nz = case["matrix"], case["nx"], case["ny"], case["nz"]
    if kind == "lap":
        s = matrices.laplace3d(nx, ny, nz)
        m = _Matrix(s.n, s.ptr, s.row, s.val)
        r, c = m.row - 1, m.col
        off = r != c
        v = np.empty(m.val.size)
        v[off] = -rng.uniform(0.8, 1.25, int(off.sum()))
        total = np.bincount(r[off], -v[off], m.n) + np.bincount(c[off], -v[off], m.n)
        # a shifted operator, indefinite on grids of more than a few points;
        # the positive-definite one has a reaction term instead
        v[~off] = total[r[~off]] + (0.05 if case["posdef"] else -0.3)
        m.val = m.analysed = v
        return m
    if kind == "kktr":
        s = matrices.kkt_random(nx, seed=matrices.SEED_BASE + seed)
        return _Matrix(s.n, s.ptr, s.row, s.val)
    g = nx
    if kind == "kkt27":
        s = matrices.kkt_stencil27(g, max(1, g ** 3 * 88000 // 512000),
                                   seed=matrices.SEED_BASE + seed)
    else:
        s = matrices.kkt_laplace(grid=g, m_con=max(1, g ** 3 // (4 if g <= 16 else 8)),
                                 seed=matrices.SEED_BASE + seed)
    m = _Matrix(s.n, s.ptr, s.row, s.val)
    if case["barrier"]:
        d = np.nonzero((m.row - 1 == m.col) & (m.col < g ** 3))[0]
        m.val = m.val.copy()
        m.val[d] += 10.0 ** rng.uniform(-case["barrier"], case["barrier"], d.size)
    return m


def _batch_sizes(case):
    """The orders of a batch's systems, the same for every seed."""
    lo, hi = math.log(case["nx"]), math.log(case["ny"])
    t = _rng(case["count"]).uniform(lo, hi, case["count"])
    return [int(round(math.exp(v))) for v in t]


def _batch(case, seed):
    mats = []
    for i, n in enumerate(_batch_sizes(case)):
        s = matrices.kkt_random(n, seed=matrices.SEED_BASE + 1000 * seed + i)
        mats.append(_Matrix(s.n, s.ptr, s.row, s.val))
    return mats


def _rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _options(case, use_gpu=True):
    return ssids.SSIDSOptions(ordering=case["ordering"], scaling=case["scaling"],
                              schur_precision=1 if case["mixed"] else 0, use_gpu=use_gpu)


def _analyse(case, m, opts):
    grid = (case["nx"], case["ny"], case["nz"]) if case["ordering"] == 3 else None
    ak, inf = ssids.ssids_analyse(False, m.n, m.ptr, m.row, opts, grid=grid, val=m.analysed)
    if inf.flag < 0:
        raise RuntimeError("analyse failed (%d)" % inf.flag)
    return ak


class _State:
    """What a program keeps between calls; freed with it."""
    ak = fk = numeric = batch = None

    def __del__(self):
        try:
            if self.numeric:
                _lib.lib().spral_ssids_hip_destroy_numeric(self.numeric)
            if self.batch is not None:
                batch.batch_free(self.batch)
            ssids.ssids_free(self.ak, self.fk)
        except Exception:
            pass


def _x_true(rng, n, k):
    return rng.uniform(-1.0, 1.0, (n, k))


def prepare(case, seed):
    rng = _rng(seed)
    s = _State()
    s.case = case
    s.opts = _options(case)
    if case["do"] == "batch":
        mats = _batch(case, seed)
        s.batch, inf = batch.batch_analyse(mats, s.opts)
        if inf.flag < 0:
            raise RuntimeError("analyse failed (%d)" % inf.flag)
        s.val = np.concatenate([m.val for m in mats])
        s.rhs = np.concatenate([m.times(_x_true(rng, m.n, 1))[:, 0] for m in mats])
        return s
    m = _system(case, rng, seed)
    s.n, s.val = m.n, m.val
    s.b = m.times(_x_true(rng, m.n, case["nrhs"]))
    s.ak = _analyse(case, m, s.opts)
    if case["do"] in ("refactor", "jobs"):
        s.fk, inf = ssids.ssids_factor(case["posdef"], m.analysed if case["do"] == "refactor"
                                       else m.val, s.ak, s.opts)
        if inf.flag < 0:
            raise RuntimeError("factorization failed (%d)" % inf.flag)
    elif case["do"] in ("device", "solve"):
        dev = torch.device("cuda:0")
        s.d_val = torch.from_numpy(m.val).to(dev)
        s.d_scale = None
        if s.ak.scaling is not None and case["scaling"] == 3:
            s.d_scale = torch.from_numpy(s.ak.scaling[s.ak.invp].copy()).to(dev)
        s.d_b = torch.from_numpy(np.ascontiguousarray(s.b[s.ak.invp].T)).to(dev)
        s.d_x = torch.zeros_like(s.d_b)
        s.bwd, s.its = np.zeros(case["nrhs"]), C.c_int(0)
        s.copt = s.opts.to_c()
        torch.cuda.synchronize()
        st = _lib.Stats()
        s.numeric = _lib.lib().spral_ssids_hip_factor_device(
            case["posdef"], s.ak.symbolic, s.d_val.data_ptr(), m.val.size, _ptr(s.d_scale),
            C.byref(s.copt), C.byref(st))
        if not s.numeric:
            raise RuntimeError("factorization failed (%d)" % st.flag)
    return s


def _ptr(t):
    return None if t is None else t.data_ptr()


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def _need(flag):
    if flag < 0:
        raise RuntimeError("call failed (%d)" % flag)


def _solve_device(s):
    _need(_lib.lib().spral_ssids_hip_solve_refine_device(
        s.numeric, s.case["nrhs"], s.d_b.data_ptr(), s.d_x.data_ptr(), s.n, 5, 1e-14, s.bwd,
        C.byref(s.its), None))
    return {"x": s.d_x}


def run(state):
    s = state
    case = s.case
    do = case["do"]
    if do == "solve":
        return _solve_device(s)
    if do == "device":
        st = _lib.Stats()
        _need(_lib.lib().spral_ssids_hip_refactor_device(
            s.numeric, s.d_val.data_ptr(), _ptr(s.d_scale), C.byref(s.copt), C.byref(st)))
        out = _solve_device(s)
        out["num_neg"], out["num_zero"] = int(st.num_neg), int(st.num_zero)
        return out
    if do == "batch":
        inf, neg, rank = batch.batch_factor(s.batch, s.val)
        _need(inf.flag)
        return {"x": batch.batch_solve(s.batch, s.rhs), "num_neg": neg, "rank": rank}
    x = s.b.copy()
    if do == "jobs":
        _need(ssids.ssids_solve(x, s.ak, s.fk, s.opts, job=ssids.SSIDS_SOLVE_JOB_FWD).flag)
        _need(ssids.ssids_solve(x, s.ak, s.fk, s.opts,
                                job=ssids.SSIDS_SOLVE_JOB_DIAG_BWD).flag)
        return {"x": x}
    if do == "refactor":
        s.fk, inf = ssids.ssids_factor(case["posdef"], s.val, s.ak, s.opts, fkeep=s.fk)
        fk = s.fk
    else:
        fk, inf = ssids.ssids_factor(case["posdef"], s.val, s.ak, s.opts)
    _need(inf.flag)
    if case["refine"]:
        sinf, bwd, its = ssids.ssids_solve_refine(x, s.ak, fk, s.opts)
    else:
        sinf = ssids.ssids_solve(x, s.ak, fk, s.opts)
    _need(sinf.flag)
    out = {"x": x, "num_neg": int(inf.num_neg), "rank": int(inf.matrix_rank)}
    if case["posdef"]:
        out["d"], dinf = ssids.ssids_enquire_posdef(s.ak, fk)
        _need(dinf.flag)
    if do == "fresh":
        ssids.ssids_free(fkeep=fk)
    return out


# --------------------------------------------------------------------------
# what a pass cannot do without, and what it should return
# --------------------------------------------------------------------------
def work(case):
    """Factorization: the analyse's flops; the values read and the factors
    written once.  Solve: 4 flops per factor entry and right-hand side, the
    factors read once in each direction.  One correction step of a refined
    solve is a second solve, needed only where the first misses the target,
    and is not counted."""
    rng = _rng(1)
    if case["do"] == "batch":
        mats, k = _batch(case, 1), 1
    else:
        mats, k = [_system(case, rng, 1)], case["nrhs"]
    opts = _options(dict(case, ordering=4) if case["ordering"] == 2 else case, use_gpu=False)
    nf = fl = nz = n = 0
    for m in mats:
        ak = _analyse(dict(case, ordering=opts.ordering), m, opts)
        nf, fl, nz, n = nf + ak.num_factor, fl + ak.num_flops, nz + m.val.size, n + m.n
    nbytes, flops = 2 * 8.0 * nf + 16.0 * n * k, 4.0 * nf * k
    if case["do"] not in ("solve", "jobs"):
        nbytes, flops = nbytes + 8.0 * nz + 8.0 * nf, flops + float(fl)
    return {"bytes": nbytes, "flops": flops}


def exact(case, seed):
    """x_true, the solution the right-hand sides were made from."""
    rng = _rng(seed)
    if case["do"] == "batch":
        mats = _batch(case, seed)
        return {"x": np.concatenate([_x_true(rng, m.n, 1)[:, 0] for m in mats]),
                "num_neg": None, "rank": None}
    m = _system(case, rng, seed)
    x = _x_true(rng, m.n, case["nrhs"])
    if case["do"] in ("device", "solve"):
        # in elimination order, a right-hand side a row
        opts = _options(case, use_gpu=False)
        ak = _analyse(case, m, opts)
        x = np.ascontiguousarray(x[ak.invp].T)
    out = {"x": x}
    if case["do"] != "solve" and case["do"] != "jobs":
        out["num_neg"] = None
        out["num_zero" if case["do"] == "device" else "rank"] = None
    if case["posdef"] and case["do"] != "device":
        out["d"] = None
    return out
