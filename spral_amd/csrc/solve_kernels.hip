// Forward / diagonal / backward solve kernels over the resident factors.
//
// Positions of a front (after pivoting): [0, ne) eliminated, [ne, n) failed
// fully-summed columns passed on to the parent, [n, m) the rows below.  X
// (m x nrhs per front, ld m) holds the forward values of the front's positions;
// X and the backward partial sums live in the call's workspace ws (solve_X,
// solve_P).  Every kernel writes what it reads of ws earlier in the same
// solve, so ws needs no clearing between calls.
//
// Forward (levels leaves -> root), two launches per level:
//   k_fwd_tri : a workgroup per front (ne <= kBigTri) and group of right-hand
//               sides: X[0:n] = own b + the children's updates that land on
//               fully-summed positions, then the unit-lower triangle on
//               X[0:ne]; the eliminated values go to x by variable.
//   k_fwd_rows: 64-row workgroups over [ne, m): the children's updates that
//               land on the rows (summed in LDS in a fixed order) minus
//               L[rows, 0:ne] X[0:ne].  X[ne:m] is what the parent gathers.
// Backward (root -> leaves), two launches per level:
//   k_bwd_rows: 256-row workgroups over [ne, m) write partial sums of
//               L[rows, 0:ne]^T x[rows];
//   k_bwd_tri : a workgroup per front (ne <= kBigTri) and group of right-hand
//               sides: the partials reduced in workgroup order, then the
//               triangle with L11^T.
// Fronts with ne > kBigTri (separators at the top of the tree) take two
// launches per level for the same: their positions' values (k_big_fwd_init,
// k_big_bwd_init), 64 to a workgroup, and the triangle over 64-column blocks,
// the blocks of a front chained by their solutions (k_big_fwd_lvl,
// k_big_bwd_lvl).
// The products run on FP64 MFMA with the right-hand sides as the 16 output
// columns, in groups of 16, of four, or one; an output column depends on its
// own right-hand side alone, so every column is summed exactly as a
// single-right-hand-side solve sums it.
//
// Loads of L are issued together ahead of what they are multiplied with, with
// indices clamped into the block (or past a buffer's length, read as zero)
// instead of guarded, and the 64-step diagonal-block substitutions broadcast
// each solved value with a lane read.
// Reference semantics: src/ssids/cpu/NumericSubtree.hxx:286-406 and
// src/ssids/cpu/kernels/ldlt_app.cxx:2537-2589.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <cmath>

#include "dev.hpp"

namespace ssids_hip {

constexpr int kRows = 64;                  // rows per workgroup of the row kernels
constexpr int kGroups = kThreads / kRows;  // column groups (one wave each)
constexpr int kBigTri = 256;
constexpr int kTriCap = 1024;  // fully-summed positions gathered in LDS

// FP64 MFMA accumulators of the multi-right-hand-side products
typedef double mr_acc_t __attribute__((ext_vector_type(4)));
// independent accumulators per output (4-position step u goes to u % kMrSplit,
// the partial sums added in order at the end): 16 dependent MFMAs become
// 4 chains of 4
constexpr int kMrSplit = 4;
// right-hand sides a wave substitutes through a diagonal block together when
// there are more than four (independent chains of lane reads and FMAs in
// one instruction stream; each right-hand side keeps its own sequence)
constexpr int kDiagGroup = 4;

// A solution entry not yet published: a quiet NaN with a payload no operation
// makes.  An entry that came out as these bits (an input NaN's payload carried
// through) is published as another NaN.
constexpr unsigned long long kUnset = 0x7ff85e7b19c3d24aull;
__device__ inline bool is_unset(double v) {
  return (unsigned long long)__double_as_longlong(v) == kUnset;
}

// value of v in lane j (j uniform)
__device__ inline double bcast_lane(double v, int j) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, j);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), j);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Substitution through a diagonal block for G right-hand sides: lane i holds
// v[r] of row i (forward) or column i (backward) and takes part j (ascending
// forward, descending backward) from lane j; l[j] is lane i's factor for
// part j, zero where there is none.
template <bool FWD, int G>
__device__ inline void substitute(const double (&l)[kBlk], double (&v)[G]) {
#pragma unroll
  for (int jj = 0; jj < kBlk; ++jj) {
    const int j = FWD ? jj : kBlk - 1 - jj;
#pragma unroll
    for (int r = 0; r < G; ++r) v[r] = fma(-l[j], bcast_lane(v[r], j), v[r]);
  }
}

// The same with the block in LDS (lb[i][j] = L[j0+i, j0+j] below the diagonal,
// else 0), where a front's chain is short and registers would cost workgroups
template <bool FWD, int G>
__device__ inline void substitute_lds(const double (*lb)[kBlk + 1], int lane, double (&v)[G]) {
  constexpr int kPart = 16;  // factors read ahead of their use
  double l[2][kPart];
  auto read = [&](int p) {
#pragma unroll
    for (int k = 0; k < kPart; ++k) {
      const int jj = p * kPart + k, j = FWD ? jj : kBlk - 1 - jj;
      l[p & 1][k] = FWD ? lb[lane][j] : lb[j][lane];
    }
  };
  read(0);
#pragma unroll
  for (int p = 0; p < kBlk / kPart; ++p) {
    if (p + 1 < kBlk / kPart) read(p + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kPart; ++k) {
      const int jj = p * kPart + k, j = FWD ? jj : kBlk - 1 - jj;
#pragma unroll
      for (int r = 0; r < G; ++r) v[r] = fma(-l[p & 1][k], bcast_lane(v[r], j), v[r]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// l[j] = L[j0+lane, j0+j] for j < lane < wb, else 0: a lane's factors of the
// forward substitution
__device__ inline void load_rows(const double *L, int ldl, int j0, int wb, int lane,
                                 double (&l)[kBlk]) {
  const LoadBuffer<double> B(L + (size_t)j0 * ldl + j0, (int64_t)wb * ldl * 8);
#pragma unroll
  for (int j = 0; j < kBlk; ++j)
    l[j] = B((j < lane && lane < wb) ? (unsigned)(j * ldl + lane) * 8u : kNoLoad);
}

// A thread's part of the block L[j0:j0+wb, j0:j0+wb] below the diagonal (zeros
// elsewhere), coalesced, and its place in LDS: lb[i][j], from which the
// backward substitution reads columns
constexpr int kStage = kBlk * kBlk / kThreads;
__device__ inline void load_lower(const double *L, int ldl, int j0, int wb,
                                  double (&v)[kStage]) {
  ldl = fresh(ldl);
  const LoadBuffer<double> B(L + (size_t)j0 * ldl + j0, (int64_t)wb * ldl * 8);
#pragma unroll
  for (int it = 0; it < kStage; ++it) {
    const int i = threadIdx.x & (kBlk - 1), j = threadIdx.x / kBlk + it * kGroups;
    v[it] = B((j < i && i < wb) ? (unsigned)(j * ldl + i) * 8u : kNoLoad);
  }
}
__device__ inline void store_lower(const double (&v)[kStage], double (*lb)[kBlk + 1]) {
#pragma unroll
  for (int it = 0; it < kStage; ++it)
    lb[threadIdx.x & (kBlk - 1)][threadIdx.x / kBlk + it * kGroups] = v[it];
}

__device__ inline mr_acc_t mr_sum(const mr_acc_t (&a)[kMrSplit]) {
  mr_acc_t s;
#pragma unroll
  for (int rg = 0; rg < 4; ++rg) s[rg] = ((a[0][rg] + a[1][rg]) + a[2][rg]) + a[3][rg];
  return s;
}

// Right-hand sides of a front kernel's workgroup: one, or a group of up to
// kRhsGroup.  The latency of the chain (children, diagonal blocks, products)
// bounds these kernels, whatever the number of right-hand sides, so a group
// costs little more than one: the products of a block run on FP64 MFMA
// (rows or columns of the block by 16 right-hand sides) and the waves
// substitute four right-hand sides each.  One right-hand side and groups of
// four (a wave each) take the same steps on their columns, so a column is the
// same whatever nrhs.
// With a workgroup per right-hand side (lane products, one wave substituting)
// the 1,025 leaf fronts of a 48^3 stencil took 869 us forward with 64
// right-hand sides.
constexpr int kRhsGroup = 16, kRhsFew = 4;
constexpr int kRhsGroupsPar = 64;  // groups in parallel (gridDim.y)
// entries of one child a wave takes at a time
constexpr int kChildBatch = 4;

// ---- forward --------------------------------------------------------------
// One workgroup per front and group of NR right-hand sides.  X[0:n] = own b +
// the children's updates on fully-summed positions (children taken four at a
// time, a wave each, 256 entries of a child at a time; their adds applied wave
// by wave, so every position is summed in a fixed order), then the triangle
// X[0:ne] <- L11^{-1} X[0:ne] when ne <= kBigTri.
template <int NR>
__global__ __launch_bounds__(kThreads, 2) void k_fwd_tri(const SolveNode *sn, int s0,
                                                      const int *child_list, double *x,
                                                      int ldx, int nrhs, double *ws) {
  constexpr int kCap = (NR == 1) ? kTriCap : kBigTri, kLdx = kCap + 2;
  __shared__ double xs[NR][kLdx];
  __shared__ double lb[kBlk][kBlk + 1];
  __shared__ int nchunk[kGroups];
  const SolveNode &P = sn[s0 + blockIdx.x];
  const double *PL = P.L;
  gcint *Pperm = (gcint *)P.perm;
  gcint *Pipos = (gcint *)P.ipos;
  gcint *Prows = (gcint *)P.rows;
  gcint *Pctab = (gcint *)P.ctab;
  const int ldl = P.ldl, m = P.m, n = P.n, nd = P.nd, ne = P.nelim;
  const int cbeg = P.cbeg, cend = P.cend;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ri = lane & 15, kq = lane >> 4;
  if (ne > kBigTri) return;  // k_big_fwd_init and k_big_fwd_lvl
  const int T = idiv_up(m, 64), Tn = idiv_up(n, 64);
  // positions and right-hand sides of this thread in the loops over both: a
  // wave takes a right-hand side and a lane a position, or (NR = 1) a thread a
  // position
  const int p0 = (NR == 1) ? tid : lane, dp = (NR == 1) ? kThreads : 64;
  const int q0 = (NR == 1) ? 0 : wave;
  for (int rc = NR * blockIdx.y; rc < nrhs; rc += NR * gridDim.y) {
    const int nr = imin(NR, nrhs - rc);
    double *X = solve_X(ws, P, nrhs) + (size_t)rc * m;
    double *xr = x + (size_t)rc * ldx;
    double st[kStage];  // the first diagonal block, on its way during the gather
    if (ne > 0) load_lower(PL, ldl, 0, imin(kBlk, ne), st);
    const bool in_lds = n <= kCap;
    double *acc = in_lds ? &xs[0][0] : X;
    const size_t lda = in_lds ? (size_t)kLdx : (size_t)m;
    for (int p = p0; p < n; p += dp) {
      const int vrow = (p >= nd) ? Prows[p - nd] : -1, pos = Pipos[p];
#pragma unroll 4
      for (int q = q0; q < nr; q += kGroups)
        acc[q * lda + pos] = (vrow >= 0) ? xr[(size_t)q * ldx + vrow] : 0.0;
    }
    for (int c0 = cbeg; c0 < cend; c0 += kGroups) {
      const int ci = c0 + wave;
      int kb = 0, ke = 0, cn = 0, cne = 0, cdoff = 0, cm = 0;
      gcint *crmap = nullptr;
      gcdouble *cX = nullptr;
      if (ci < cend) {
        const SolveNode &c = sn[child_list[ci]];
        cn = c.n;
        cne = c.nelim;
        cdoff = c.doff;
        cm = c.m;
        crmap = (gcint *)c.rmap;
        cX = (gcdouble *)(solve_X(ws, c, nrhs) + (size_t)rc * cm);
        gcint *tab = Pctab + (size_t)(ci - cbeg) * (T + 1);
        kb = tab[0];
        ke = tab[Tn];
      }
      if (lane == 0) nchunk[wave] = idiv_up(ke - kb, 64 * kChildBatch);
      __syncthreads();
      const int nch = imax(imax(nchunk[0], nchunk[1]), imax(nchunk[2], nchunk[3]));
      __syncthreads();  // nchunk is rewritten by the next group
      for (int it = 0; it < nch; ++it) {
        int pos[kChildBatch], kk[kChildBatch];
#pragma unroll
        for (int h = 0; h < kChildBatch; ++h) {
          const int k = kb + (it * kChildBatch + h) * 64 + lane;
          kk[h] = imin(k, ke - 1);
          pos[h] = -1;
          if (k < ke) {
            const int pre = (k < cn) ? cdoff + (k - cne) : nd + crmap[k - cn];
            if (pre < n) pos[h] = Pipos[pre];
          }
        }
        constexpr int kQ = (NR == 1) ? 1 : 4;  // right-hand sides a round
        for (int q0 = 0; q0 < nr; q0 += kQ) {
          double val[kQ][kChildBatch];
#pragma unroll
          for (int q = 0; q < kQ; ++q)
#pragma unroll
            for (int h = 0; h < kChildBatch; ++h)
              val[q][h] = (pos[h] >= 0) ? cX[(size_t)imin(q0 + q, nr - 1) * cm + kk[h]] : 0.0;
          for (int w = 0; w < kGroups; ++w) {
            if (wave == w)
#pragma unroll
              for (int q = 0; q < kQ; ++q)
#pragma unroll
                for (int h = 0; h < kChildBatch; ++h)
                  if (pos[h] >= 0 && q0 + q < nr) acc[(q0 + q) * lda + pos[h]] += val[q][h];
            __syncthreads();
          }
        }
      }
    }
    if (ne > 0) store_lower(st, lb);
    __syncthreads();
    if (!in_lds) {
      for (int p = p0; p < ne; p += dp)
        for (int q = q0; q < nr; q += kGroups) xs[q][p] = X[(size_t)q * m + p];
      __syncthreads();
    }
    for (int j0 = 0; j0 < ne; j0 += kBlk) {
      const int j1 = imin(j0 + kBlk, ne), wb = j1 - j0;
      const int nrb = idiv_up(ne - j1, kBlk);  // 64-row blocks below, at most 3
      // the first's part of L, on its way during the substitution: the wave's
      // 16 rows (clamped), 4 columns a step
      double av[16];
      auto load_below = [&](int rb) {
        const int ld = fresh(ldl);
        const LoadBuffer<double> B(PL + (size_t)j0 * ld, (int64_t)kBlk * ld * 8);
        const unsigned off =
            (unsigned)(kq * ld + imin(j1 + 64 * rb + 16 * wave + ri, ne - 1)) * 8u;
#pragma unroll
        for (int u = 0; u < 16; ++u) av[u] = B(off, (unsigned)(4 * u * ld) * 8u);
      };
      if (nrb > 0) load_below(0);
      auto diag = [&](auto grp) {
        constexpr int G = decltype(grp)::value;
        double v[G];
#pragma unroll
        for (int r = 0; r < G; ++r)
          v[r] = (lane < wb) ? xs[imin(wave * G + r, NR - 1)][j0 + lane] : 0.0;
        substitute_lds<true, G>(lb, lane, v);
#pragma unroll
        for (int r = 0; r < G; ++r)
          if (lane < wb && wave * G + r < nr) xs[wave * G + r][j0 + lane] = v[r];
      };
      if (NR > kGroups && nr > kGroups) {
        diag(std::integral_constant<int, kDiagGroup>());
      } else if (wave < nr) {
        diag(std::integral_constant<int, 1>());
      }
      __syncthreads();
      if (j1 < ne) load_lower(PL, ldl, j1, imin(kBlk, ne - j1), st);
      double bv[16];
      if (nrb > 0) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          bv[u] = xs[imin(ri, NR - 1)][j0 + 4 * u + kq];
        }
      }
      for (int rb = 0; rb < nrb; ++rb) {
        mr_acc_t a[kMrSplit];
#pragma unroll
        for (int t = 0; t < kMrSplit; ++t) a[t] = (mr_acc_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int u = 0; u < 16; ++u)
          a[u % kMrSplit] =
              __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv[u], a[u % kMrSplit], 0, 0, 0);
        if (rb + 1 < nrb) load_below(rb + 1);
        const mr_acc_t s = mr_sum(a);
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const int row = j1 + 64 * rb + 16 * wave + kq + 4 * rg;
          if (row < ne && ri < NR) xs[ri][row] -= s[rg];
        }
      }
      if (j1 < ne) store_lower(st, lb);
      __syncthreads();
    }
    for (int p = p0; p < ne; p += dp) {
      const int var = Pperm[p];
#pragma unroll 4
      for (int q = q0; q < nr; q += kGroups) {
        const double v = xs[q][p];
        xr[(size_t)q * ldx + var] = v;
        X[(size_t)q * m + p] = v;
      }
    }
    if (in_lds)
      for (int p = ne + p0; p < n; p += dp)
        for (int q = q0; q < nr; q += kGroups) X[(size_t)q * m + p] = xs[q][p];
    __syncthreads();
  }
}

// 64-row workgroups over [ne, m) of every front of the level and groups of NR
// right-hand sides:
//   X[i] = (gathered fully-summed value, i < n) or (sum of the children's
//          updates on row i, i >= n)  -  L[i, 0:ne] X[0:ne]
// Of each 64 columns wave w takes columns 16w..16w+15 for the 64 rows (four
// 16-row MFMA outputs, so a right-hand side value serves four products); the
// waves' sums are added in wave order.  L is read once, in whole 512-byte
// column pieces, the next 64 columns under way during the current ones.
template <int NR>
__global__ __launch_bounds__(kThreads, NR == 1 ? 4 : 2) void k_fwd_rows(const SolveNode *sn, int s0,
                                                       const int *child_list,
                                                       const int *wg_off, int nlvl, int nrhs,
                                                       double *ws) {
  __shared__ double xs[NR][kRows];
  __shared__ double red[kGroups][NR][kRows + 2];
  int before;
  const int li = front_of(wg_off, nlvl, blockIdx.x, before);
  if (li < 0) return;
  const SolveNode &P = sn[s0 + li];
  const int ne = P.nelim, m = P.m;
  const int r0 = ne + (blockIdx.x - before) * kRows, r1 = imin(m, r0 + kRows);
  if (r0 >= r1) return;  // front without rows below
  const double *PL = P.L;
  gcint *Pctab = (gcint *)P.ctab;
  const int ldl = P.ldl, n = P.n, nd = P.nd, cbeg = P.cbeg, cend = P.cend;
  const int tid = threadIdx.x, lane = tid & 63, g = tid >> 6;
  const int ri = lane & 15, kq = lane >> 4;
  const int T = idiv_up(m, 64);
  const int lo = imax(r0, n), I0 = lo / 64, I1 = idiv_up(r1, 64);
  // this lane's row of each 16-row output (clamped) in its first column
  unsigned oa[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
    oa[t] = (unsigned)((16 * g + kq) * ldl + imin(r0 + 16 * t + ri, r1 - 1)) * 8u;
  for (int rc = NR * blockIdx.y; rc < nrhs; rc += NR * gridDim.y) {
    const int nr = imin(NR, nrhs - rc);
    gdouble *X = (gdouble *)(solve_X(ws, P, nrhs) + (size_t)rc * m);
    gdouble *Xq = X + (size_t)imin(ri, nr - 1) * m;
    // columns j0 + 16 g + 4 u + kq of L and of this lane's right-hand side
    auto load = [&](int j0, double (&av)[4][4], double (&bv)[4]) {
      // (columns past ne read as zero)
      const LoadBuffer<double> B(PL + (size_t)j0 * ldl, (int64_t)imin(64, ne - j0) * ldl * 8);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = j0 + 16 * g + 4 * u + kq;
#pragma unroll
        for (int t = 0; t < 4; ++t) av[t][u] = B(oa[t] + (unsigned)(4 * u * ldl) * 8u);
        bv[u] = masked(Xq[imin(j, ne - 1)], j < ne && ri < nr);
      }
    };
    double av[4][4], bv[4];
    if (ne > 0) load(0, av, bv);
    for (int idx = tid; idx < NR * kRows; idx += kThreads) {
      const int q = idx / kRows, i = idx % kRows, rw = r0 + i;
      xs[q][i] = (q < nr && rw < n && rw < r1) ? X[(size_t)q * m + rw] : 0.0;
    }
    __syncthreads();
    if (lo < r1) {
      // children four at a time (a wave each); a 64-row range holds at most
      // 128 positions, so at most two indices per lane
      for (int c0 = cbeg; c0 < cend; c0 += kGroups) {
        const int ci = c0 + g;
        int pos[2] = {-1, -1};
        double val[2][NR];
        if (ci < cend) {
          const SolveNode &c = sn[child_list[ci]];
          const int cn = c.n, cne = c.nelim, cdoff = c.doff, cm = c.m;
          gcint *crmap = (gcint *)c.rmap;
          gcdouble *cX = (gcdouble *)(solve_X(ws, c, nrhs) + (size_t)rc * cm);
          gcint *tab = Pctab + (size_t)(ci - cbeg) * (T + 1);
          const int kb = tab[I0], ke = tab[I1];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int k = kb + lane + 64 * h;
            if (k < ke) {
              const int pre = (k < cn) ? cdoff + (k - cne) : nd + crmap[k - cn];
              if (pre >= lo && pre < r1) {
                pos[h] = pre - r0;
#pragma unroll
                for (int q = 0; q < NR; ++q) val[h][q] = cX[(size_t)imin(q, nr - 1) * cm + k];
              }
            }
          }
        }
        for (int w = 0; w < kGroups; ++w) {
          if (g == w) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
              if (pos[h] >= 0) {
#pragma unroll
                for (int q = 0; q < NR; ++q) xs[q][pos[h]] += val[h][q];
              }
          }
          __syncthreads();
        }
      }
    }
    mr_acc_t acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = (mr_acc_t){0.0, 0.0, 0.0, 0.0};
    for (int j0 = 0; j0 < ne; j0 += 64) {
      double an[4][4], bn[4];
      if (NR > 1 && j0 + 64 < ne) load(j0 + 64, an, bn);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[t][u], bv[u], acc[t], 0, 0, 0);
      if constexpr (NR > 1) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          bv[u] = bn[u];
#pragma unroll
          for (int t = 0; t < 4; ++t) av[t][u] = an[t][u];
        }
      } else if (j0 + 64 < ne) {
        load(j0 + 64, av, bv);
      }
    }
    // element (row 16 t + kq + 4 rg, right-hand side ri)
    if (ri < NR) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) red[g][ri][16 * t + kq + 4 * rg] = acc[t][rg];
    }
    __syncthreads();
    for (int idx = tid; idx < NR * kRows; idx += kThreads) {
      const int q = idx / kRows, i = idx % kRows;
      if (q < nr && r0 + i < r1)
        X[(size_t)q * m + r0 + i] =
            xs[q][i] - (((red[0][q][i] + red[1][q][i]) + red[2][q][i]) + red[3][q][i]);
    }
    __syncthreads();
  }
}

// x = D^{-1} x over every front; half = 1 (positive definite, 1x1 pivots
// only): x = D^{-1/2} x
__global__ void k_dsolve(const SolveNode *sn, int nslots, double *x, int ldx, int nrhs,
                         int half) {
  const int s = blockIdx.x;
  if (s >= nslots) return;
  const SolveNode &P = sn[s];
  gcint *Pperm = (gcint *)P.perm;
  gcdouble *d = (gcdouble *)P.D;
  const int ne = P.nelim;
  for (int i = threadIdx.x; i < ne; i += blockDim.x) {
    bool first2 = (i + 1 < ne) && !isfinite(d[2 * i + 2]);
    bool second2 = !isfinite(d[2 * i]);
    for (int r = 0; r < nrhs; ++r) {
      double *xr = x + (size_t)r * ldx;
      if (half) {
        xr[Pperm[i]] *= sqrt(d[2 * i]);
      } else if (first2) {
        double x1 = xr[Pperm[i]], x2 = xr[Pperm[i + 1]];
        xr[Pperm[i]] = d[2 * i] * x1 + d[2 * i + 1] * x2;
        xr[Pperm[i + 1]] = d[2 * i + 1] * x1 + d[2 * i + 3] * x2;
      } else if (!second2) {
        xr[Pperm[i]] *= d[2 * i];
      }
    }
  }
}

// ---- backward -------------------------------------------------------------
// Workgroups over 256-row blocks of [ne, m) times kBwdCols-column chunks of
// [0, ne), for every front of the level:
// part[rb][r][j] = sum over row block rb's rows i of L[i, j] x[var(i), r].
// Each (rb, j) is written by exactly one workgroup, so the sums do not depend
// on the split.
// On FP64 MFMA for any number of right-hand sides (one kernel for every nrhs,
// so each column is the same whatever nrhs): wave w takes rows 64w..64w+63 for
// the 64 columns (four outputs of 16 columns by 16 right-hand sides, so a
// value of x serves four products) and the waves' sums are added in wave
// order.  Of the wave's rows lane quarter kq takes 16 kq..16 kq + 15, one a
// step, so a lane's loads of a column are 128 contiguous bytes; all of a
// wave's part of L is on its way before the variables of its rows are known.
// With a wave per 16 columns, stepping through the 256 rows in eight batches,
// each batch waited for its x: 19 us where 17 workgroups run (now 14), and
// with 64 right-hand sides 103 us for a level of 510 (now 75).
constexpr int kBwdCols = 64;
typedef double double2_u __attribute__((ext_vector_type(2), aligned(8)));
__global__ __launch_bounds__(kThreads, 2) void k_bwd_rows(const SolveNode *sn,
                                                             int s0,
                                                             const int *wg_off, int nlvl,
                                                             const double *x, int ldx, int nrhs,
                                                             double *ws) {
  constexpr int kSteps = 16;  // rows of a lane
  __shared__ double red[kGroups][kRhsGroup][kBwdCols + 2];
  int before;
  const int li = front_of(wg_off, nlvl, blockIdx.x, before);
  if (li < 0) return;
  const SolveNode &P = sn[s0 + li];
  gcint *Pperm = (gcint *)P.perm;
  gcint *Prows = (gcint *)P.rows;
  gdouble *part = (gdouble *)solve_P(ws, P, nrhs);  // count x nrhs x ne
  const int ldl = P.ldl, m = P.m, n = P.n, nd = P.nd, ne = P.nelim;
  const int nchunk = idiv_up(imax(ne, 1), kBwdCols);
  const int local_all = blockIdx.x - before;
  const int local = local_all / nchunk, chunk = local_all - local * nchunk;
  const int jbeg = chunk * kBwdCols, jend = imin(ne, jbeg + kBwdCols);
  const int r0 = ne + local * kThreads, r1 = imin(m, r0 + kThreads);
  if (jend <= jbeg || r1 <= r0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ri = lane & 15, kq = lane >> 4;
  const int i0 = r0 + 64 * wave;      // the wave's rows
  const bool whole = i0 + 64 <= r1;
  // A operand: this lane's column of each 16 (clamped), rows from 16 kq
  gcdouble *La[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
    La[t] = (gcdouble *)P.L + (size_t)imin(jbeg + 16 * t + ri, jend - 1) * ldl + i0 + 16 * kq;
  double av[4][kSteps];
  if (whole) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int u = 0; u < kSteps; u += 2) {
        const double2_u v = *(const double2_u __attribute__((address_space(1))) *)(La[t] + u);
        av[t][u] = v.x;
        av[t][u + 1] = v.y;
      }
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        const int i = i0 + 16 * kq + u;
        av[t][u] = masked(La[t][imin(i, r1 - 1) - i0 - 16 * kq], i < r1);
      }
  }
  int var[kSteps];  // variables of this lane's 16 rows (clamped)
#pragma unroll
  for (int u = 0; u < kSteps; ++u) {
    const int i = imin(i0 + 16 * kq + u, r1 - 1);
    var[u] = (i < n) ? Pperm[i] : Prows[i - nd];
  }
  for (int rc = kRhsGroup * blockIdx.y; rc < nrhs; rc += kRhsGroup * gridDim.y) {
    const int nr = imin(kRhsGroup, nrhs - rc);
    const double *xq = x + (size_t)(rc + imin(ri, nr - 1)) * ldx;
    double bv[kSteps];
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
      bv[u] = masked(xq[var[u]], ri < nr && i0 + 16 * kq + u < r1);
    mr_acc_t acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = (mr_acc_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[t][u], bv[u], acc[t], 0, 0, 0);
    // element (column 16 t + kq + 4 rg of the chunk, right-hand side ri)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) red[wave][ri][16 * t + kq + 4 * rg] = acc[t][rg];
    __syncthreads();
    for (int q = wave; q < nr; q += kGroups)
      if (jbeg + lane < jend)
        part[((size_t)local * nrhs + rc + q) * ne + jbeg + lane] =
            ((red[0][q][lane] + red[1][q][lane]) + red[2][q][lane]) + red[3][q][lane];
    __syncthreads();
  }
}

// Value of position j after x = D^{-1} x (the expressions of k_dsolve, so
// the result is the same whether the diagonal solve runs on its own or
// inside the backward solve)
__device__ inline double dinv_at(gcdouble *d, gcint *perm, const double *xr, int j, int ne) {
  const bool first2 = (j + 1 < ne) && !isfinite(d[2 * j + 2]);
  const bool second2 = !isfinite(d[2 * j]);
  if (first2) return d[2 * j] * xr[perm[j]] + d[2 * j + 1] * xr[perm[j + 1]];
  if (second2) return d[2 * j - 1] * xr[perm[j - 1]] + d[2 * j + 1] * xr[perm[j]];
  return xr[perm[j]] * d[2 * j];
}

// Sum of the row workgroups' partials at p: four sums, of every fourth
// workgroup, added in order
__device__ inline double part_sum(gcdouble *p, size_t stride, int count) {
  double s[kGroups];
#pragma unroll
  for (int k = 0; k < kGroups; ++k) s[k] = 0.0;
  for (int w = 0; w < count; w += kGroups)
#pragma unroll
    for (int k = 0; k < kGroups; ++k)
      s[k] += masked(p[(size_t)imin(w + k, count - 1) * stride], w + k < count);
  return ((s[0] + s[1]) + s[2]) + s[3];
}

// One workgroup per front (ne <= kBigTri) of the level and group of NR
// right-hand sides: X[j] = x[perm[j]] - sum of the row workgroups' partials, then the triangle
// L11^T X = X, 64-column blocks from the last, and x[perm[j]] = X[j].
template <int NR>
__global__ __launch_bounds__(kThreads, NR == 1 ? 3 : 2) void k_bwd_tri(const SolveNode *sn, int s0,
                                                      const int *wg_off, double *x, int ldx,
                                                      int nrhs, double *ws, int dfuse) {
  constexpr int kLdx = kBigTri + 2;
  __shared__ double xt[NR][kLdx];
  __shared__ double lb[kBlk][kBlk + 1];
  const int li = blockIdx.x;
  const SolveNode &P = sn[s0 + li];
  const double *PL = P.L;
  gcdouble *Pd = (gcdouble *)P.D;
  gcint *Pperm = (gcint *)P.perm;
  const int ldl = P.ldl, m = P.m, ne = P.nelim;
  const int count = wg_off[li + 1] - wg_off[li];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ri = lane & 15, kq = lane >> 4;
  if (ne > kBigTri) return;  // k_big_bwd_init and k_big_bwd_lvl
  const int p0 = (NR == 1) ? tid : lane, dp = (NR == 1) ? kThreads : 64;  // as k_fwd_tri
  const int q0 = (NR == 1) ? 0 : wave;
  for (int rc = NR * blockIdx.y; rc < nrhs; rc += NR * gridDim.y) {
    const int nr = imin(NR, nrhs - rc);
    gcdouble *part = (gcdouble *)(solve_P(ws, P, nrhs) + (size_t)rc * ne);
    double *xr = x + (size_t)rc * ldx;
    double st[kStage], av[16];
    // block b's part of L, on its way during the work before it: its own
    // block and the wave's 16 columns of the first 64 rows after it
    auto load_after = [&](int b, int rb) {
      const int j0 = b * kBlk, i0 = j0 + kBlk + 64 * rb, ld = fresh(ldl);
      const LoadBuffer<double> B(PL + (size_t)j0 * ld, (int64_t)kBlk * ld * 8);
      const unsigned off = (unsigned)((16 * wave + ri) * ld) * 8u;
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int i = i0 + 4 * u + kq;
        av[u] = B(i < ne ? off + (unsigned)i * 8u : kNoLoad);
      }
    };
    auto load = [&](int b) {
      load_lower(PL, ldl, b * kBlk, imin(kBlk, ne - b * kBlk), st);
      if ((b + 1) * kBlk < ne) load_after(b, 0);
    };
    const int nb = idiv_up(ne, kBlk);
    if (nb > 0) load(nb - 1);
    for (int j = p0; j < ne; j += dp)
      for (int q = q0; q < nr; q += kGroups) {
        double *xq = xr + (size_t)q * ldx;
        xt[q][j] = (dfuse ? dinv_at(Pd, Pperm, xq, j, ne) : xq[Pperm[j]]) -
                   part_sum(part + (size_t)q * ne + j, (size_t)nrhs * ne, count);
      }
    __syncthreads();
    for (int b = nb - 1; b >= 0; --b) {
      const int j0 = b * kBlk, wb = imin(kBlk, ne - j0), j1 = j0 + wb;
      store_lower(st, lb);
      // X[j] -= sum over the triangle's rows i in [j1, ne) of L[i, j] X[i]
      if (j1 < ne) {
        mr_acc_t a[kMrSplit];
#pragma unroll
        for (int t = 0; t < kMrSplit; ++t) a[t] = (mr_acc_t){0.0, 0.0, 0.0, 0.0};
        for (int rb = 0; j1 + 64 * rb < ne; ++rb) {
          if (rb > 0) load_after(b, rb);
#pragma unroll
          for (int u = 0; u < 16; ++u) {
            const int i = j1 + 64 * rb + 4 * u + kq;
            double bv = xt[imin(ri, NR - 1)][imin(i, ne - 1)];
            if (i >= ne) bv = 0.0;
            a[u % kMrSplit] =
                __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv, a[u % kMrSplit], 0, 0, 0);
          }
        }
        const mr_acc_t s = mr_sum(a);
        // (a block with rows after it is a whole one)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg)
          if (ri < NR) xt[ri][j0 + 16 * wave + kq + 4 * rg] -= s[rg];
      }
      __syncthreads();
      if (b > 0) load(b - 1);
      auto diag = [&](auto grp) {
        constexpr int G = decltype(grp)::value;
        double v[G];
#pragma unroll
        for (int r = 0; r < G; ++r)
          v[r] = (lane < wb) ? xt[imin(wave * G + r, NR - 1)][j0 + lane] : 0.0;
        substitute_lds<false, G>(lb, lane, v);
#pragma unroll
        for (int r = 0; r < G; ++r)
          if (lane < wb && wave * G + r < nr) xt[wave * G + r][j0 + lane] = v[r];
      };
      if (NR > kGroups && nr > kGroups) {
        diag(std::integral_constant<int, kDiagGroup>());
      } else if (wave < nr) {
        diag(std::integral_constant<int, 1>());
      }
      __syncthreads();
    }
    for (int j = p0; j < ne; j += dp) {
      const int var = Pperm[j];
#pragma unroll 4
      for (int q = q0; q < nr; q += kGroups) xr[(size_t)q * ldx + var] = xt[q][j];
    }
    __syncthreads();
  }
}

// ---- big fronts: one launch per tree level ---------------------------------
// Fronts with ne > kBigTri solve their triangle, L11 y = X[0:ne] (forward) or
// L11^T x = X[0:ne] (backward), in one launch per tree level over 64-column
// blocks: a workgroup per block of every big front of the level and per group
// of 16 right-hand sides (gridDim.y groups, up to kBigGroups).  Within a
// front and group, workgroups take their blocks by ticket (an atomic counter;
// forward in increasing, backward in decreasing block order), so a workgroup
// waits only for blocks whose workgroups took their tickets earlier and are
// running: every wait ends.  Block b's workgroup accumulates the products of
// the blocks it depends on in block order (not arrival order) and solves its
// diagonal block, right-hand sides dealt to the waves.
// The chain of blocks bounds it: what a hop costs is the time from one block's
// solution to the next one's.  A block's solution is its own flag: the front's
// part of P (unused while the triangle is solved) is set to kUnset by the
// launch before, the solution is stored there with device-scope stores, and
// the readers load the values themselves until none is kUnset.  With a flag of
// its own a block put a release (a write-back of the XCD's L2) and a second
// round trip into every hop: on a 4,160-column root with one right-hand side
// a hop took 5.3 us and takes 2.95; on a 2,350-column root with 64, all in
// one group, it took 27 us and takes 6.5 in four groups.
// The tickets (per big front nb + 1 words for the forward solve, of which the
// first kBigGroups are used, then as many for the backward solve; nb > 4)
// live after the call's workspace and are cleared by k_big_sync_clear at the
// start of every solve.
constexpr int kBigGroups = 4;
__device__ inline double load_dev(const double *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void publish(double *p, double v) {
  if (is_unset(v)) v = __longlong_as_double((long long)(kUnset ^ 1));
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// v[u] = y[off(u)], once every lane's 16 entries are published
template <class Off>
__device__ inline void wait_values(const double *y, Off off, double (&v)[16]) {
  bool miss;
  do {
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = load_dev(y + off(u));
    miss = false;
#pragma unroll
    for (int u = 0; u < 16; ++u) miss |= is_unset(v[u]);
  } while (__ballot(miss) != 0);
}

__global__ void k_big_sync_clear(int *sync, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) sync[i] = 0;
}

// Big fronts before their triangles, a workgroup per 64 positions and four
// right-hand sides (one a wave in the loops over both).  Forward: X[0:n] = own
// b + the children's updates, 64 pre-pivot positions at a time (ctab holds a
// child's entries of them, at most one a lane), summed in LDS in child order.
// As one workgroup per front, with its barriers for every 64 entries of a
// child, a 4,160-column root's took 105 us.  Backward: X[j] = x[perm[j]] minus
// the partial sums.  Both leave the front's solution unpublished.
constexpr int kInitRhs = 4, kInitPar = 64;
__global__ __launch_bounds__(kThreads) void k_big_fwd_init(const SolveNode *sn, const int *boff,
                                                           const int *bslot, int nbig,
                                                           const int *child_list,
                                                           const double *x, int ldx, int nrhs,
                                                           double *ws) {
  __shared__ double xs[kInitRhs][kBlk];
  int before;  // (the grid is the table's total)
  const int li = front_of(boff, nbig, blockIdx.x, before);
  if (li < 0) return;
  const SolveNode &P = sn[bslot[li]];
  gcint *Pipos = (gcint *)P.ipos;
  gcint *Prows = (gcint *)P.rows;
  gcint *Pctab = (gcint *)P.ctab;
  const int m = P.m, n = P.n, nd = P.nd, ne = P.nelim, cbeg = P.cbeg, cend = P.cend;
  const int T = idiv_up(m, 64), Tn = idiv_up(n, 64), nb = idiv_up(ne, kBlk);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int rc = kInitRhs * blockIdx.y; rc < nrhs; rc += kInitRhs * gridDim.y) {
    const int nr = imin(kInitRhs, nrhs - rc);
    double *X = solve_X(ws, P, nrhs) + (size_t)rc * m;
    double *Y = solve_P(ws, P, nrhs) + (size_t)rc * ne;
    for (int t = blockIdx.x - before; t < Tn; t += nb) {
      const int pre0 = 64 * t, pp = pre0 + lane;
      int pos = -1;
      if (pp < n) {
        pos = Pipos[pp];
        if (wave < nr)
          xs[wave][lane] = (pp >= nd) ? x[(size_t)(rc + wave) * ldx + Prows[pp - nd]] : 0.0;
      }
      __syncthreads();
      for (int c0 = cbeg; c0 < cend; c0 += kGroups) {
        const int ci = c0 + wave;
        int at = -1;
        double val[kInitRhs];
        if (ci < cend) {
          const SolveNode &c = sn[child_list[ci]];
          const int cn = c.n, cm = c.m;
          gcint *tab = Pctab + (size_t)(ci - cbeg) * (T + 1) + t;
          const int k = tab[0] + lane, ke = tab[1];
          if (k < ke) {
            const int pre =
                (k < cn) ? c.doff + (k - c.nelim) : nd + ((gcint *)c.rmap)[k - cn];
            if (pre < n) {
              at = pre - pre0;
              gcdouble *cX = (gcdouble *)(solve_X(ws, c, nrhs) + (size_t)rc * cm);
#pragma unroll
              for (int q = 0; q < kInitRhs; ++q) val[q] = cX[(size_t)imin(q, nr - 1) * cm + k];
            }
          }
        }
        for (int w = 0; w < kGroups; ++w) {
          if (wave == w && at >= 0) {
#pragma unroll
            for (int q = 0; q < kInitRhs; ++q) xs[q][at] += val[q];
          }
          __syncthreads();
        }
      }
      if (wave < nr) {
        if (pos >= 0) X[(size_t)wave * m + pos] = xs[wave][lane];
        if (pp < ne) Y[(size_t)wave * ne + pp] = __longlong_as_double((long long)kUnset);
      }
      __syncthreads();
    }
  }
}

__global__ __launch_bounds__(kThreads) void k_big_bwd_init(const SolveNode *sn, const int *boff,
                                                           const int *bslot, int nbig,
                                                           const double *x, int ldx, int nrhs,
                                                           double *ws, int dfuse) {
  int before;  // (the grid is the table's total)
  const int li = front_of(boff, nbig, blockIdx.x, before);
  if (li < 0) return;
  const SolveNode &P = sn[bslot[li]];
  const int m = P.m, ne = P.nelim, count = idiv_up(m - ne, kThreads);
  const int j = (blockIdx.x - before) * kBlk + (threadIdx.x & 63);
  if (j >= ne) return;
  gcint *Pperm = (gcint *)P.perm;
  double *PX = solve_X(ws, P, nrhs), *PY = solve_P(ws, P, nrhs);
  for (int q = kInitRhs * blockIdx.y + (threadIdx.x >> 6); q < nrhs; q += kInitRhs * gridDim.y) {
    const double *xq = x + (size_t)q * ldx;
    double *y = PY + (size_t)q * ne + j;
    PX[(size_t)q * m + j] =
        (dfuse ? dinv_at((gcdouble *)P.D, Pperm, xq, j, ne) : xq[Pperm[j]]) -
        part_sum((gcdouble *)y, (size_t)nrhs * ne, count);
    *y = __longlong_as_double((long long)kUnset);  // this thread's own first partial sum
  }
}

// The products of the other blocks go to FP64 MFMA (v_mfma_f64_16x16x4f64)
// for a group of up to 16 right-hand sides: wave w takes 16 rows (forward) or
// 16 columns (backward) of block b, the right-hand sides are the 16-wide
// output columns, and the 64 positions of each other block are the K
// dimension in steps of 4, in block order.  An output column depends only
// on its own right-hand side, so every column is the same whatever nrhs.
// The diagonal block is then solved once per right-hand side (lane = row,
// the right-hand sides dealt to the waves in turn).  The next block's part of
// L is loaded before the wait for the current one.

// L of one wave's 16 outputs against the 64 positions of a block, and the
// accumulation of a block's product
__device__ inline void big_mfma(const double (&av)[16], const double (&bv)[16], bool on,
                                mr_acc_t (&acc)[kMrSplit]) {
#pragma unroll
  for (int u = 0; u < 16; ++u)
    acc[u % kMrSplit] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], on ? bv[u] : 0.0,
                                                             acc[u % kMrSplit], 0, 0, 0);
}

// The diagonal block for the group's right-hand sides, G to a wave: lane i
// starts from its initial value x0 minus the products' sum (red) and takes
// part j of the substitution (in ascending order forward, descending backward)
// from lane j; l[j] is lane i's factor for part j.  Published to Y, kept in X
// and x.
template <bool FWD, int G>
__device__ inline void big_diag(const double (&l)[kBlk], const double (*red)[kBlk],
                                const double (&x0)[kDiagGroup], double *X, size_t m, double *Y,
                                size_t ldy, double *x, size_t ldx, int var, int j0, int wb,
                                int nr, int lane, int wave) {
  double v[G];
#pragma unroll
  for (int r = 0; r < G; ++r) v[r] = (lane < wb) ? x0[r] - red[wave * G + r][lane] : 0.0;
  substitute<FWD, G>(l, v);
#pragma unroll
  for (int r = 0; r < G; ++r) {
    const int q = wave * G + r;
    if (q < nr && lane < wb) publish(Y + (size_t)q * ldy + j0 + lane, v[r]);
  }
#pragma unroll
  for (int r = 0; r < G; ++r) {
    const int q = wave * G + r;
    if (q < nr && lane < wb) {
      X[(size_t)q * m + j0 + lane] = v[r];
      x[(size_t)q * ldx + var] = v[r];
    }
  }
}
// right-hand sides a wave takes in a group of nr (16 / kGroups = kDiagGroup)
static_assert(kDiagGroup * kGroups == kRhsGroup, "a group's right-hand sides, once over the waves");
__device__ inline void big_x0(const double *X, size_t m, int j0, int wb, int nr, int lane,
                              int wave, double (&x0)[kDiagGroup]) {
  const int G = (nr > kGroups) ? kDiagGroup : 1;
#pragma unroll
  for (int r = 0; r < kDiagGroup; ++r)
    x0[r] = masked(X[(size_t)imin(wave * G + r, nr - 1) * m + j0 + imin(lane, wb - 1)],
                   r < G && wave * G + r < nr);
}

// forward: block b's rows minus L[b rows, earlier columns] Y[earlier]
__global__ __launch_bounds__(kThreads) void k_big_fwd_lvl(const SolveNode *sn, const int *boff,
                                                          const int *bslot, const int *bsync,
                                                          int nbig, double *x, int ldx,
                                                          int nrhs, int rg, double *ws, int *sync) {
  __shared__ double red[kRhsGroup][kBlk];
  __shared__ int s_b;
  int before;  // (the grid is the table's total)
  const int li = front_of(boff, nbig, blockIdx.x, before);
  if (li < 0) return;
  const SolveNode &P = sn[bslot[li]];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ri = lane & 15, kq = lane >> 4;
  if (tid == 0) s_b = atomicAdd(sync + bsync[li] + blockIdx.y, 1);
  __syncthreads();
  const int b = s_b;
  gcdouble *PL = (gcdouble *)P.L;
  gcint *Pperm = (gcint *)P.perm;
  double *PX = solve_X(ws, P, nrhs), *PY = solve_P(ws, P, nrhs);
  const int ldl = P.ldl, m = P.m, ne = P.nelim;
  const int j0 = b * kBlk, j1 = imin(j0 + kBlk, ne), wb = j1 - j0;
  const int var = Pperm[j0 + imin(lane, wb - 1)];
  // A operand row of this lane (the wave's 16 rows of block b, clamped)
  gcdouble *La = PL + j0 + imin(16 * wave + ri, wb - 1);
  // L of the diagonal block for the substitutions (lane = row), loaded once
  double l[kBlk];
  load_rows(P.L, ldl, j0, wb, lane, l);
  for (int rc = rg * blockIdx.y; rc < nrhs; rc += rg * gridDim.y) {
    const int nr = imin(rg, nrhs - rc);
    double *X = PX + (size_t)rc * m, *Y = PY + (size_t)rc * ne;
    const double *y = Y + (size_t)imin(ri, nr - 1) * ne + kq;
    double x0[kDiagGroup];
    big_x0(X, m, j0, wb, nr, lane, wave, x0);
    mr_acc_t acc[kMrSplit];
#pragma unroll
    for (int t = 0; t < kMrSplit; ++t) acc[t] = (mr_acc_t){0.0, 0.0, 0.0, 0.0};
    double av[16];
    // every block before b is a full block
#pragma unroll
    for (int u = 0; u < 16; ++u) av[u] = La[(size_t)(b > 0 ? 4 * u + kq : 0) * ldl];
    for (int j = 0; j < b; ++j) {
      const int cn = imin(j + 1, b - 1) * kBlk;
      double an[16], bv[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) an[u] = La[(size_t)(cn + 4 * u + kq) * ldl];
      wait_values(y + j * kBlk, [](int u) { return 4 * u; }, bv);
      big_mfma(av, bv, ri < nr, acc);
#pragma unroll
      for (int u = 0; u < 16; ++u) av[u] = an[u];
    }
    // element (row kq + 4 rg of the wave's rows, right-hand side ri)
    const mr_acc_t sum = mr_sum(acc);
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) red[ri][16 * wave + kq + 4 * rg] = sum[rg];
    __syncthreads();
    if (nr > kGroups)
      big_diag<true, kDiagGroup>(l, red, x0, X, m, Y, ne, x + (size_t)rc * ldx, ldx, var, j0,
                                  wb, nr, lane, wave);
    else if (wave < nr)
      big_diag<true, 1>(l, red, x0, X, m, Y, ne, x + (size_t)rc * ldx, ldx, var, j0, wb, nr,
                         lane, wave);
    __syncthreads();
  }
}

// backward: block b's values minus L[later rows, b columns]^T X[later]
__global__ __launch_bounds__(kThreads) void k_big_bwd_lvl(const SolveNode *sn, const int *boff,
                                                          const int *bslot, const int *bsync,
                                                          int nbig, double *x, int ldx,
                                                          int nrhs, int rg, double *ws,
                                                          int *sync) {
  __shared__ double lb[kBlk][kBlk + 1];
  __shared__ double red[kRhsGroup][kBlk];
  __shared__ int s_b;
  int before;  // (the grid is the table's total)
  const int li = front_of(boff, nbig, blockIdx.x, before);
  if (li < 0) return;
  const SolveNode &P = sn[bslot[li]];
  const int ne = P.nelim, nb = idiv_up(ne, kBlk);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ri = lane & 15, kq = lane >> 4;
  if (tid == 0) s_b = nb - 1 - atomicAdd(sync + bsync[li] + nb + 1 + blockIdx.y, 1);
  __syncthreads();
  const int b = s_b;
  gcdouble *PL = (gcdouble *)P.L;
  gcint *Pperm = (gcint *)P.perm;
  double *PX = solve_X(ws, P, nrhs), *PY = solve_P(ws, P, nrhs);
  const int ldl = P.ldl, m = P.m;
  const int j0 = b * kBlk, j1 = imin(j0 + kBlk, ne), wb = j1 - j0;
  const int var = Pperm[j0 + imin(lane, wb - 1)];
  double c[kBlk];
  double st[kStage];
  load_lower(P.L, ldl, j0, wb, st);
  store_lower(st, lb);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kBlk; ++i) c[i] = lb[i][lane];
  // A operand column of this lane (the wave's 16 columns of block b, clamped)
  gcdouble *La = PL + (size_t)(j0 + imin(16 * wave + ri, wb - 1)) * ldl;
  auto load_a = [&](int j, double (&a)[16]) {
    const int r0 = j * kBlk, rows = imin(kBlk, ne - r0);
#pragma unroll
    for (int u = 0; u < 16; ++u)
      a[u] = masked(La[r0 + imin(4 * u + kq, rows - 1)], 4 * u + kq < rows);
  };
  for (int rc = rg * blockIdx.y; rc < nrhs; rc += rg * gridDim.y) {
    const int nr = imin(rg, nrhs - rc);
    double *X = PX + (size_t)rc * m, *Y = PY + (size_t)rc * ne;
    const double *y = Y + (size_t)imin(ri, nr - 1) * ne;
    double x0[kDiagGroup];
    big_x0(X, m, j0, wb, nr, lane, wave, x0);
    mr_acc_t acc[kMrSplit];
#pragma unroll
    for (int t = 0; t < kMrSplit; ++t) acc[t] = (mr_acc_t){0.0, 0.0, 0.0, 0.0};
    double av[16];
    load_a(nb - 1, av);
    for (int j = nb - 1; j > b; --j) {
      const int r0 = j * kBlk, rows = imin(kBlk, ne - r0);
      double an[16], bv[16];
      load_a(imax(j - 1, b + 1), an);
      wait_values(y + r0, [&](int u) { return imin(4 * u + kq, rows - 1); }, bv);
      // (rows past the last block's end: zero in av, and 0 * NaN is avoided)
      if (rows < kBlk) {
#pragma unroll
        for (int u = 0; u < 16; ++u) bv[u] = masked(bv[u], 4 * u + kq < rows);
      }
      big_mfma(av, bv, ri < nr, acc);
#pragma unroll
      for (int u = 0; u < 16; ++u) av[u] = an[u];
    }
    // element (row kq + 4 rg of the wave's columns, right-hand side ri)
    const mr_acc_t sum = mr_sum(acc);
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) red[ri][16 * wave + kq + 4 * rg] = sum[rg];
    __syncthreads();
    if (nr > kGroups)
      big_diag<false, kDiagGroup>(c, red, x0, X, m, Y, ne, x + (size_t)rc * ldx, ldx, var, j0,
                                  wb, nr, lane, wave);
    else if (wave < nr)
      big_diag<false, 1>(c, red, x0, X, m, Y, ne, x + (size_t)rc * ldx, ldx, var, j0, wb, nr,
                         lane, wave);
    __syncthreads();
  }
}

// ---- launchers ----------------------------------------------------------------
int big_tri_threshold() { return kBigTri; }
int fwd_rows_per_wg() { return kRows; }
int bwd_rows_per_wg() { return kThreads; }
int bwd_cols_per_wg() { return kBwdCols; }

// tab: the level's big fronts, [boff (nbig+1) | slots (nbig) | sync offsets
// (nbig)]; nwg = boff[nbig], the level's 64-column blocks
// Right-hand sides a group of the front kernels takes: a hop or a front's chain
// takes about as long for four (a wave each) as for one, and for 16 about
// twice as long, so groups are of four while all of their workgroups run at
// once (the big fronts' kernels keep one a CU and at most kBigGroups groups).
// The chain of a
// 1,791-column KKT root, backward with 16 right-hand sides: 176 us in one group
// of 16, 95 in four of four.
static int big_group(int nwg, int nrhs) {
  return (nrhs <= kRhsFew * kBigGroups && nwg * idiv_up(nrhs, kRhsFew) <= 256) ? kRhsFew
                                                                                : kRhsGroup;
}
static bool rhs_few(int nwg, int nrhs) {
  return nrhs <= kRhsFew || (int64_t)nwg * idiv_up(nrhs, kRhsFew) <= 512;
}
static int rhs_groups(int nrhs, int group) {
  return imin(idiv_up(nrhs, group), kRhsGroupsPar);
}

void launch_big_fwd_lvl(hipStream_t st, const SolveNode *sn, const int *tab, int nbig, int nwg,
                        const int *child_list, double *x, int ldx, int nrhs, double *ws,
                        int *sync) {
  if (nbig <= 0) return;
  hipLaunchKernelGGL(k_big_fwd_init, dim3(nwg, imin(idiv_up(nrhs, kInitRhs), kInitPar)),
                     dim3(kThreads), 0, st, sn, tab, tab + nbig + 1, nbig, child_list, x, ldx,
                     nrhs, ws);
  const int rg = big_group(nwg, nrhs);
  hipLaunchKernelGGL(k_big_fwd_lvl, dim3(nwg, imin(idiv_up(nrhs, rg), kBigGroups)),
                     dim3(kThreads), 0, st, sn, tab, tab + nbig + 1, tab + 2 * nbig + 1, nbig, x,
                     ldx, nrhs, rg, ws, sync);
}
void launch_big_bwd_lvl(hipStream_t st, const SolveNode *sn, const int *tab, int nbig, int nwg,
                        double *x, int ldx, int nrhs, double *ws, int *sync, int dfuse) {
  if (nbig <= 0) return;
  hipLaunchKernelGGL(k_big_bwd_init, dim3(nwg, imin(idiv_up(nrhs, kInitRhs), kInitPar)),
                     dim3(kThreads), 0, st, sn, tab, tab + nbig + 1, nbig, x, ldx, nrhs, ws,
                     dfuse);
  const int rg = big_group(nwg, nrhs);
  hipLaunchKernelGGL(k_big_bwd_lvl, dim3(nwg, imin(idiv_up(nrhs, rg), kBigGroups)),
                     dim3(kThreads), 0, st, sn, tab, tab + nbig + 1, tab + 2 * nbig + 1, nbig, x,
                     ldx, nrhs, rg, ws, sync);
}
void launch_big_sync_clear(hipStream_t st, int *sync, int n) {
  if (n > 0)
    hipLaunchKernelGGL(k_big_sync_clear, dim3((n + 255) / 256), dim3(256), 0, st, sync, n);
}

void launch_fwd_tri(hipStream_t st, int nlvl, const SolveNode *sn, int s0,
                    const int *child_list, double *x, int ldx, int nrhs, double *ws) {
  if (nlvl <= 0) return;
  if (nrhs == 1)
    hipLaunchKernelGGL(k_fwd_tri<1>, dim3(nlvl), dim3(kThreads), 0, st, sn, s0, child_list, x,
                       ldx, nrhs, ws);
  else if (rhs_few(nlvl, nrhs))
    hipLaunchKernelGGL(k_fwd_tri<kRhsFew>, dim3(nlvl, rhs_groups(nrhs, kRhsFew)),
                       dim3(kThreads), 0, st, sn, s0, child_list, x, ldx, nrhs, ws);
  else
    hipLaunchKernelGGL(k_fwd_tri<kRhsGroup>, dim3(nlvl, rhs_groups(nrhs, kRhsGroup)),
                       dim3(kThreads), 0, st, sn, s0, child_list, x, ldx, nrhs, ws);
}
void launch_fwd_rows(hipStream_t st, int nlvl, const SolveNode *sn, int s0,
                     const int *child_list, int nrhs, const int *wg_off, int nwg, double *ws) {
  if (nlvl <= 0 || nwg <= 0) return;
  if (nrhs == 1)
    hipLaunchKernelGGL(k_fwd_rows<1>, dim3(nwg), dim3(kThreads), 0, st, sn, s0, child_list,
                       wg_off, nlvl, nrhs, ws);
  else if (rhs_few(nwg, nrhs))
    hipLaunchKernelGGL(k_fwd_rows<kRhsFew>, dim3(nwg, rhs_groups(nrhs, kRhsFew)),
                       dim3(kThreads), 0, st, sn, s0, child_list, wg_off, nlvl, nrhs, ws);
  else
    hipLaunchKernelGGL(k_fwd_rows<kRhsGroup>, dim3(nwg, rhs_groups(nrhs, kRhsGroup)),
                       dim3(kThreads), 0, st, sn, s0, child_list, wg_off, nlvl, nrhs, ws);
}
void launch_dsolve(hipStream_t st, int nslots, const SolveNode *sn, double *x, int ldx,
                   int nrhs, int half) {
  if (nslots > 0)
    hipLaunchKernelGGL(k_dsolve, dim3(nslots), dim3(64), 0, st, sn, nslots, x, ldx, nrhs,
                       half);
}
// rows_off: the level's 256-row workgroup table (per front); chunk_off /
// nwg: the row workgroups x column chunks table of k_bwd_rows and its total
void launch_bwd(hipStream_t st, int nlvl, const SolveNode *sn, int s0, double *x,
                int ldx, int nrhs, const int *rows_off, const int *chunk_off, int nwg,
                double *ws, int dfuse, int ntri) {
  if (nlvl <= 0) return;
  if (nwg > 0)
    hipLaunchKernelGGL(k_bwd_rows, dim3(nwg, rhs_groups(nrhs, kRhsGroup)), dim3(kThreads), 0,
                       st, sn, s0, chunk_off, nlvl, x, ldx, nrhs, ws);
  if (ntri <= 0) return;  // big fronts only
  if (nrhs == 1)
    hipLaunchKernelGGL(k_bwd_tri<1>, dim3(nlvl), dim3(kThreads), 0, st, sn, s0, rows_off, x,
                       ldx, nrhs, ws, dfuse);
  else if (rhs_few(nlvl, nrhs))
    hipLaunchKernelGGL(k_bwd_tri<kRhsFew>, dim3(nlvl, rhs_groups(nrhs, kRhsFew)),
                       dim3(kThreads), 0, st, sn, s0, rows_off, x, ldx, nrhs, ws, dfuse);
  else
    hipLaunchKernelGGL(k_bwd_tri<kRhsGroup>, dim3(nlvl, rhs_groups(nrhs, kRhsGroup)),
                       dim3(kThreads), 0, st, sn, s0, rows_off, x, ldx, nrhs, ws, dfuse);
}

}  // namespace ssids_hip
