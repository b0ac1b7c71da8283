// Numeric factorization kernels for gfx950 (CDNA4, wave64).
//
// One tree level is processed per launch sequence; a launch covers every
// front of the level.  Workgroups find their front by binary search in a
// per-level prefix array of workgroup counts (wg_off).
//
//  k_gather     gather assembly: a workgroup builds a 64x64 tile of one parent
//               front in registers from its children (children in order =>
//               deterministic sums) through maps in LDS, computing the
//               children's Schur complements on MFMA on the way.
//  k_diag       one workgroup per front: factor the w<=64 column diagonal
//               block with complete pivoting (1x1/2x2) in registers
//               (pivot rules of src/ssids/cpu/kernels/block_ldlt.hxx:213-414).
//  k_apply      L = A Lbb^{-T} D^{-1} for the rows below the block, keeping a
//               backup and the columns with an |l| > 1/u (a posteriori test,
//               src/ssids/cpu/kernels/ldlt_app.cxx:304-414).
//  k_update     restore failed columns and apply the accepted pivots to the
//               trailing panel columns with v_mfma_f64_16x16x4_f64 on 64x64
//               tiles (the contribution block is updated lazily by k_gather).
//  k_update_diag  on large fronts, all but the first tile column of that,
//               beside the next step's pivot blocks.
//  k_swap       move failed columns behind the unprocessed candidates.
//  k_tail       end of a level, one workgroup per front: APP result,
//               threshold partial pivoting on the failed columns
//               (src/ssids/cpu/kernels/ldlt_tpp.cxx:166-270), D and L21 D
//               operands of the parent's gather, solve position index.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "dev.hpp"

namespace ssids_hip {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef double double16_t __attribute__((ext_vector_type(16)));
typedef unsigned uint16v_t __attribute__((ext_vector_type(16)));

// front of workgroup b in a level table, or -1 past the table's total (grids
// sized for the plan's capacities may be larger than the level needs)
// element (i,j), i>=j, of the front (panel for j<n, contribution block else)
__device__ inline double *front_at(const NodeDev &N, int i, int j) {
  if (j < N.n) return N.L + (size_t)j * N.ldl + i;
  return N.C + (size_t)(j - N.n) * N.ldc + (i - N.n);
}

// parent position of trailing index k of child c (monotone in k)
__device__ inline int child_pos(const NodeDev &c, int doff, int pnd, int k) {
  if (k < c.n) return doff + (k - c.nelim);
  return pnd + c.rmap[k - c.n];
}

__device__ inline const double *child_src(const NodeDev &c, int kr, int k) {
  if (k < c.n) return c.L + (size_t)k * c.ldl + kr;
  return c.C + (size_t)(k - c.n) * c.ldc + (kr - c.n);
}

// ---------------------------------------------------------------------------
// Diagonal block factorization, NW waves per front.  Lane i of wave v keeps
// columns [vR, vR+R) (R = 64/NW) of row i of the symmetric w x w block in
// registers; pivots are tracked in a uniform bit mask (no physical swaps).
// Per pivot step, with one workgroup barrier unless the maximum lies off the
// diagonal:
//  * search: every lane takes the maximum |a(i,j)| of its live columns j <= i
//    (the lower triangle, as block_ldlt.hxx:77-101 searches it: each
//    symmetric pair once, in one orientation, so a maximum off the diagonal
//    gives the pair (column, row) with column < row whatever the rounding of
//    the two mirrored entries).  The wave reduces the maxima's high words
//    with DPP; the low words, and the order (smallest column, then row) among
//    equal values, are looked at only when two lanes share the high word;
//  * each wave publishes its candidate through LDS before the barrier: the
//    value, its position, its reciprocal (the division runs while the
//    position is found) and the whole column, which one wave holds, so no
//    second exchange follows the merge.  The waves hold ascending columns,
//    so the first wave with the largest value has the smallest column;
//  * a maximum off the diagonal fetches the second column the same way;
//  * rank-1 / rank-2 update of every row's columns in registers: the lane's
//    own column entry times L of the wave's R columns, which sit in the lanes
//    of each row of 16 and reach the FMAs by DPP (row_newbcast);
//  * the L column(s) of the step go to LDS, indexed by elimination step.
// Pivot rules of src/ssids/cpu/kernels/block_ldlt.hxx:289-414: maximum on the
// diagonal -> 1x1; else the 2x2 test of block_ldlt.hxx:213-218, else the
// larger diagonal as 1x1.  A maximum below `small` makes every remaining
// index a zero pivot.  The a posteriori test of k_apply then checks
// |l| <= 1/u over the full column.  The elimination order lp[] permutes the
// block on write back.
// The block is bound by the chain of its 64 steps on one CU: about 300
// instructions of one wave per SIMD at 4 cycles, two LDS round trips and a
// barrier (1,760 cycles a step, 132,000 a block).  The layout with a column
// per lane and 16 rows a wave needed the search's merge and the column's
// broadcast one after the other, two barriers a step: 250,000 cycles, 118 us
// a block against 64 us (64 x 64, one front).  Eight waves of 8 columns take
// 83 us: the second wave of a SIMD waits for its issue slots.
// ---------------------------------------------------------------------------
constexpr int kDiagWaves = 4;
constexpr int kDiagCols = kBlk / kDiagWaves;  // columns of a wave: 16

// max of two values that hold no signalling NaN (a NaN loses), one
// instruction: fmax would quiet both operands first
__device__ inline double max_f64(double x, double y) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
  return r;
}

// a condition every lane of the wave agrees on, as a scalar
__device__ inline bool uniform_true(bool c) { return __builtin_amdgcn_ballot_w64(c) != 0ull; }

// v permuted within rows of lanes by a DPP control
template <int CTRL>
__device__ inline double dpp_f64(double v) {
  const int hi = __double2hiint(v), lo = __double2loint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, true));
}
// the larger of v and its permuted value (no NaN)
template <int CTRL>
__device__ inline double dpp_max_f64(double v) {
  const double o = dpp_f64<CTRL>(v);
  return o > v ? o : v;
}

// value of v in lane j (j uniform), as a scalar
__device__ inline double lane_value(double v, int j) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), j),
                          __builtin_amdgcn_readlane(__double2loint(v), j));
}

// Largest |a[j]| over j = 0..15 in the lanes >= c0 + j only (the lower
// triangle of a wave's columns); NaN never wins.  Called with every lane of
// the wave active.
__device__ __forceinline__ double max_lower(double16_t a, int c0) {
  double m0 = 0.0, m1 = 0.0;
#define SSIDS_MAX(m, r) \
  "v_max_f64 %" #m ", %" #m ", |%" #r "|\n\ts_lshl_b64 exec, exec, 1\n\t"
  asm("s_lshl_b64 exec, -1, %18\n\t" SSIDS_MAX(0, 2) SSIDS_MAX(1, 3) SSIDS_MAX(0, 4)
          SSIDS_MAX(1, 5) SSIDS_MAX(0, 6) SSIDS_MAX(1, 7) SSIDS_MAX(0, 8) SSIDS_MAX(1, 9)
              SSIDS_MAX(0, 10) SSIDS_MAX(1, 11) SSIDS_MAX(0, 12) SSIDS_MAX(1, 13)
                  SSIDS_MAX(0, 14) SSIDS_MAX(1, 15) SSIDS_MAX(0, 16) SSIDS_MAX(1, 17)
      "s_mov_b64 exec, -1"
      : "+v"(m0), "+v"(m1)
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]),
        "v"(a[7]), "v"(a[8]), "v"(a[9]), "v"(a[10]), "v"(a[11]), "v"(a[12]), "v"(a[13]),
        "v"(a[14]), "v"(a[15]), "s"(c0)
      : "scc");
#undef SSIDS_MAX
  return max_f64(m0, m1);
}

// One bit per j: h[j] = m in this lane (bit 15 - j).  The compares go to four
// scalar pairs in turn, so that no add-with-carry waits for the compare just
// before it.
__device__ __forceinline__ unsigned equal_bits(uint16v_t h, unsigned m) {
  unsigned bits = 0;
  unsigned long long s0, s1, s2, s3;
#define SSIDS_EQ4(j)                                                                   \
  asm("v_cmp_eq_u32 %1, %5, %9\n\tv_cmp_eq_u32 %2, %6, %9\n\t"                         \
      "v_cmp_eq_u32 %3, %7, %9\n\tv_cmp_eq_u32 %4, %8, %9\n\t"                         \
      "v_addc_co_u32 %0, vcc, %0, %0, %1\n\tv_addc_co_u32 %0, vcc, %0, %0, %2\n\t"     \
      "v_addc_co_u32 %0, vcc, %0, %0, %3\n\tv_addc_co_u32 %0, vcc, %0, %0, %4"         \
      : "+v"(bits), "=&s"(s0), "=&s"(s1), "=&s"(s2), "=&s"(s3)                         \
      : "v"(h[j]), "v"(h[j + 1]), "v"(h[j + 2]), "v"(h[j + 3]), "s"(m)                 \
      : "vcc")
  SSIDS_EQ4(0);
  SSIDS_EQ4(4);
  SSIDS_EQ4(8);
  SSIDS_EQ4(12);
#undef SSIDS_EQ4
  return bits;
}

// a[j] = fma(c, l_j, a[j]) for j = 0..15, l_j the value of `l` in lane j of
// the lane's own row of 16; with `two`, a[j] = fma(c2, l2_j, a[j]) first.
// The leading s_nop separates the writes of l and l2 from their DPP reads.
// The branch sits inside the statement, so that the registers stay where
// they are on both paths.
__device__ __forceinline__ void rank_update(double16_t &a, double c, double l, int two,
                                            double c2, double l2) {
#define SSIDS_FMAC(n, l, c) \
  "v_fmac_f64_dpp %" #n ", %" #l ", %" #c " row_newbcast:" #n " row_mask:0xf bank_mask:0xf\n\t"
#define SSIDS_FMAC16(l, c)                                                               \
  SSIDS_FMAC(0, l, c) SSIDS_FMAC(1, l, c) SSIDS_FMAC(2, l, c) SSIDS_FMAC(3, l, c)         \
  SSIDS_FMAC(4, l, c) SSIDS_FMAC(5, l, c) SSIDS_FMAC(6, l, c) SSIDS_FMAC(7, l, c)         \
  SSIDS_FMAC(8, l, c) SSIDS_FMAC(9, l, c) SSIDS_FMAC(10, l, c) SSIDS_FMAC(11, l, c)       \
  SSIDS_FMAC(12, l, c) SSIDS_FMAC(13, l, c) SSIDS_FMAC(14, l, c) SSIDS_FMAC(15, l, c)
  double a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3], a4 = a[4], a5 = a[5], a6 = a[6],
         a7 = a[7], a8 = a[8], a9 = a[9], a10 = a[10], a11 = a[11], a12 = a[12], a13 = a[13],
         a14 = a[14], a15 = a[15];
  asm("s_nop 1\n\ts_cmp_eq_u32 %20, 0\n\ts_cbranch_scc1 .Lrank1_%=\n\t" SSIDS_FMAC16(18, 19)
      ".Lrank1_%=:\n\t" SSIDS_FMAC16(16, 17)
      : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5), "+v"(a6), "+v"(a7),
        "+v"(a8), "+v"(a9), "+v"(a10), "+v"(a11), "+v"(a12), "+v"(a13), "+v"(a14), "+v"(a15)
      : "v"(l), "v"(c), "v"(l2), "v"(c2), "s"(two)
      : "scc");
  a[0] = a0, a[1] = a1, a[2] = a2, a[3] = a3, a[4] = a4, a[5] = a5, a[6] = a6, a[7] = a7;
  a[8] = a8, a[9] = a9, a[10] = a10, a[11] = a11, a[12] = a12, a[13] = a13, a[14] = a14,
  a[15] = a15;
#undef SSIDS_FMAC16
#undef SSIDS_FMAC
}

// Rows 16b..16b+15 of the inverse's diagonal block b: lane j of every row of
// 16 lanes holds column j in m, and lane i of a row holds L(i, k) in lk[k];
// m[i] -= L(i, k) m[k] for k ascending, L by DPP.
template <int K>
__device__ __forceinline__ void unit_lower_columns(double (&m)[16], const double (&lk)[15]) {
  if constexpr (K < 15) {
    const double c = -m[K];
#pragma unroll
    for (int i = K + 1; i < 16; ++i)
      asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
          : "+v"(m[i])
          : "v"(lk[K]), "v"(c), "n"(i));
    unit_lower_columns<K + 1>(m, lk);
  }
}

// W (64 x 64 row-major) = M = (I + N)^{-1}, N the strictly lower matrix with
// N(i, k) = mi[k][i]; ms is scratch.  Wave b inverts the 16 x 16 diagonal
// block b in registers, then blocks join by pairs on FP64 MFMA:
//   [M11 0; -M22 (L21 M11) M22]
// first to 32 x 32 (two waves), then to 64 x 64 (a 16 x 16 tile a wave).  A
// product's result (row i, column j in lane j + 16 (i % 4), register i / 4)
// is the next product's right operand as it stands.  Against 63 substitution
// steps on all 64 rows (7.5 us a block, most of it instruction fetch of the
// unrolled steps) this takes about 1 us.
__device__ __forceinline__ void block_inverse(const double (&mi)[kBlk][kBlk + 1],
                                              double (&ms)[kBlk][kBlk + 1], int wv, int lane,
                                              gdouble *W) {
  const int ri = lane & 15, kq = lane >> 4;
  {
    const int b0 = 16 * wv;
    double lk[15], m[16];
#pragma unroll
    for (int k = 0; k < 15; ++k) lk[k] = mi[b0 + k][b0 + ri];
#pragma unroll
    for (int i = 0; i < 16; ++i) m[i] = (i == ri) ? 1.0 : 0.0;
    // the loads above have returned and their last reader below is two
    // instructions away from any write of a DPP source
    asm volatile("s_nop 1");
    unit_lower_columns<0>(m, lk);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if ((i >> 2) == kq) ms[b0 + i][b0 + ri] = m[i];
  }
  __syncthreads();
  // acc += A B over 16 pivots, A(i, k) from `ld`, B(k, j) in b[k / 4]
  auto mul = [&](double4_t &acc, const double (&A)[kBlk][kBlk + 1], int r, int c, bool trans,
                 const double4_t &b) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double av = trans ? A[c + 4 * u + kq][r + ri] : A[r + ri][c + 4 * u + kq];
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av, b[u], acc, 0, 0, 0);
    }
  };
  auto right = [&](int r, int c) {  // the block of M at (r, c) as a right operand
    double4_t b;
#pragma unroll
    for (int u = 0; u < 4; ++u) b[u] = ms[r + 4 * u + kq][c + ri];
    return b;
  };
  auto put = [&](int r, int c, const double4_t &v) {
#pragma unroll
    for (int u = 0; u < 4; ++u) ms[r + 4 * u + kq][c + ri] = -v[u];
  };
  const double4_t zero = {0.0, 0.0, 0.0, 0.0};
  if (wv < 2) {
    const int b0 = 32 * wv;
    double4_t x = zero, y = zero;
    mul(x, mi, b0 + 16, b0, true, right(b0, b0));
    mul(y, ms, b0 + 16, b0 + 16, false, x);
    put(b0 + 16, b0, y);
  }
  __syncthreads();
  {
    // tile (I, J) of the lower left 32 x 32; X = L21 M11 for column block J
    const int I = wv >> 1, J = wv & 1;
    double4_t x0 = zero, x1 = zero, y = zero;
    for (int k = J; k < 2; ++k) {  // M11 is lower triangular by blocks
      const double4_t b = right(16 * k, 16 * J);
      mul(x0, mi, 32, 16 * k, true, b);
      mul(x1, mi, 48, 16 * k, true, b);
    }
    mul(y, ms, 32 + 16 * I, 32, false, x0);
    if (I == 1) mul(y, ms, 48, 48, false, x1);
    put(32 + 16 * I, 16 * J, y);
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 16; ++it) {
    const int r = 16 * wv + it;
    W[r * kBlk + lane] = masked(ms[r][lane], (lane >> 4) <= wv);
  }
}

constexpr int kGT = 64;  // gather tile edge
constexpr int kGatherInv = 3 * 2 * kGT;  // ints of LDS for its maps

template <int PART, typename CT>
__device__ __forceinline__ int gather_tile(
    NodeDev *nodes, int s0, const int *wg_off, int nlvl,
    const int *child_list, const double *aval, const int64_t *asrc, const int *arow,
    const int *acix, const double *scaling, double (&acc)[kGT][kGT + 1], int *inv);

struct GatherArgs {  // the level's gather inputs (a pivot launch that assembles)
  const int *wg_off;
  int nlvl;
  const int *child_list;
  const double *aval;
  const int64_t *asrc;
  const int *arow;
  const int *acix;
  const double *scaling;
};

// FIRST: one workgroup per front gathers the front's diagonal tile (0, 0)
// (the gather's part 1) and runs step 0's pivot block on it, as soon as its
// block is assembled and in a workgroup that already holds its CU, instead of
// queueing behind the rest of the level's gather.  The first tile column's
// other tiles (part 3) are gathered by k_gather, whose smaller LDS fits
// twice as many workgroups on a CU.
// C32 (FIRST only): the children's contribution blocks are FP32
template <int NW, bool FIRST, bool C32>
__device__ __forceinline__ void diag_front(NodeDev *nodes, int s0, int step, FactorParams fp,
                                           GatherArgs ga) {
  constexpr int R = kBlk / NW;
  static_assert(NW == kDiagWaves && R == kDiagCols, "a row of lanes holds L of a wave's columns");
  __shared__ double t[kBlk][kBlk + 1];  // load staging, then L by step: t[k][row]
  __shared__ double ccol[2][NW][kBlk];  // the waves' candidate columns (by step parity)
  struct alignas(16) Cand {
    int lo, hi;  // |value|
    int code;    // column << 6 | row
    int pad;
  };
  __shared__ Cand cand[2][NW];
  __shared__ double col2[kBlk];                // column of an off-diagonal maximum's row
  __shared__ double dinv[2 * kBlk + 2];
  __shared__ int lp[kBlk], inv_lp[kBlk], kind[kBlk];
  __shared__ double mi[kBlk][kBlk + 1];  // L_bb's strict lower part by columns
  int s;
  if constexpr (FIRST) {
    static_assert(64 * NW == kThreads, "one workgroup shape for both phases");
    static_assert(kGT == kBlk, "the gather tile is the pivot block's staging array");
    // the tile's LDS is the pivot block's own (t, mi), used in turn
    static_assert(sizeof(mi) >= kGatherInv * sizeof(int), "mi holds the gather's maps");
    typedef typename std::conditional<C32, float, double>::type CT;
    s = gather_tile<1, CT>(nodes, s0, ga.wg_off, ga.nlvl, ga.child_list, ga.aval,
                           ga.asrc, ga.arow, ga.acix, ga.scaling, t, (int *)mi);
    if (s < 0) return;
    __syncthreads();  // the block's stores are visible to the whole workgroup
  } else {
    s = s0 + blockIdx.x;
  }
  NodeDev &N = nodes[s];
  if (step >= N.nsteps) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = uni((int)threadIdx.x >> 6), c0 = wv * R;
  int p, q;
  if (step == 0) {
    p = 0;
    q = N.n;
  } else {
    p = N.p + N.npass;
    q = N.q - (N.w - N.npass);
  }
  const int w = max(0, min(kBlk, q - p));
  __syncthreads();  // every thread has read N.p/N.npass before they change
  if (tid == 0) {
    N.p = p;
    N.q = q;
    N.w = w;
    N.npass = 0;
  }
  if (w == 0) return;
  const int ldl = N.ldl;
  double *L = N.L;
  // The block's lower triangle, t[row][column] (a front's first block is still
  // there from its assembly); every thread's loads are unconditional (indices
  // clamped into the block) so they are all in flight together.
  if constexpr (!FIRST) {
    gcdouble *Lg = (gcdouble *)L;
    double v[R];
#pragma unroll
    for (int j = 0; j < R; ++j)
      v[j] = Lg[(size_t)(p + imin(c0 + j, w - 1)) * ldl + p + imin(lane, w - 1)];
#pragma unroll
    for (int j = 0; j < R; ++j) t[lane][c0 + j] = v[j];
  }
  if (tid == 0) N.fail = 0ull;
  __syncthreads();
  double16_t a;   // columns c0 .. c0 + 15 of row `lane`, zero outside the block
  uint16v_t msk;  // high-word mask of the search (0 above the diagonal)
#pragma unroll
  for (int j = 0; j < R; ++j) {
    a[j] = masked(t[imax(lane, c0 + j)][imin(lane, c0 + j)], lane < w && c0 + j < w);
    msk[j] = (lane >= c0 + j) ? 0x7fffffffu : 0u;
  }
  {
    // the backup the failed columns are restored from, a column a store
    gdouble *dbak = (gdouble *)N.dbak;
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (lane < w) dbak[lane + (c0 + j) * kBlk] = a[j];
  }
  __syncthreads();
  int livem = (lane < w) ? -1 : 0;  // -1: row `lane` is not eliminated
  int k = 0, par = 0, stop = 0;
  // a maximum below `small`, or of exactly zero, ends the block
  const double small = !(fp.small <= 4.9406564584124654e-324) ? fp.small
                                                              : 4.9406564584124654e-324;
  const int sl = c0 + (lane & (R - 1));  // the column whose L this lane passes to rank_update
  int plp = 0;  // lane k: pivot k's index | kind << 8 and D^{-1} entries
  double pd0 = 0.0, pd1 = 0.0;
  // v in the live rows, zero elsewhere
  auto live_value = [&](double v) {
    return __hiloint2double(__double2hiint(v) & livem, __double2loint(v) & livem);
  };
  // The end of a step: pivot pv's update a -= z (the lane's row) L (the wave's
  // columns, ls of lane sl), after z2, ls2 of a 2x2 block's second column
  // (two); L(:, k) = lj to LDS (every wave has the column: each stores its
  // rows); D^{-1} to lane k.  The pivot's own column takes the coefficient 1
  // and becomes exactly zero, out of the search; the published columns hold
  // zeros for eliminated rows, so it stays zero.
  auto finish = [&](int pv, double z, double ls, double lj, double e0, double e1, int two,
                    double z2, double ls2) __attribute__((always_inline)) {
    ls = (sl == pv) ? 1.0 : ls;
    rank_update(a, -z, ls, two, -z2, ls2);
    if (lane / R == wv) t[k][lane] = lj;
    const bool mine = lane == k;
    plp = mine ? (pv | (two + 1) << 8) : plp;
    pd0 = mine ? e0 : pd0;
    pd1 = mine ? e1 : pd1;
    livem = (lane == pv) ? 0 : livem;
    k += two + 1;
  };
  // The LDS exchanges alternate between two buffers: a wave that publishes
  // the next step's candidate must not overwrite what a slower wave still
  // reads of this one's.
  if (fp.posdef) {
    // Cholesky order: the lowest remaining index, always 1x1
    do {
      const double cv = a[k & (R - 1)];
      if (wv == k / R) ccol[par][0][lane] = live_value(cv);
      __syncthreads();
      const double z = ccol[par][0][lane], zs = ccol[par][0][sl];
      par ^= 1;
      const double d = lane_value(z, k);
      if (!uniform_true(d > 0.0)) {
        stop = -6;
        break;
      }
      const double e0 = 1.0 / d;
      finish(k, z, zs * e0, z * e0, e0, 0.0, 0, 0.0, 0.0);
    } while (k < w);
  } else {
    do {
      // ---- search this lane's live columns, by the high words
      uint16v_t h;
#pragma unroll
      for (int j = 0; j < R; ++j) h[j] = (unsigned)__double2hiint(a[j]) & msk[j];
      unsigned m0 = max(max(h[0], h[1]), h[2]), m1 = max(max(h[3], h[4]), h[5]);
#pragma unroll
      for (int j = 6; j < R - 2; j += 4) {
        m0 = max(max(m0, h[j]), h[j + 1]);
        m1 = max(max(m1, h[j + 2]), h[j + 3]);
      }
      m0 = max(max(m0, h[R - 2]), h[R - 1]);
      const unsigned mh = max(m0, m1) & (unsigned)livem;
      const unsigned H = (unsigned)uni((int)wave_max_u32(mh));
      const unsigned long long hit = __builtin_amdgcn_ballot_w64(mh == H);
      // the wave's candidate: row ci, column c0 + cj, |value| = (mhi, mlo)
      int ci = __builtin_ctzll(hit);
      const unsigned eq = (unsigned)__builtin_amdgcn_readlane((int)equal_bits(h, H), ci);
      int cj;
      unsigned mhi, mlo;
      double cv;
      if (__builtin_expect(
              __builtin_popcountll(hit) + __builtin_popcount(eq) + (H >= 0x7ff00000u ? 1 : 0) == 2,
              1)) {
        cj = __builtin_clz(eq) - (32 - R);
        cv = a[cj];
        mhi = H;
        mlo = (unsigned)__builtin_amdgcn_readlane(__double2loint(cv), ci);
      } else {
        // Two entries share the largest high word, or it is zero, a
        // subnormal's or a NaN's.
        unsigned low = 0;
#pragma unroll
        for (int j = 0; j < R; ++j) low |= msk[j] ? (unsigned)__double2loint(a[j]) : 0u;
        cj = ci = 0;
        mhi = mlo = 0u;
        // (zeros only: every column of the wave is eliminated)
        if (H != 0u || uniform_true((low & (unsigned)livem) != 0u)) {
          // exact maxima (NaN never wins), then the smallest column and row
          const double mx = max_lower(a, c0);
          const unsigned long long ml =
              livem ? (unsigned long long)__double_as_longlong(mx) : 0ull;
          const unsigned long long kw = wave_max_u64(ml);
          int jf = R - 1;
#pragma unroll
          for (int j = R - 2; j >= 0; --j) jf = (fabs(a[j]) == mx) ? j : jf;
          const unsigned code =
              ~wave_max_u32((livem && ml == kw) ? ~(unsigned)((jf << 6) | lane) : 0u);
          cj = uni((int)(code >> 6) & (R - 1));
          ci = uni((int)(code & 63u));
          mhi = (unsigned)uni((int)(kw >> 32));
          mlo = (unsigned)uni((int)(kw & 0xffffffffull));
        }
        cv = a[cj];
      }
      ccol[par][wv][lane] = live_value(cv);
      Cand c;
      c.lo = (int)mlo;
      c.hi = (int)mhi;
      c.code = ((c0 + cj) << 6) | ci;
      c.pad = 0;
      if (lane == 0) cand[par][wv] = c;
      __syncthreads();
      // the first wave holding the largest value wins: lane u looks at wave
      // u % NW's candidate
      const Cand cu = cand[par][lane & (NW - 1)];
      const double vm = __hiloint2double(cu.hi, cu.lo);
      const double vmax = dpp_max_f64<0x4E>(dpp_max_f64<0xB1>(vm));
      const int win = __builtin_ctzll(__builtin_amdgcn_ballot_w64(vm == vmax));
      const double x0 = ccol[par][win][lane], y0 = ccol[par][win][sl];
      par ^= 1;
      const double rcp = 1.0 / vmax;  // in the shadow of the column's loads
      const int code = __builtin_amdgcn_readlane(cu.code, win);
      const int p1 = code >> 6, r1 = code & 63;
      if (!uniform_true(vmax >= small)) {
        stop = -5;
        break;
      }
      const double a11 = lane_value(x0, p1);
      int pv = p1, two = 0;
      double z = x0, z2 = 0.0, ls2 = 0.0;
      // 1 / a11 = the reciprocal of |a11| with the pivot's sign
      double e0 = copysign(rcp, a11), e1 = 0.0;
      double ls = y0 * e0;
      if (__builtin_expect(p1 != r1, 0)) {
        // ---- off the diagonal: column r1 as well
        const double cv2 = a[r1 & (R - 1)];
        if (wv == r1 / R) col2[lane] = live_value(cv2);
        __syncthreads();
        const double y = col2[lane], ys = col2[sl];
        const double a21 = lane_value(x0, r1), a22 = lane_value(y, r1);
        // explicit fma throughout the block (no contraction left to the
        // compiler), so the oracle's restatement can round the same way;
        // detscale = 1 / |a21| (the largest entry)
        const double detscale = rcp;
        const double detpiv = fma(a11 * detscale, a22, -fabs(a21));
        if (uniform_true(fabs(detpiv) >= fabs(a21) / 2)) {
          two = 1;
          e0 = (a22 * detscale) / detpiv;
          e1 = (-a21 * detscale) / detpiv;
          const double e3 = (a11 * detscale) / detpiv;
          const double l2 = fma(e1, x0, e3 * y), l2s = fma(e1, y0, e3 * ys);
          if (lane / R == wv) t[k + 1][lane] = l2;
          if (lane == k + 1) {
            plp = r1 | 3 << 8;
            pd0 = INFINITY;
            pd1 = e3;
          }
          livem = (lane == r1) ? 0 : livem;
          // column r1 becomes a - y 1 = 0 first and column p1 a - x 1 = 0 next
          z2 = y;
          ls2 = sl == r1 ? 1.0 : sl == p1 ? 0.0 : l2s;
          ls = sl == r1 ? 0.0 : fma(e0, y0, e1 * ys);
        } else {
          // the larger diagonal as a 1x1 pivot
          const bool first = uniform_true(fabs(a11) > fabs(a22));
          e0 = 1.0 / (first ? a11 : a22);
          pv = first ? p1 : r1;
          z = first ? x0 : y;
          ls = (first ? y0 : ys) * e0;
        }
      }
      finish(pv, z, ls, fma(e0, z, e1 * z2), e0, e1, two, z2, ls2);
    } while (k < w);
  }
  if (wv == 1) {
    if (lane < k) {
      lp[lane] = plp & 63;
      kind[lane] = plp >> 8;
      dinv[2 * lane] = pd0;
      dinv[2 * lane + 1] = pd1;
    }
    // the rest: every remaining index a zero pivot, in increasing index
    // order (stop -6: a non-positive pivot of the positive-definite
    // factorization)
    const unsigned long long rest = __builtin_amdgcn_ballot_w64(livem != 0);
    if (stop != 0 && livem) {
      const int kk = k + __popcll(rest & ((1ull << lane) - 1ull));
      lp[kk] = lane;
      kind[kk] = 0;
      dinv[2 * kk] = 0.0;
      dinv[2 * kk + 1] = 0.0;
    }
    if (stop != 0 && lane == 0) {
      if (stop == -6) {
        N.flag = -6;
      } else {
        N.nzero += w - k;
        if (!fp.action) N.flag = -5;
      }
    }
  }
  if (stop != 0)
    for (int kk = k + wv; kk < w; kk += NW) t[kk][lane] = 0.0;
  __syncthreads();
  // ---- write back L_bb (rows permuted into elimination order), D^{-1}, lp;
  // mi[k][i] = L_bb[i][k], the strict lower part in elimination order
  {
    const int li = (lane < w) ? lp[lane] : 0, ki = (lane < w) ? kind[lane] : 0;
    const unsigned long long two = __builtin_amdgcn_ballot_w64(ki == 2);
    const unsigned long long zero = __builtin_amdgcn_ballot_w64(ki == 0);
    gdouble *Lw = (gdouble *)L;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int kk = c0 + j;  // elimination column kk, row `lane`
      const bool low = lane > kk && lane < w && !(lane == kk + 1 && ((two >> kk) & 1));
      const double v = masked(t[kk][li], low);
      mi[kk][lane] = v;
      if (lane >= kk && lane < w)
        Lw[(size_t)(p + kk) * ldl + p + lane] = (lane == kk) ? (((zero >> kk) & 1) ? 0.0 : 1.0) : v;
    }
  }
  for (int j = tid; j < w; j += 64 * NW) {
    N.D[2 * (p + j)] = dinv[2 * j];
    N.D[2 * (p + j) + 1] = dinv[2 * j + 1];
    N.lp[j] = lp[j];
  }
  __syncthreads();
  block_inverse(mi, t, wv, lane, (gdouble *)N.W);
  // permute the variable list (rows of earlier eliminated columns: k_apply)
  const int pv = (tid < w) ? N.perm[p + lp[tid]] : 0;
  __syncthreads();
  if (tid < w) N.perm[p + tid] = pv;
}
template <int NW, bool FIRST, bool C32>
__global__ __launch_bounds__(64 * NW) void k_diag(NodeDev *nodes, int s0,
                                                  int step, FactorParams fp, GatherArgs ga) {
  diag_front<NW, FIRST, C32>(nodes, s0, step, fp, ga);
}

// ---------------------------------------------------------------------------
// Apply the block pivots to the rows below and record the columns that fail
// the a posteriori test.
// The MFMA's output rows are the pivots and its columns the front's rows, so
// a store covers four columns of 16 consecutive rows (whole lines) straight
// from the accumulators; the block inverse is lower triangular, so pivot
// block g takes 4 (g + 1) of the 16 pivot steps.  A column's largest |l| only
// matters against 1/u: lanes compare, a wave's failures go to one 64-bit mask
// by a ballot, and a workgroup without a failure writes none.  (With the
// maxima kept as values, each workgroup reduced 64 columns by shuffles and
// made 256 atomics on the front's 64 words.)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads, 4) void k_apply(NodeDev *nodes, int s0,
                                                    const int *wg_off, int nlvl, int step,
                                                    FactorParams fp) {
  // M = L_bb^{-1} (or the left-rows chunk)
  __shared__ double ms[kBlk][kBlk + 1];
  __shared__ double dv[2 * kBlk + 2];
  __shared__ int lps[kBlk];
  int before;
  const int li = front_of(wg_off, nlvl, blockIdx.x, before);
  if (li < 0) return;
  NodeDev &N = nodes[s0 + li];
  const int nsteps = N.nsteps, p = N.p, w = N.w, ldl = N.ldl, m = N.m;
  double *L = N.L;
  const double *NW = N.W, *ND = N.D;
  loaded(nsteps, p, w, ldl, m, L, NW, ND);
  int local = blockIdx.x - before;
  if (step >= nsteps || w == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // the first nleft workgroups permute rows p..p+w-1 of the eliminated
  // columns left of p into the block's elimination order (64-column chunks)
  const int nleft = step;  // upper bound on ceil(p / 64)
  if (local < nleft) {
    const int cb = local * kBlk;
    if (cb >= p) return;
    gdouble *Lg = (gdouble *)L;
    const int r = lane;
    double v[kBlk / 4];
#pragma unroll
    for (int u = 0; u < kBlk / 4; ++u)
      v[u] = Lg[(size_t)imin(cb + wave + 4 * u, p - 1) * ldl + p + imin(r, w - 1)];
#pragma unroll
    for (int u = 0; u < kBlk / 4; ++u) ms[r][wave + 4 * u] = v[u];
    const int lr = N.lp[imin(r, w - 1)];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kBlk / 4; ++u) {
      const int cc = wave + 4 * u;
      if (r < w && cb + cc < p) Lg[(size_t)(cb + cc) * ldl + p + r] = ms[lr][cc];
    }
    return;
  }
  local -= nleft;
  // ---- rows [rb, rb+64) below the block: X^T = M A21[:, lp]^T on MFMA
  const int r0 = p + w;
  const int rb = r0 + local * kBlk;
  if (rb >= m) return;
  gcdouble *Wg = (gcdouble *)NW;
  gcdouble *Dg = (gcdouble *)ND;
  gcint *lpg = (gcint *)N.lp;
  double wv[kBlk / 4];
#pragma unroll
  for (int u = 0; u < kBlk / 4; ++u) wv[u] = Wg[tid + u * kThreads];
  if (tid < kBlk) lps[tid] = lpg[imin(tid, w - 1)];
  else if (tid >= 2 * kBlk && tid < 4 * kBlk && tid - 2 * kBlk < 2 * w)
    dv[tid - 2 * kBlk] = Dg[2 * p + tid - 2 * kBlk];
  if (tid == 0) {
    dv[2 * w] = 0.0;
    dv[2 * w + 1] = 0.0;
  }
  __syncthreads();
  const int ri = lane & 15, kq = lane >> 4;
  const int r = rb + wave * 16 + ri;  // A row of this lane (fragment layout)
  const bool rok = r < m;
  double av[kBlk / 4];
  {  // unconditional loads (row and pivot clamped into range), unused masked
    const int rc = imin(r, m - 1);
    gcdouble *Lg = (gcdouble *)L;
#pragma unroll
    for (int u = 0; u < kBlk / 4; ++u) {
      const int k = 4 * u + kq;
      av[u] = masked(Lg[(size_t)(p + lps[k]) * ldl + rc], rok && k < w);
    }
  }
#pragma unroll
  for (int u = 0; u < kBlk / 4; ++u)
    ms[(tid + u * kThreads) / kBlk][tid & (kBlk - 1)] = wv[u];
  // descriptor fields once: the global stores below could otherwise alias
  // them and force a reload per iteration
  gdouble *bak = (gdouble *)N.bak;
  gdouble *LD = (gdouble *)N.LD;
  gdouble *X = (gdouble *)N.X;
  gdouble *Lw = (gdouble *)L;
  const int ldbak = N.ldbak, nfs = N.n;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kBlk / 4; ++u) {
    const int k = 4 * u + kq;
    if (rok && k < w) bak[(size_t)k * ldbak + (r - r0)] = av[u];
  }
  double4_t acc[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) acc[g] = (double4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int u = 0; u < kBlk / 4; ++u) {
#pragma unroll
    for (int g = u / 4; g < 4; ++g)  // A[j][k] = M[j][k], zero for k > j
      acc[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(ms[g * 16 + ri][4 * u + kq], av[u], acc[g],
                                                    0, 0, 0);
  }
  // ---- x D^{-1}: acc[g][q] is row r, pivot j = 16 g + 4 q + kq
  const double lim = 1.0 / fp.u;
  // the partner of a 2x2 pivot is one lane group up (down), or the next
  // (previous) register's first (last) group; uniform over the workgroup
  bool two = false;
  for (int j = lane; j < w; j += 64) two = isinf(dv[2 * j]);
  two = __builtin_amdgcn_ballot_w64(two) != 0ull;
  const int up = (lane + 16) & 63, dn = (lane - 16) & 63;
  double nx[17], pvx[17];
  if (two) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      nx[i] = __shfl(acc[i / 4][i % 4], up);
      pvx[i + 1] = __shfl(acc[i / 4][i % 4], dn);
    }
    nx[16] = 0.0;
    pvx[0] = 0.0;
  }
  unsigned long long fail = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int j = 4 * i + kq;
    const double xj = acc[i / 4][i % 4];
    const double d11 = dv[2 * imin(j, w)];
    double y = xj * d11;
    bool zero_piv = d11 == 0.0;
    if (zero_piv) y = (fabs(xj) < fp.small) ? 0.0 : INFINITY * xj;
    if (two) {
      const double xn = kq < 3 ? nx[i] : nx[i + 1], xp = kq > 0 ? pvx[i + 1] : pvx[i];
      if (j + 1 < w && isinf(dv[2 * j + 2])) {
        y = d11 * xj + dv[2 * j + 1] * xn;
        zero_piv = false;
      } else if (j > 0 && j < w && isinf(d11)) {
        y = dv[2 * j - 1] * xp + dv[2 * j + 1] * xj;
      }
    }
    const bool ok = rok && j < w;
    if (ok) {
      Lw[(size_t)(p + j) * ldl + r] = y;
      // L21 D is the product before D^{-1} (zero for a zero pivot): the
      // trailing update's operand for the fully-summed rows, the parent's
      // gather operand for the contribution rows
      const double x = zero_piv ? 0.0 : xj;
      if (r < nfs) X[(size_t)j * ldbak + (r - r0)] = x;
      else if (LD) LD[(size_t)(p + j) * ldl + r] = x;
    }
    // a NaN fails too
    unsigned long long f = __builtin_amdgcn_ballot_w64(ok && !(fabs(y) <= lim));
    if (f) {  // bit 16 k' + row: pivot 4 i + k'
      for (int k = 0; k < 4; ++k)
        if ((f >> (16 * k)) & 0xffffull) fail |= 1ull << (4 * i + k);
    }
  }
  if (fail && lane == 0) atomicOr(&N.fail, fail);
}

// number of block pivots that pass the threshold test (split 2x2 avoided):
// the first column holding an |l| above 1/u; wave-uniform.
__device__ inline int block_npass(const NodeDev &N, int p, int w, unsigned long long fail) {
  int np = fail ? __ffsll((long long)fail) - 1 : w;
  if (np > 0 && np < w) {
    double d11 = N.D[2 * (p + np - 1)], d21 = N.D[2 * (p + np - 1) + 1];
    if (isfinite(d11) && d21 != 0.0) np--;
  }
  return np;
}

// D for pivot k (from the stored D^{-1}); two: 0 = 1x1, 1 = first of 2x2,
// 2 = second of 2x2.
__device__ inline void pivot_d(const double *D, int k, int kend, double &e1, double &e2,
                               int &two) {
  double d11 = D[2 * k];
  if (!isfinite(d11)) {  // second of a 2x2 block
    double a11 = D[2 * (k - 1)], a21 = D[2 * (k - 1) + 1], a22 = D[2 * k + 1];
    double det = a11 * a22 - a21 * a21;
    e1 = -a21 / det;  // off-diagonal of D block
    e2 = a11 / det;   // D22
    two = 2;
  } else if (k + 1 < kend && !isfinite(D[2 * k + 2])) {
    double a11 = d11, a21 = D[2 * k + 1], a22 = D[2 * k + 3];
    double det = a11 * a22 - a21 * a21;
    e1 = a22 / det;   // D11
    e2 = -a21 / det;  // off-diagonal
    two = 1;
  } else {
    e1 = (d11 != 0.0) ? 1.0 / d11 : 0.0;
    e2 = 0.0;
    two = 0;
  }
}

// ---------------------------------------------------------------------------
// Panel update with MFMA:  F[i,j] -= sum_k L[i,a0+k] (L D)[j,a0+k]
// mode 0 (APP step): accepted pivots [p, p+npass) applied to the panel's
//   trailing columns [t0, n), rows [t0, m); failed block columns are restored
//   from the backup first.  The contribution block is NOT touched here: its
//   Schur update is applied lazily when the parent gathers it (k_gather).
// mode 1: subtree roots with a contribution block: all nelim pivots applied
//   to [n, m)^2 so the block can be exported.
// ---------------------------------------------------------------------------
constexpr int kTile = 64;

// lower tiles (I >= J), column-major over J: column J starts at
// J TI - J (J - 1) / 2.  The root of that quadratic in single precision is at
// most a column off, which the two loops correct.
__device__ inline void tile_of(int tile, int TI, int TJ, int &I, int &J) {
  auto first = [&](int j) { return j * TI - j * (j - 1) / 2; };
  const float h = 2.0f * (float)TI + 1.0f;
  J = (int)(0.5f * (h - __builtin_sqrtf(fmaxf(h * h - 8.0f * (float)tile, 0.0f))));
  J = uni(imax(0, imin(J, TJ - 1)));  // the tile number is the workgroup's
  while (J > 0 && first(J) > tile) --J;
  while (J + 1 < TJ && first(J + 1) <= tile) ++J;
  I = J + (tile - first(J));
}

__global__ __launch_bounds__(kThreads, 4) void k_update(NodeDev *nodes, int s0,
                                                     const int *wg_off, int nlvl, int step,
                                                     int mode, FactorParams fp) {
  // 32-pivot K chunks: the two operand tiles take 34 KB, four workgroups a CU
  constexpr int kUpdK = 32;
  __shared__ double As[kTile][kUpdK + 1];
  __shared__ double Bs[kTile][kUpdK + 1];
  int before;
  const int li = front_of(wg_off, nlvl, blockIdx.x, before);
  if (li < 0) return;
  NodeDev &N = nodes[s0 + li];
  const int local = blockIdx.x - before, count = wg_off[li + 1] - before;
  if (local >= count) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int a0, K, t0, cend, fa, fb, p = 0, w = 0;
  if (mode == 0) {
    if (step >= N.nsteps) return;
    p = N.p;
    w = N.w;
    if (w == 0) return;
    int np = fp.posdef ? N.w : block_npass(N, p, w, N.fail);
    if (local == 0 && tid == 0) N.npass = np;
    a0 = p;
    K = np;
    t0 = p + np;
    cend = N.n;
    fa = p + np;
    fb = p + w;
  } else {
    if (!N.is_root || N.m <= N.n) return;
    a0 = 0;
    K = N.nelim;
    t0 = N.n;
    cend = N.m;
    fa = fb = 0;
    if (K <= 0) return;
  }
  const int m = N.m;
  if (m - t0 <= 0 || cend - t0 <= 0) return;
  const int TI = (m - t0 + kTile - 1) / kTile, TJ = (cend - t0 + kTile - 1) / kTile;
  const int ntiles = TJ * TI - TJ * (TJ - 1) / 2;
  const double *D = N.D;
  const int ldl = N.ldl;
  const int Kc = kUpdK;  // K chunk
  // descriptor fields once (the stores below could alias them)
  gdouble *NL = (gdouble *)N.L;
  gdouble *NC = (gdouble *)N.C;
  float __attribute__((address_space(1))) *NCf = (float __attribute__((address_space(1))) *)N.C;
  const bool c32 = fp.c32;  // the contribution block (mode 1 only) is FP32
  gcdouble *dbak = (gcdouble *)N.dbak;
  gcdouble *bak = (gcdouble *)N.bak;
  const int *lpv = N.lp;
  const int nfs = N.n, ldc = N.ldc, ldbak = N.ldbak;
  const int gmax = imin(m, cend) - 1;  // last row a B operand reads
  for (int tile = local; tile < ntiles; tile += count) {
    int I, J;
    tile_of(tile, TI, TJ, I, J);
    const int r0 = t0 + I * kTile, c0 = t0 + J * kTile;
    const bool has_fail = (fb > fa) && (c0 < fb) && (c0 + kTile > fa);
    if (K == 0 && !has_fail) continue;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    double4_t acc[2][2];
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj) acc[bi][bj] = (double4_t){0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < K; k0 += Kc) {
      const int kn = min(Kc, K - k0);
      const int Kp = (kn + 3) & ~3;
      __syncthreads();
      // every thread's loads unconditional (pivot and rows clamped, a 2x2
      // partner always inside the pivots), the entries past the chunk or the
      // front masked to zero.  B = L D keeps the expression of each pivot
      // kind as it is (its rounding is part of the result).
#pragma unroll
      for (int it = 0; it < kTile * kUpdK / kThreads; ++it) {
        const int idx = tid + it * kThreads, i = idx % kTile, kk = idx / kTile;
        const int kc = imin(kk, kn - 1), k = a0 + k0 + kc;
        const int gi = r0 + i, gj = c0 + i, gjc = imin(gj, gmax);
        const double av = masked(NL[(size_t)k * ldl + imin(gi, m - 1)], kk < kn && gi < m);
        double e1, e2;
        int two;
        pivot_d(D, k, a0 + K, e1, e2, two);
        const int ofs = (two == 1) ? 1 : (two == 2) ? -1 : 0;
        const double lk = NL[(size_t)k * ldl + gjc];
        const double lo = NL[(size_t)(k + ofs) * ldl + gjc];
        double bv = (two == 0) ? lk * e1 : (two == 1) ? lk * e1 + lo * e2 : lo * e1 + lk * e2;
        As[i][kk] = av;
        Bs[i][kk] = masked(bv, kk < kn && gj <= gmax);
      }
      __syncthreads();
      for (int kk = 0; kk < Kp; kk += 4) {
        const int kl = kk + (lane >> 4);
#pragma unroll
        for (int bi = 0; bi < 2; ++bi) {
          double av = As[wr + bi * 16 + (lane & 15)][kl];
#pragma unroll
          for (int bj = 0; bj < 2; ++bj) {
            double bv = Bs[wc + bj * 16 + (lane & 15)][kl];
            acc[bi][bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc[bi][bj], 0, 0, 0);
          }
        }
      }
    }
    // element (i,j) of a 16x16 block lives in lane j + 16*(i%4), register i/4
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          int i = wr + bi * 16 + (lane >> 4) + 4 * rg;
          int j = wc + bj * 16 + (lane & 15);
          int gi = r0 + i, gj = c0 + j;
          if (gi < m && gj < cend && gi >= gj && gj >= nfs && c32) {
            float __attribute__((address_space(1))) *dc =
                NCf + (size_t)(gj - nfs) * ldc + (gi - nfs);
            *dc = (float)((double)*dc - acc[bi][bj][rg]);
          } else if (gi < m && gj < cend && gi >= gj) {
            gdouble *dst = (gj < nfs) ? NL + (size_t)gj * ldl + gi
                                      : NC + (size_t)(gj - nfs) * ldc + (gi - nfs);
            double old;
            if (gj >= fa && gj < fb) {
              int jj = gj - p;
              if (gi < p + w) old = dbak[lpv[gi - p] + lpv[jj] * kBlk];
              else old = bak[(size_t)jj * ldbak + (gi - p - w)];
            } else {
              old = *dst;
            }
            *dst = old - acc[bi][bj][rg];
          }
        }
  }
}

// ---------------------------------------------------------------------------
// The APP step's trailing panel update (k_update mode 0) with the MFMA
// operands loaded straight into the 16x16x4 fragment layout.
//
// A step whose 64-column block passed whole (nearly every step of a
// well-ordered matrix): update_tiles.  Output rows are the panel's columns and
// output columns its rows, so a load or store of the panel covers four
// columns of 16 consecutive rows (whole lines).  L D is the apply's product
// before D^{-1}, stored by it (X), so no coefficients or 2x2 partners are
// needed.  A workgroup takes a run of consecutive tiles (column by column);
// all of a tile's loads are out before its products, and each operand
// register is reloaded for the next tile right after its last use, so a tile
// costs its products and not the memory latency.
//
// Other steps (failed columns, a last narrower block): lane i + 16 kq holds row i of A (= L, pivot kq of
// the 4-pivot step) and column i of B = L D for the same pivot; two register
// buffers of two steps each alternate, so the loads of the next 8 pivots are
// in flight during the MFMAs.  The per-pivot coefficients of L D come from
// pivot_d once per workgroup.
// ---------------------------------------------------------------------------
// Addresses are a uniform base plus a 32-bit lane offset inside 64 columns.
__device__ __forceinline__ double load_at(gcdouble *base, unsigned off) { return base[off]; }

__device__ __forceinline__ void update_tiles(gdouble *NL, int ldl, gcdouble *X, int ldx, int p,
                                             int m, int n, int TI, int TJ, int tile, int tend) {
  const int t0 = p + kBlk;
  const int lane = threadIdx.x & 63, wave = uni((int)threadIdx.x >> 6);
  const int ri = lane & 15, kq = lane >> 4;
  const int wr = t0 + (wave >> 1) * 32, wc = (wave & 1) * 32;
  int I, J;
  tile_of(tile, TI, TJ, I, J);
  gcdouble *Lp = (gcdouble *)NL + (size_t)p * ldl;
  double xa[2][kBlk / 4], la[2][kBlk / 4], old[2][2][4];
  unsigned lo[2], xo[2];  // lane offsets of the tile being loaded
  int rn[2];              // its rows
  auto place = [&](int I, int J) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      rn[b] = imin(wr + I * kTile + 16 * b + ri, m - 1);
      lo[b] = (unsigned)(kq * ldl + rn[b]);
      xo[b] = (unsigned)(kq * ldx + imin(t0 + J * kTile + wc + 16 * b + ri, n - 1) - t0);
    }
  };
  auto load_x = [&](int u) {
#pragma unroll
    for (int b = 0; b < 2; ++b) xa[b][u] = load_at(X + (size_t)(4 * u) * ldx, xo[b]);
  };
  auto load_l = [&](int u) {
#pragma unroll
    for (int b = 0; b < 2; ++b) la[b][u] = load_at(Lp + (size_t)(4 * u) * ldl, lo[b]);
  };
  auto load_old = [&](int J) {
    gcdouble *Cb = (gcdouble *)NL + (size_t)(t0 + J * kTile) * ldl;
    const int cl = n - 1 - (t0 + J * kTile);  // last column of the tile column
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int c = imin(wc + 16 * bi + kq + 4 * rg, cl);
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
          old[bi][bj][rg] = load_at(Cb, (unsigned)(c * ldl + rn[bj]));
      }
  };
  place(I, J);
#pragma unroll
  for (int u = 0; u < kBlk / 4; ++u) {
    load_x(u);
    load_l(u);
  }
  load_old(J);
  while (true) {
    // the next tile of the run
    int In = I, Jn = J;
    ++tile;
    const bool more = tile < tend;
    if (more) {
      ++In;
      if (In >= TI) In = ++Jn;
    }
    place(In, Jn);
    double4_t acc[2][2];
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj) acc[bi][bj] = (double4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < kBlk / 4; ++u) {
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
          acc[bi][bj] =
              __builtin_amdgcn_mfma_f64_16x16x4f64(xa[bi][u], la[bj][u], acc[bi][bj], 0, 0, 0);
      if (more) load_l(u);
    }
    if (Jn != J) {
#pragma unroll
      for (int u = 0; u < kBlk / 4; ++u) load_x(u);
    }
    gdouble *Cb = NL + (size_t)(t0 + J * kTile) * ldl;
    const int c0 = t0 + J * kTile, r0 = wr + I * kTile + ri;
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int c = wc + 16 * bi + kq + 4 * rg;
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) {
          const int r = r0 + 16 * bj;
          if (r < m && c0 + c < n && r >= c0 + c)
            Cb[(unsigned)(c * ldl + r)] = old[bi][bj][rg] - acc[bi][bj][rg];
        }
      }
    if (!more) break;
    load_old(Jn);
    I = In;
    J = Jn;
  }
}

// Workgroup `local` of `count` on tiles [first, first + ntiles): a run of
// consecutive tiles each; workgroups go to the eight XCDs in turn, and the runs
// of one XCD's workgroups are neighbours, so that its L2 holds the operands of
// few tile columns.
__device__ __forceinline__ void update_run(gdouble *NL, int ldl, gcdouble *X, int ldx, int p,
                                           int m, int n, int TI, int TJ, int first, int ntiles,
                                           int local, int count) {
  const int used = imin(count, ntiles);
  if (local >= used) return;
  const int c8 = used >> 3;
  const int run = (local < 8 * c8) ? (local & 7) * c8 + (local >> 3) : local;
  const int tb = (int)((int64_t)run * ntiles / used);
  const int te = (int)((int64_t)(run + 1) * ntiles / used);
  update_tiles(NL, ldl, X, ldx, p, m, n, TI, TJ, first + tb, first + te);
}

__global__ __launch_bounds__(kThreads, 2) void k_update_panel(NodeDev *nodes,
                                                           int s0,
                                                           const int *wg_off, int nlvl,
                                                           int step, int ahead,
                                                           FactorParams fp) {
  __shared__ double ce1[kBlk], ce2[kBlk];
  __shared__ int ctwo[kBlk];
  int before;
  const int li = front_of(wg_off, nlvl, blockIdx.x, before);
  if (li < 0) return;
  NodeDev &N = nodes[s0 + li];
  const int local = blockIdx.x - before, count = wg_off[li + 1] - before;
  const int nsteps = N.nsteps, p = N.p, w = N.w, m = N.m, cend = N.n, nl = N.ldl,
            nldbak = N.ldbak;
  double *const nL = N.L, *const nX = N.X;
  const unsigned long long fail = N.fail;
  loaded(count, nsteps, p, w, m, cend, nl, nldbak, nL, nX, fail);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (local >= count || step >= nsteps || w == 0) return;
  const int np = fp.posdef ? w : block_npass(N, p, w, fail);
  if (local == 0 && tid == 0) N.npass = np;
  const int a0 = p, K = np, t0 = p + np, fa = p + np, fb = p + w;
  if (m - t0 <= 0 || cend - t0 <= 0) return;
  const int TI = (m - t0 + kTile - 1) / kTile, TJ = (cend - t0 + kTile - 1) / kTile;
  const int ntiles = TJ * TI - TJ * (TJ - 1) / 2;
  if (np == kBlk) {
    // ahead: the first tile column, the rest beside the next pivot block
    if (ahead && local == 0 && tid == 0) {
      N.ahead_p = p;
      N.ahead_step = step + 1;
    }
    update_run((gdouble *)nL, nl, (gcdouble *)nX, nldbak, p, m, cend, TI, TJ, 0,
               ahead ? TI : ntiles, local, count);
    return;
  }
  {
    const double *D = N.D;
    for (int t = tid; t < K; t += kThreads) {
      double e1, e2;
      int two;
      pivot_d(D, a0 + t, a0 + K, e1, e2, two);
      ce1[t] = e1;
      ce2[t] = e2;
      ctwo[t] = two;
    }
  }
  __syncthreads();
  const int ldl = N.ldl;
  gdouble *NL = (gdouble *)N.L;
  gcdouble *dbak = (gcdouble *)N.dbak;
  gcdouble *bak = (gcdouble *)N.bak;
  const int *lpv = N.lp;
  const int ldbak = N.ldbak;
  const int gmax = imin(m, cend) - 1;  // last row a B operand reads
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int ri = lane & 15, kq = lane >> 4;
  constexpr int KC = 2;  // 4-pivot steps per register buffer
  for (int tile = local; tile < ntiles; tile += count) {
    int I, J;
    tile_of(tile, TI, TJ, I, J);
    const int r0 = t0 + I * kTile, c0 = t0 + J * kTile;
    const bool has_fail = (fb > fa) && (c0 < fb) && (c0 + kTile > fa);
    if (K == 0 && !has_fail) continue;
    double4_t acc[2][2];
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj) acc[bi][bj] = (double4_t){0.0, 0.0, 0.0, 0.0};
    const int ra0 = r0 + wr + ri, ra1 = ra0 + 16, cb0 = c0 + wc + ri, cb1 = cb0 + 16;
    const int ra0c = imin(ra0, m - 1), ra1c = imin(ra1, m - 1);
    const int cb0c = imin(cb0, gmax), cb1c = imin(cb1, gmax);
    // raw operands of KC steps: A rows 0/1, L of B columns 0/1 (pivot and
    // its 2x2 partner)
    double xa0[KC], xa1[KC], xk0[KC], xo0[KC], xk1[KC], xo1[KC];
    double ya0[KC], ya1[KC], yk0[KC], yo0[KC], yk1[KC], yo1[KC];
    auto load = [&](int T0, double *A0, double *A1, double *K0, double *O0, double *K1,
                    double *O1) {
#pragma unroll
      for (int u = 0; u < KC; ++u) {
        const int kc = imin(T0 + 4 * u + kq, K - 1);
        const int two = ctwo[kc];
        const int ofs = (two == 1) ? 1 : (two == 2) ? -1 : 0;
        const size_t ok = (size_t)(a0 + kc) * ldl, oo = (size_t)(a0 + kc + ofs) * ldl;
        A0[u] = NL[ok + ra0c];
        A1[u] = NL[ok + ra1c];
        K0[u] = NL[ok + cb0c];
        O0[u] = NL[oo + cb0c];
        K1[u] = NL[ok + cb1c];
        O1[u] = NL[oo + cb1c];
      }
    };
    auto mfma = [&](int T0, const double *A0, const double *A1, const double *K0,
                    const double *O0, const double *K1, const double *O1) {
#pragma unroll
      for (int u = 0; u < KC; ++u) {
        if (T0 + 4 * u >= K) break;
        const int kk = T0 + 4 * u + kq;
        const bool kok = kk < K;
        const int kc = imin(kk, K - 1);
        const double e1 = ce1[kc], e2 = ce2[kc];
        const int two = ctwo[kc];
        const double b0 = (two == 0) ? K0[u] * e1
                          : (two == 1) ? K0[u] * e1 + O0[u] * e2 : O0[u] * e1 + K0[u] * e2;
        const double b1 = (two == 0) ? K1[u] * e1
                          : (two == 1) ? K1[u] * e1 + O1[u] * e2 : O1[u] * e1 + K1[u] * e2;
        const double av0 = masked(A0[u], kok && ra0 < m), av1 = masked(A1[u], kok && ra1 < m);
        const double bv0 = masked(b0, kok && cb0 <= gmax), bv1 = masked(b1, kok && cb1 <= gmax);
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(av0, bv0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(av0, bv1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(av1, bv0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(av1, bv1, acc[1][1], 0, 0, 0);
      }
    };
    if (K > 0) {
      load(0, xa0, xa1, xk0, xo0, xk1, xo1);
      load(4 * KC, ya0, ya1, yk0, yo0, yk1, yo1);
      for (int T = 0; T < K; T += 8 * KC) {
        if (T > 0) load(T + 4 * KC, ya0, ya1, yk0, yo0, yk1, yo1);
        mfma(T, xa0, xa1, xk0, xo0, xk1, xo1);
        if (T + 4 * KC >= K) break;
        load(T + 8 * KC, xa0, xa1, xk0, xo0, xk1, xo1);
        mfma(T + 4 * KC, ya0, ya1, yk0, yo0, yk1, yo1);
      }
    }
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const int gi = r0 + wr + bi * 16 + kq + 4 * rg, gj = c0 + wc + bj * 16 + ri;
          if (gi < m && gj < cend && gi >= gj) {
            double old;
            if (gj >= fa && gj < fb) {
              const int jj = gj - p;
              old = (gi < p + w) ? dbak[lpv[gi - p] + lpv[jj] * kBlk]
                                 : bak[(size_t)jj * ldbak + (gi - p - w)];
            } else {
              old = NL[(size_t)gj * ldl + gi];
            }
            NL[(size_t)gj * ldl + gi] = old - acc[bi][bj][rg];
          }
        }
  }
}

// The next step's pivot blocks (a workgroup per front, the first ones) beside
// what k_update_panel left of this step's update: when a front's whole block
// passed, the tiles beyond the first tile column, which the pivot blocks do
// not touch.  A pivot block is a chain on one CU (56 us in a 64^3
// factorization) that needs the first tile column only, and the rest of the
// update takes up to 90 us of the other CUs; one after the other they bounded
// every step of a large front.  The launch takes enough LDS for one workgroup
// a CU, `share` of them a front in one round: an update workgroup on a pivot
// block's CU shares its FP64 units (72 us a launch against 63).  64^3 refactor
// + solve 34.9 -> 32.7 ms.  What is left of the update is read from ahead_p and
// ahead_step, as the pivot block moves p on; the apply, which overwrites L21 D
// and moves rows of this step's L, comes after this launch.
__global__ __launch_bounds__(kThreads, 1) void k_update_diag(NodeDev *nodes, int s0, int nlvl,
                                                          int share, int step,
                                                          FactorParams fp) {
  if (blockIdx.x < (unsigned)nlvl) {
    diag_front<kDiagWaves, false, false>(nodes, s0, step + 1, fp, GatherArgs{});
    return;
  }
  const int b = blockIdx.x - nlvl, local = b / nlvl;
  NodeDev &N = nodes[s0 + (b - local * nlvl)];
  const int p = N.ahead_p, tag = N.ahead_step, m = N.m, n = N.n, ldl = N.ldl, ldx = N.ldbak;
  double *const nL = N.L, *const nX = N.X;
  loaded(p, tag, m, n, ldl, ldx, nL, nX);
  if (tag != step + 1) return;
  const int t0 = p + kBlk;
  const int TI = (m - t0 + kTile - 1) / kTile, TJ = (n - t0 + kTile - 1) / kTile;
  update_run((gdouble *)nL, ldl, (gcdouble *)nX, ldx, p, m, n, TI, TJ, TI,
             TJ * TI - TJ * (TJ - 1) / 2 - TI, local, share);
}

// D (not its inverse) per pivot for the lazy contribution update:
// Dd[3k] = D_kk, Dd[3k+1] = D_k,partner, Dd[3k+2] = partner offset.
// ---------------------------------------------------------------------------
// Gather assembly of one level (replaces zero + scatter + extend-add + the
// Schur update of the children's contribution blocks).  A workgroup owns a
// 64x64 tile of one parent front and builds it in registers:
//   for each child in order, the child's trailing index ranges that map into
//   the tile come from the k_maptab tables, and the tile's rows and columns
//   look up their trailing index in LDS; failed (delayed) columns are copied
//   from the child panel; contribution columns are added as C_c minus
//   L21 (D L21)^T on MFMA (K = the child's nelim; operands straight from
//   global memory in the fragment layout), both loaded by the tile's own
//   rows and columns;
//   then the tile's A entries are added (through LDS) and it is stored once.
// The tile stays in the MFMA's registers from the first child to the store.
// Built in LDS, it took three barriers a child and scattered adds: 32^3 27-point
// KKT (150 levels of one front with a block of 64 pivots, where the gather
// streams the contribution block) 77.9 -> 74.5 ms.  What bounds it there is the
// L1's address path (busy 72% of the time), not memory (2.1 TB/s); in FP64 with
// many pivots it is the matrix cores (half the time busy, the rest waits for
// operands).  FP64 needs 166 registers, three workgroups a CU (four spill 25
// registers: 12.4 against 10.7 ms of a 64^3 factorization's gathers); FP32 fits
// four.  Three or four steps a buffer are slower (11.4 and 12.5 ms).
// ---------------------------------------------------------------------------
// Per level, for every child of the level's fronts: the parent position of
// each trailing index (pmap) and, for each 64-row tile of the parent, the
// first trailing index whose parent position reaches the tile (ptab).
constexpr int kMapParts = 8;  // workgroups per front (trailing indices strided over them)
__global__ __launch_bounds__(kThreads) void k_maptab(NodeDev *nodes, int s0,
                                                     const int *child_list) {
  const NodeDev &P = nodes[s0 + blockIdx.x];
  if (P.skip) return;
  const int part = blockIdx.y;
  const int T = (P.m + kGT - 1) / kGT;
  int doff = 0;
  for (int ci = P.cbeg; ci < P.cend; ++ci) {
    NodeDev &c = nodes[child_list[ci]];
    int *tab = P.ctab + (size_t)(ci - P.cbeg) * (T + 1);
    const int cdoff = doff;
    doff += c.n - c.nelim;
    const int nt = c.m - c.nelim;
    for (int t = part * kThreads + threadIdx.x; t < nt; t += kMapParts * kThreads) {
      const int k = c.nelim + t;
      const int pk = child_pos(c, cdoff, P.nd, k);
      c.pmap[t] = pk;
      const int tile = pk / kGT;
      const int prev = (t == 0) ? -1 : child_pos(c, cdoff, P.nd, k - 1) / kGT;
      for (int I = prev + 1; I <= tile; ++I) tab[I] = k;
      if (t == nt - 1)
        for (int I = tile + 1; I <= T; ++I) tab[I] = c.m;
    }
    if (nt == 0 && part == 0)
      for (int I = threadIdx.x; I <= T; I += kThreads) tab[I] = c.m;
  }
}

// Tile of a front's workgroup `local` of `count`, for the lower tiles of a
// T x T front from tile column `jfirst` on.  Workgroups go to the eight XCDs in
// turn, each with an L2 of its own, so workgroups 8 apart take neighbouring
// tiles: of every 1,024 (what runs at once) an XCD takes 128 in sequence, in
// strips of eight tile columns traversed by rows.  The 128 tiles read some 16
// + 8 rows of 64 of the children's L21 and L21 D; down the columns and across
// the XCDs it was up to T + 16.  64^3: 1,396 -> 749 MB read a launch; 32^3
// 27-point KKT, mixed: 78.3 -> 74.4 ms.
constexpr int kXcd = 8, kXcdRun = 128, kStrip = 8;
__device__ inline void gather_place(int local, int count, int T, int jfirst, int &I, int &J) {
  const int base = local & ~(kXcd * kXcdRun - 1), l = local - base;
  const int rem = imin(count - base, kXcd * kXcdRun);
  const int x = l & (kXcd - 1), q = rem / kXcd, r = rem & (kXcd - 1);
  const int at = base + x * q + imin(x, r) + l / kXcd;
  auto first = [&](int j) { return j * T - j * (j - 1) / 2; };  // tiles before column j
  const int start = first(jfirst);
  tile_of(start + at, T, T, I, J);
  const int c = J - ((J - jfirst) & (kStrip - 1)), w = imin(kStrip, T - c);
  int in = start + at - first(c);
  const int tri = w * (w + 1) / 2;
  if (in < tri) {
    I = c;
    while (in > I - c) in -= I++ - c + 1;
    J = c + in;
  } else {
    in -= tri;
    I = c + w + in / w;
    J = c + in % w;
  }
}

// PART 0: every tile of the level's fronts; 1: the first tile column only
// (the pivot block and the rows below it); 2: the remaining tiles
// Returns the front's slot when this workgroup built the front's first
// diagonal tile (0, 0), else -1.

// CT: element type of the contribution blocks (double, or float for the
// mixed-precision factorization, whose Schur terms then run on FP32 MFMA)
template <int PART, typename CT>
__device__ __forceinline__ int gather_tile(
    NodeDev *nodes, int s0, const int *wg_off, int nlvl,
    const int *child_list, const double *aval, const int64_t *asrc, const int *arow,
    const int *acix, const double *scaling, double (&acc)[kGT][kGT + 1], int *inv) {
  constexpr bool F32 = sizeof(CT) == 4;
  int before;
  const int li = front_of(wg_off, nlvl, blockIdx.x, before);
  if (li < 0) return -1;
  const int s = s0 + li;
  NodeDev &P = nodes[s];
  // descriptor fields once, into registers (loads below never wait on them)
  const int m = P.m, n = P.n, nd = P.nd, pldl = P.ldl, pldc = P.ldc;
  const int cbeg = P.cbeg, cend = P.cend;
  gdouble *PL = (gdouble *)P.L;
  CT __attribute__((address_space(1))) *PC = (CT __attribute__((address_space(1))) *)P.C;
  gcint *pctab = (gcint *)P.ctab;
  gcint *prows = (gcint *)P.rows;
  const int64_t *pacol = P.acol;
  const int T = (m + kGT - 1) / kGT;
  // PART 1: the diagonal tile (0, 0); 3: the first tile column's other
  // tiles; 2: the tiles outside the first column; 0: every tile
  const int local = blockIdx.x - before;
  const int count = PART == 1 ? imin(T, 1)
                    : PART == 3 ? T - 1
                    : PART == 2 ? T * (T - 1) / 2
                                : T * (T + 1) / 2;
  if (local >= count) return -1;
  int I, J;
  if constexpr (PART == 1 || PART == 3) {
    I = local + (PART == 3 ? 1 : 0);
    J = 0;
  } else {
    gather_place(local, count, T, PART == 2 ? 1 : 0, I, J);
  }
  const int r0 = I * kGT, c0 = J * kGT;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid < 2 * kGT) {
#pragma unroll
    for (int b = 0; b < 3; ++b) inv[2 * kGT * b + tid] = -1;
  }
  // fully-summed variable list (diagonal tiles own their columns)
  if (I == J) {
    for (int j = c0 + tid; j < min(c0 + kGT, n); j += kThreads) {
      int v;
      if (j >= nd) {
        v = prows[j - nd];
      } else {
        int doff = 0;
        v = -1;
        for (int ci = cbeg; ci < cend; ++ci) {
          const NodeDev &c = nodes[child_list[ci]];
          int nf = c.n - c.nelim;
          if (j >= doff && j < doff + nf) {
            v = c.perm[c.nelim + (j - doff)];
            break;
          }
          doff += nf;
        }
      }
      P.perm[j] = v;
      P.perm0[j] = v;
    }
  }
  // this tile's A entries (entry -> column precomputed), loaded up front
  constexpr int kAE = 1;  // entries per thread held in registers
  const int cs0 = max(c0, nd) - nd, cs1 = min(c0 + kGT, n) - nd;
  int64_t ae0 = 0, ae1 = 0;
  if (cs1 > cs0) {
    ae0 = pacol[cs0];
    ae1 = pacol[cs1];
  }
  double av_[kAE];
  int ar_[kAE], ac_[kAE];
#pragma unroll
  for (int u = 0; u < kAE; ++u) {
    const int64_t e = ae0 + tid + (int64_t)u * kThreads;
    ar_[u] = -1;
    av_[u] = 0.0;
    ac_[u] = 0;
    if (e < ae1) {
      ar_[u] = arow[e] + nd;
      ac_[u] = acix[e];
      av_[u] = aval[asrc[e]];
    }
  }
  __syncthreads();
  // Each wave a 32x32 quadrant in registers: row 16 bi + ri, and with
  // v_mfma_f64_16x16x4_f64 column 16 bj + kq + 4 rg, with
  // v_mfma_f32_16x16x4_f32 column 16 bj + 4 kq + rg (the columns' operand is
  // the first one, so that rows run along the lanes in loads and stores)
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int ri = lane & 15, kq = lane >> 4;
  auto col = [&](int bj, int rg) { return wc + 16 * bj + (F32 ? 4 * kq + rg : kq + 4 * rg); };
  const bool below = I != J || wr >= wc;  // not the quadrant above the diagonal
  double sum[2][2][4];
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) sum[bi][bj][rg] = 0.0;
  int buf = 0;
  for (int ci = cbeg; ci < cend; ++ci) {
    const NodeDev &c = nodes[child_list[ci]];
    const int cn = c.n, cm = c.m, kb = c.nelim, cldl = c.ldl, cldc = c.ldc;
    gcdouble *cL = (gcdouble *)c.L;
    const double *cLD = c.LD;
    const CT *cC = (const CT *)c.C;
    gcint *cpmap = (gcint *)c.pmap;
    if (cm <= kb) continue;
    gcint *tab = pctab + (size_t)(ci - cbeg) * (T + 1);
    const int kr0 = uni(tab[I]), kr1 = uni(tab[I + 1]);
    const int k0 = uni(tab[J]), k1 = uni(tab[J + 1]);
    if (kr1 <= kr0 || k1 <= k0 || kr1 - 1 < k0) continue;
    // the child's trailing index at each of the tile's rows (inv[0..63]) and
    // columns (inv[64..127]), -1 where it has none.  Three copies in turn: one
    // is read while the one before is cleared and the next filled, so a child
    // costs one barrier
    int *iv = inv + 2 * kGT * buf;
    if (wave == 0 && lane < kr1 - kr0) iv[cpmap[kr0 + lane - kb] - r0] = kr0 + lane;
    if (wave == 1 && lane < k1 - k0) iv[kGT + cpmap[k0 + lane - kb] - c0] = k0 + lane;
    __syncthreads();
    const int last = buf == 0 ? 2 : buf - 1;
    if (tid < 2 * kGT) inv[2 * kGT * last + tid] = -1;
    buf = buf == 2 ? 0 : buf + 1;
    if (!below) continue;
    int kr[2], kc[2], kcol[2][4];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      kr[b] = iv[wr + 16 * b + ri];
      kc[b] = iv[kGT + wc + 16 * b + ri];
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) kcol[b][rg] = iv[kGT + col(b, rg)];
    }
    // failed (delayed) columns of the child: from its panel
    if (k0 < cn) {
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
          for (int rg = 0; rg < 4; ++rg) {
            const int k = kcol[bj][rg];
            if (k >= 0 && k < cn && kr[bi] >= k)
              sum[bi][bj][rg] += cL[(size_t)k * cldl + kr[bi]];
          }
    }
    // nothing of the contribution block in this quadrant
    if (!uniform_true(imax(kr[0], kr[1]) >= cn) || !uniform_true(imax(kc[0], kc[1]) >= cn))
      continue;
    // L21 (L21 D)^T, operands in the 16x16x4 fragment layout (lane i+16k
    // holds row i, pivot k) straight from L21 and the child's L21 D; two
    // register buffers alternate so the loads of the next 8 pivots are in
    // flight during the MFMAs.  Mixed precision: operands rounded to FP32,
    // FP32 accumulation
    const int K = kb;
    unsigned oa[2], ob[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      oa[b] = kr[b] >= cn ? (unsigned)(kq * cldl + kr[b]) * 8u : kNoLoad;
      ob[b] = kc[b] >= cn ? (unsigned)(kq * cldl + kc[b]) * 8u : kNoLoad;
    }
    constexpr int KC = 2;  // k-steps (of 4 pivots) per buffer
    struct Operands {
      double a[2][KC], b[2][KC];
    } x, y;
    auto load = [&](int T0, Operands &o) {
#pragma unroll
      for (int u = 0; u < KC; ++u) {
        // the length ends with pivot K - 1: a lane whose pivot T + kq is past
        // it loads nothing
        const int T = T0 + 4 * u;
        const int64_t left = (int64_t)(K - T) * cldl * 8;
        const LoadBuffer<double> Lb((const double *)cL + (size_t)T * cldl, left);
        const LoadBuffer<double> Db(cLD + (size_t)T * cldl, left);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          o.a[b][u] = Lb(oa[b]);
          o.b[b][u] = Db(ob[b]);
        }
      }
    };
    load(0, x);
    // C_c, lower part: all loads issued before any use
    CT cv[2][2][4];
    unsigned has = 0;  // bit 8 bi + 4 bj + rg: the block has the entry
    {
      const int kc0 = imax(k0, cn);
      const LoadBuffer<CT> Cb(cC + (size_t)(kc0 - cn) * cldc,
                              (int64_t)kGT * cldc * sizeof(CT));
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const int k = kcol[bj][rg];
          const unsigned o = (unsigned)((k - kc0) * cldc - cn) * sizeof(CT);
#pragma unroll
          for (int bi = 0; bi < 2; ++bi) {
            const bool in = k >= cn && kr[bi] >= k;
            cv[bi][bj][rg] = Cb(in ? o + (unsigned)kr[bi] * sizeof(CT) : kNoLoad);
            has |= in ? 1u << (8 * bi + 4 * bj + rg) : 0u;
          }
        }
    }
    if constexpr (F32) load(4 * KC, y);
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) sum[bi][bj][rg] += (double)cv[bi][bj][rg];
    if constexpr (!F32) load(4 * KC, y);  // (with the FP64 entries: too many registers)
    typedef typename std::conditional<F32, float4_t, double4_t>::type acc4_t;
    acc4_t g[2][2];
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj) g[bi][bj] = (acc4_t){0, 0, 0, 0};
    auto mfma = [&](int T0, const Operands &o) {
#pragma unroll
      for (int u = 0; u < KC; ++u) {
        if (T0 + 4 * u >= K) break;
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
          for (int bj = 0; bj < 2; ++bj) {
            if constexpr (F32)
              g[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x4f32((float)o.b[bj][u],
                                                               (float)o.a[bi][u], g[bi][bj],
                                                               0, 0, 0);
            else
              g[bi][bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.b[bj][u], o.a[bi][u],
                                                               g[bi][bj], 0, 0, 0);
          }
      }
    };
    for (int t0 = 0; t0 < K; t0 += 8 * KC) {
      if (t0 > 0) load(t0 + 4 * KC, y);
      mfma(t0, x);
      if (t0 + 4 * KC >= K) break;
      load(t0 + 8 * KC, x);
      mfma(t0 + 4 * KC, y);
    }
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const double v = sum[bi][bj][rg] - (double)g[bi][bj][rg];
          sum[bi][bj][rg] = (has >> (8 * bi + 4 * bj + rg) & 1) ? v : sum[bi][bj][rg];
        }
  }
  // a tile without A entries goes to the front from the registers
  if (PART != 1 && ae1 <= ae0) {
    if (below) {
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
          for (int rg = 0; rg < 4; ++rg) {
            const int gr = r0 + wr + 16 * bi + ri, gc = c0 + col(bj, rg);
            if (gr < m && gr >= gc) {
              if (gc < n) PL[(size_t)gc * pldl + gr] = sum[bi][bj][rg];
              else PC[(size_t)(gc - n) * pldc + (gr - n)] = (CT)sum[bi][bj][rg];
            }
          }
    }
    return (I == 0 && J == 0) ? s : -1;
  }
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg)
        acc[wr + 16 * bi + ri][col(bj, rg)] = sum[bi][bj][rg];
  __syncthreads();
  // A entries
#pragma unroll
  for (int u = 0; u < kAE; ++u) {
    const int r = ar_[u];
    if (r < r0 || r >= r0 + kGT) continue;
    const int cc = ac_[u];
    double v = av_[u];
    if (scaling) v *= scaling[prows[r - nd]] * scaling[prows[cc]];
    acc[r - r0][cc + nd - c0] += v;
  }
  for (int64_t e = ae0 + tid + (int64_t)kAE * kThreads; e < ae1; e += kThreads) {
    const int r = arow[e] + nd;
    if (r < r0 || r >= r0 + kGT) continue;
    const int cc = acix[e];
    double v = aval[asrc[e]];
    if (scaling) v *= scaling[prows[r - nd]] * scaling[prows[cc]];
    acc[r - r0][cc + nd - c0] += v;
  }
  __syncthreads();
  // store the tile once: panel columns to L, contribution columns to C
  for (int idx = tid; idx < kGT * kGT; idx += kThreads) {
    const int i = idx % kGT, j = idx / kGT;
    const int gr = r0 + i, gc = c0 + j;
    if (gr < m && gc < m && gr >= gc) {
      if (gc < n) PL[(size_t)gc * pldl + gr] = acc[i][j];
      else PC[(size_t)(gc - n) * pldc + (gr - n)] = (CT)acc[i][j];
    }
  }
  return (I == 0 && J == 0) ? s : -1;
}

template <int PART, typename CT>
__global__ __launch_bounds__(kThreads, sizeof(CT) == 4 ? 4 : 3) void k_gather(
    NodeDev *nodes, int s0, const int *wg_off, int nlvl,
    const int *child_list, const double *aval, const int64_t *asrc, const int *arow,
    const int *acix, const double *scaling) {
  __shared__ double acc[kGT][kGT + 1];
  __shared__ int inv[kGatherInv];
  gather_tile<PART, CT>(nodes, s0, wg_off, nlvl, child_list, aval, asrc, arow, acix,
                        scaling, acc, inv);
}


// ---------------------------------------------------------------------------
// Move failed columns of this step behind the unprocessed candidates:
// disjoint interchanges f_i = p+npass+i <-> u_i = q-ns+i, i < ns = min(nf, nu),
// of rows and columns.  The interchanges are an involution on the front's
// entries, so an entry and its image form a pair that one thread swaps in
// place: (f_i, x) <-> (u_i, x) for every other x, and inside the
// interchanged set (f_i, f_j) <-> (u_i, u_j), j <= i, and (f_i, u_j) <->
// (u_i, f_j), j < i.  One launch, most of them with nothing to do (two
// launches through a gather buffer cost 9.2 us a step, this one 4.6).
// ---------------------------------------------------------------------------
__device__ inline double *swp_at(double *L, int ldl, int a, int b) {
  return L + (size_t)imin(a, b) * ldl + imax(a, b);
}

__global__ __launch_bounds__(kThreads) void k_swap(NodeDev *nodes, int s0,
                                                   const int *wg_off, int nlvl, int step) {
  int before;
  const int li = front_of(wg_off, nlvl, blockIdx.x, before);
  if (li < 0) return;
  NodeDev &N = nodes[s0 + li];
  const int local = blockIdx.x - before, count = wg_off[li + 1] - before;
  const int nsteps = N.nsteps, p = N.p, w = N.w, npass = N.npass, q = N.q;
  loaded(count, nsteps, p, w, npass, q);
  const int f0 = p + npass, pw = p + w;
  const int ns = imin(pw - f0, q - pw);
  if (local >= count || step >= nsteps || w == 0 || ns <= 0) return;
  const int u0 = q - ns, m = N.m, ldl = N.ldl;
  double *L = N.L;
  const int total = ns * m;
  for (int idx = local * kThreads + threadIdx.x; idx < total; idx += count * kThreads) {
    const int i = idx / m, x = idx - i * m;
    int y = x;  // the image of x
    if (x >= f0 && x < f0 + ns) {
      if (x - f0 > i) continue;
      y = u0 + (x - f0);
    } else if (x >= u0 && x < u0 + ns) {
      if (x - u0 >= i) continue;
      y = f0 + (x - u0);
    }
    double *a = swp_at(L, ldl, f0 + i, x), *b = swp_at(L, ldl, u0 + i, y);
    const double t = *a;
    *a = *b;
    *b = t;
  }
  if (local == 0 && threadIdx.x < ns) {
    const int i = threadIdx.x, t = N.perm[f0 + i];
    N.perm[f0 + i] = N.perm[u0 + i];
    N.perm[u0 + i] = t;
  }
}

// ---------------------------------------------------------------------------
// Threshold partial pivoting on the remaining fully-summed columns
// [nelim, n) of the panel, one workgroup per front.  Updates the panel
// columns only; the contribution block is updated afterwards (k_update mode 1).
// ---------------------------------------------------------------------------
// Workgroup size of k_tail.  A level with fewer fronts than CUs gets 16
// waves per front: the TPP trailing update streams the panel from L2 and HBM,
// and more waves keep more of its loads in flight (on a delay-heavy KKT root
// 1024 threads beat 512 by 7% and 256 by 28%; the 216 bytes a lane spills at
// 1024 sit outside the update loops).  Wider levels keep 4 waves per front,
// so that many small fronts share each CU.
constexpr int kTailWide = 1024, kTailNarrow = 256, kTailWideMaxFronts = 256;

// The pivot search and elimination of one column at a time is a chain of
// dependent passes over the trailing panel, so what bounds it is the number
// of memory latencies and barriers a pivot takes.  Each pass issues its loads
// together (clamped indices, a batch of eight a lane), the pivot columns stay in
// LDS for the update, and the update's tiles (8 columns x 128 rows) are dealt
// over the waves in both directions.  With one load at a time, the front's
// pointers read again at each access and the update a column group at a time
// over the whole workgroup, a pivot of a 300-column remainder took 26 us
// (now under 7).
template <int NT>
struct TppShared {
  static constexpr int kCap = (NT >= 1024) ? 2048 : 512;  // rows below a pivot kept in LDS
  // one candidate per wave (batched scan): result code, partner, 2x2 D^-1
  int code[NT / 64];
  int tt[NT / 64];
  double dd[3][NT / 64];
  double red[NT / 64];
  // the batch's rows: per row 64 partial results (largest, second largest,
  // column of the largest with kBig set for an entry not below small)
  double m1[NT / 64][64], m2[NT / 64][64];
  int at[NT / 64][64];
  double x[2][kCap], l[2][kCap];  // the pivot columns, and times D^-1
  // rows [t0, n) of the columns APP eliminated: the row that position holds
  static constexpr int kDefer = 1024;
  int src[kDefer];
};
constexpr int kBig = 1 << 30;

template <int NT>
__device__ double wg_max(double v, TppShared<NT> &sh) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.red[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = sh.red[0];
  for (int i = 1; i < NT / 64; ++i) r = fmax(r, sh.red[i]);
  __syncthreads();
  return r;
}

// The fully-summed panel of a front
struct Panel {
  gdouble *L;
  int ldl;
  __device__ gdouble &operator()(int r, int c) const { return L[(size_t)c * ldl + r]; }
};

constexpr int kTppLoads = 8;  // independent loads a lane issues in a scan

template <int NT>
__device__ double tpp_rc_max(const Panel &A, int col, int nelim, int m, TppShared<NT> &sh) {
  double best = 0.0;
  for (int c = nelim + threadIdx.x; c < col; c += NT) best = fmax(best, fabs(A(col, c)));
  for (int r = col + 1 + threadIdx.x; r < m; r += NT) best = fmax(best, fabs(A(r, col)));
  return wg_max(best, sh);
}

// Symmetric swap of rows/columns c1 and c2: the rows left of c1 from column cb
// on, between c1 and c2 (a column against a row), and the columns below c2, as
// one range.  src (or null): the deferred swaps of the columns before cb
template <int NT>
__device__ void tpp_swap(const Panel &A, int *perm, int cb, int *src, int c1, int c2, int m) {
  if (c1 == c2) return;
  if (c2 < c1) { int t = c1; c1 = c2; c2 = t; }
  const int tid = threadIdx.x, total = m - 2;
  constexpr int kU = 2;
  for (int i0 = cb + tid; i0 < total; i0 += kU * NT) {
    gdouble *p[kU], *q[kU];
    double vp[kU], vq[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = imin(i0 + u * NT, total - 1);
      if (i < c1) {
        p[u] = &A(c1, i);
        q[u] = &A(c2, i);
      } else if (i < c2 - 1) {
        p[u] = &A(i + 1, c1);
        q[u] = &A(c2, i + 1);
      } else {
        p[u] = &A(i + 2, c1);
        q[u] = &A(i + 2, c2);
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      vp[u] = *p[u];
      vq[u] = *q[u];
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
      if (i0 + u * NT < total) {
        *p[u] = vq[u];
        *q[u] = vp[u];
      }
  }
  if (tid == 0) {
    const double t = A(c1, c1);
    A(c1, c1) = A(c2, c2);
    A(c2, c2) = t;
    const int pt = perm[c1];
    perm[c1] = perm[c2];
    perm[c2] = pt;
    if (src) {
      const int st = src[c1 - cb];
      src[c1 - cb] = src[c2 - cb];
      src[c2 - cb] = st;
    }
  }
  __syncthreads();
}

// The deferred row swaps of the columns before t0: rows [t0, t0 + cnt) of each
// column in the order of src, U 64-row pieces; a wave takes NC columns at a time
// (16 loads on their way)
template <int NT, int NC>
__device__ void tpp_rows(const Panel &A, const int *src, int t0, int cnt) {
  constexpr int U = TppShared<NT>::kDefer / 64 / NC;
  const int lane = threadIdx.x & 63;
  int from[U];
#pragma unroll
  for (int u = 0; u < U; ++u) from[u] = t0 + src[imin(64 * u + lane, cnt - 1)];
  for (int c = NC * uni((int)threadIdx.x >> 6); c < t0; c += NC * (NT / 64)) {
    double v[NC][U];
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int u = 0; u < U; ++u) v[k][u] = A(from[u], imin(c + k, t0 - 1));
    __builtin_amdgcn_s_waitcnt(0);  // the columns are read before they are written
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (c + k < t0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (64 * u + lane < cnt) A(t0 + 64 * u + lane, c + k) = v[k][u];
      }
  }
}

constexpr int kTppCols = 8, kTppRows = 128;  // a wave's tile of the TPP update

// Elimination by pivot k (W = 1: D^{-1} = d0; W = 2: [d0 d1; d1 d3] on k, k+1):
// the rows below scaled, then columns [k + W, n) minus their products.  x and l
// hold the unscaled and the scaled pivot columns of row r at r - k - W; in LDS,
// or for longer columns x in the front's workspace and l in the panel.
template <int NT, int W, bool LDS>
__device__ void tpp_elim(const Panel &A, int k, int m, int n, double d0, double d1, double d3,
                         TppShared<NT> &sh, gdouble *w0, gdouble *w1) {
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int base = k + W;
  for (int r = base + tid; r < m; r += NT) {
    const int i = r - base;
    const double x0 = A(r, k);
    if (W == 1) {
      const double l0 = x0 * d0;
      A(r, k) = l0;
      if (LDS) {
        sh.x[0][i] = x0;
        sh.l[0][i] = l0;
      } else {
        w0[i] = x0;
      }
    } else {
      const double x1 = A(r, k + 1);
      const double l0 = d0 * x0 + d1 * x1, l1 = d1 * x0 + d3 * x1;
      A(r, k) = l0;
      A(r, k + 1) = l1;
      if (LDS) {
        sh.x[0][i] = x0;
        sh.x[1][i] = x1;
        sh.l[0][i] = l0;
        sh.l[1][i] = l1;
      } else {
        w0[i] = x0;
        w1[i] = x1;
      }
    }
  }
  __syncthreads();
  const int G = idiv_up(n - base, kTppCols), RB = idiv_up(m - base, kTppRows);
  for (int t = wave; t < G * RB; t += NT / 64) {
    const int rb = t / G, c0 = base + (t - rb * G) * kTppCols;
    const int r0 = c0 + rb * kTppRows;
    if (r0 >= m) continue;
    double s0[kTppCols], s1[kTppCols];
#pragma unroll
    for (int j = 0; j < kTppCols; ++j) {
      const int i = imin(c0 + j, n - 1) - base;
      s0[j] = LDS ? sh.x[0][i] : w0[i];
      if (W == 2) s1[j] = LDS ? sh.x[1][i] : w1[i];
    }
#pragma unroll
    for (int h = 0; h < kTppRows / 64; h += 2) {
      double v[2][kTppCols], l0[2], l1[2];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int r = imin(r0 + 64 * (h + g) + lane, m - 1);
        l0[g] = LDS ? sh.l[0][r - base] : A(r, k);
        if (W == 2) l1[g] = LDS ? sh.l[1][r - base] : A(r, k + 1);
#pragma unroll
        for (int j = 0; j < kTppCols; ++j) v[g][j] = A(r, imin(c0 + j, n - 1));
      }
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int r = r0 + 64 * (h + g) + lane;
#pragma unroll
        for (int j = 0; j < kTppCols; ++j)
          if (c0 + j < n && r >= c0 + j && r < m)
            A(r, c0 + j) = v[g][j] - (W == 1 ? l0[g] * s0[j] : l0[g] * s0[j] + l1[g] * s1[j]);
      }
    }
  }
  if (tid == 0) {
    A(k, k) = 1.0;
    if (W == 2) {
      A(k + 1, k) = 0.0;
      A(k + 1, k + 1) = 1.0;
    }
  }
  __syncthreads();
}

// Whether every entry of column k at and below the diagonal is below small
// (one wave; NaN is not)
__device__ inline bool tpp_wave_small(const Panel &A, int k, int m, double small) {
  const int lane = threadIdx.x & 63;
  int big = 0;
  for (int r0 = k; r0 < m; r0 += 64 * kTppLoads) {
    double v[kTppLoads];
#pragma unroll
    for (int u = 0; u < kTppLoads; ++u) v[u] = A(imin(r0 + 64 * u + lane, m - 1), k);
#pragma unroll
    for (int u = 0; u < kTppLoads; ++u)
      if (!(fabs(v[u]) < small)) big = 1;
  }
  return __ballot(big) == 0;
}

// A batch of TPP candidates p0, p0 + 1, ..., one per wave, tested reading the
// panel only (the tests of a scan are read-only, so the waves of a workgroup
// test consecutive candidates at once and the first that passes is taken, as a
// one-at-a-time scan would).  The decisions are those of the scan's steps
// (ldlt_tpp.cxx:192-259): a zero row/column; else t = the first largest
// |a(p, c)|, c in [nelim, p), the 2x2 test on (t, p) against the largest
// other entries of rows/columns t and p, else the 1x1 test on p.  Two passes:
// row p and column p give the zero test, t, row p's largest entry other
// than t (its second largest: t holds the first largest) and column p's
// largest; row t and column t give t's largest other than p.  Every maximum
// is exact, so the decision equals the one-at-a-time scan's.
//
// The batch's rows are consecutive, so the whole workgroup reads them column
// by column, a 128-byte piece (16 rows) at a time: a wave reading its own row
// touches a line per entry, 64 a load.
template <int NT>
__device__ inline void tpp_batch_rows(const Panel &A, int p0, int nelim, int n, double small,
                                      TppShared<NT> &sh) {
  constexpr int NW = NT / 64, kU = kTppLoads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = lane & (NW - 1), part = wave * (64 / NW) + lane / NW;  // of 64 columns
  const int p = imin(p0 + row, n - 1);
  double m1 = -1.0, m2 = -1.0;
  int at = kBig - 1, big = 0;
  for (int o = nelim + part; o < p0 + NW; o += 64 * kU) {
    double v[kU];
#pragma unroll
    for (int k = 0; k < kU; ++k) v[k] = A(p, imin(o + 64 * k, p - 1));
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      const int c = o + 64 * k;
      const double w = fabs(v[k]);
      if (c < p) {
        if (!(w < small)) big = kBig;
        if (w > m1) {
          m2 = m1;
          m1 = w;
          at = c;
        } else if (w > m2) {
          m2 = w;
        }
      }
    }
  }
  sh.m1[row][part] = m1;
  sh.m2[row][part] = m2;
  sh.at[row][part] = at | big;
}

// The test of candidate p, row of the batch's rows, by one wave, vc the first
// loads of its column.  Returns the code (0 fail, 1 zero column, 2 2x2, 3 1x1),
// wave-uniform; t and the 2x2 D^-1 in the out arguments.
template <int NT>
__device__ inline int tpp_wave_test(const Panel &A, int p, int row, const TppShared<NT> &sh,
                                    const double (&vc)[kTppLoads], int nelim, int m, double u,
                                    double small, int &t_out, double &d0, double &d1,
                                    double &d3) {
  const int lane = threadIdx.x & 63;
  constexpr int kU = kTppLoads;
  const double a22 = uni(vc[0]);  // (lane 0's)
  // pass A: row p over [nelim, p) and column p over [p, m)
  double m1 = sh.m1[row][lane], m2 = sh.m2[row][lane];  // largest, second (-1: none)
  int a1 = sh.at[row][lane];          // first column holding m1
  int big = a1 & kBig;                // some |entry| not below small (NaN counts)
  a1 &= ~kBig;
  double cp = 0.0;                    // column p below the diagonal
  auto column = [&](const double (&v)[kU], int o) {
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      const int r = p + o + 64 * k + lane;
      const double w = fabs(v[k]);
      if (r < m) {
        if (!(w < small)) big = 1;
        if (r > p) cp = fmax(cp, w);
      }
    }
  };
  column(vc, 0);
  for (int o = 64 * kU; o < m - p; o += 64 * kU) {
    double v[kU];
#pragma unroll
    for (int k = 0; k < kU; ++k) v[k] = A(imin(p + o + 64 * k + lane, m - 1), p);
    column(v, o);
  }
  for (int off = 32; off > 0; off >>= 1) {
    const double om1 = __shfl_xor(m1, off), om2 = __shfl_xor(m2, off);
    const int oa1 = __shfl_xor(a1, off);
    if (om1 > m1 || (om1 == m1 && oa1 < a1)) {
      m2 = fmax(om2, m1);
      m1 = om1;
      a1 = oa1;
    } else {
      m2 = fmax(m2, om1);
    }
    cp = fmax(cp, __shfl_xor(cp, off));
  }
  if (!__ballot(big)) return 1;
  // t: the first largest of row p (nelim when every entry is NaN)
  const int t = (a1 == kBig - 1) ? nelim : __builtin_amdgcn_readfirstlane(a1);
  t_out = t;
  // maxp = rc_max(p, skip t): row p without column t, column p below
  double maxp = fmax(fmax(0.0, (a1 == kBig - 1) ? -1.0 : m2), cp);
  maxp = uni(maxp);
  const double a11 = A(t, t), a21 = A(p, t);
  // 2x2 test (t < p)
  const double maxpiv = fmax(fabs(a11), fmax(fabs(a21), fabs(a22)));
  if (!(maxpiv < small)) {
    const double detscale = 1 / maxpiv;
    const double det0 = (a11 * detscale) * a22;
    const double det1 = (a21 * detscale) * a21;
    const double det = det0 - det1;
    const double e0 = (a22 * detscale) / det;
    const double e1 = (-a21 * detscale) / det;
    const double e3 = (a11 * detscale) / det;
    // (pass B only where its result can matter: maxt only adds to the sums)
    if (!(fabs(det) < fmax(small, fmax(fabs(det0 / 2), fabs(det1 / 2)))) &&
        (maxp < small || u * fmax(fabs(e1) * maxp, fabs(e3) * maxp) < 1.0)) {
      // pass B: maxt = rc_max(t, skip p): row t over [nelim, t), column t over
      // (t, m) without row p
      double mt = 0.0;
      for (int o = 0; o < imax(t - nelim, m - t - 1); o += 64 * kU) {
        double vr[kU], vt[kU];
#pragma unroll
        for (int k = 0; k < kU; ++k)
          vr[k] = A(t, imax(imin(nelim + o + 64 * k + lane, t - 1), 0));
#pragma unroll
        for (int k = 0; k < kU; ++k) vt[k] = A(imin(t + 1 + o + 64 * k + lane, m - 1), t);
#pragma unroll
        for (int k = 0; k < kU; ++k) {
          const int c = nelim + o + 64 * k + lane, r = t + 1 + o + 64 * k + lane;
          if (c < t) mt = fmax(mt, fabs(vr[k]));
          if (r < m && r != p) mt = fmax(mt, fabs(vt[k]));
        }
      }
      for (int off = 32; off > 0; off >>= 1) mt = fmax(mt, __shfl_xor(mt, off));
      const double maxt = uni(mt);
      bool ok2;
      if (fmax(maxp, maxt) < small) {
        ok2 = true;
      } else {
        const double x1 = fabs(e0) * maxt + fabs(e1) * maxp;
        const double x2 = fabs(e1) * maxt + fabs(e3) * maxp;
        ok2 = u * fmax(x1, x2) < 1.0;
      }
      if (ok2) {
        d0 = e0;
        d1 = e1;
        d3 = e3;
        return 2;
      }
    }
  }
  const double maxp2 = fmax(maxp, fabs(a21));
  return (fabs(a22) >= u * maxp2) ? 3 : 0;
}

// TPP on the columns [nelim, n) that APP left, by the whole workgroup;
// returns the new nelim (uniform) and stores it in N.nelim.
template <int NT>
__device__ int tpp_front(NodeDev &N, const FactorParams &fp, int nelim, TppShared<NT> &sh) {
  const int n = N.n, m = N.m;
  if (nelim >= n) return nelim;
  // as factor_node_indef (src/ssids/cpu/factor.hxx:77-80): TPP finishes a
  // front with no contribution block (m == n), or every front when the pivot
  // method or the failed-pivot method is TPP
  if (!(fp.pivot_tpp || m == n || fp.tpp_failed)) return nelim;
  const double u = fp.u, small = fp.small;
  const Panel A{(gdouble *)N.L, N.ldl};
  gdouble *D = (gdouble *)N.D, *w0 = (gdouble *)N.bak, *w1 = w0 + N.ldbak;
  int *perm = N.perm;
  const int tid = threadIdx.x, lane = tid & 63, wv = uni(tid >> 6);
  // the row swaps of the columns before t0 wait until the end: they are most of
  // a swap where few of many columns are left (1,500 of 1,800 at a KKT root)
  const int t0 = nelim, cnt = n - t0;
  const bool defer = cnt <= TppShared<NT>::kDefer;
  const int cb = defer ? t0 : 0;
  int *src = defer ? sh.src : nullptr;
  if (defer)
    for (int i = tid; i < cnt; i += NT) sh.src[i] = i;
  bool swapped = false, failed = false;
  auto swap = [&](int c1, int c2) {
    swapped = swapped || c1 != c2;
    tpp_swap<NT>(A, perm, cb, src, c1, c2, m);
  };
  __syncthreads();
  auto zero_pivot = [&] {
    for (int r = nelim + tid; r < m; r += NT) A(r, nelim) = 0.0;
    if (tid == 0) {
      D[2 * nelim] = 0.0;
      D[2 * nelim + 1] = 0.0;
      N.nzero++;
    }
    __syncthreads();
    ++nelim;
  };
  auto pivot1 = [&] {
    const double d = 1.0 / A(nelim, nelim);
    if (tid == 0) {
      D[2 * nelim] = d;
      D[2 * nelim + 1] = 0.0;
    }
    if (m - nelim - 1 <= TppShared<NT>::kCap)
      tpp_elim<NT, 1, true>(A, nelim, m, n, d, 0.0, 0.0, sh, w0, w1);
    else
      tpp_elim<NT, 1, false>(A, nelim, m, n, d, 0.0, 0.0, sh, w0, w1);
    nelim += 1;
  };
  while (nelim < n) {
    // candidates nelim+1, nelim+2, ... in batches of one per wave; the first
    // that passes in order is taken.  In the first batch the last wave tests
    // column nelim for a zero pivot, which goes before any candidate.
    constexpr int NW = NT / 64;
    int c = 0, t = 0, p = 0;
    double d0 = 0.0, d1 = 0.0, d3 = 0.0;
    for (int base = nelim + 1, nc = NW - 1;;) {
      const bool first = nc < NW;
      int code = 0, tw = 0;
      double e0 = 0.0, e1 = 0.0, e3 = 0.0;
      const int pw = imin(base + wv, n - 1);
      double vc[kTppLoads];
      if (base < n) {
        if (wv < nc) {
#pragma unroll
          for (int k = 0; k < kTppLoads; ++k) vc[k] = A(imin(pw + 64 * k + lane, m - 1), pw);
        }
        tpp_batch_rows<NT>(A, base, nelim, n, small, sh);
      }
      if (wv == nc) code = tpp_wave_small(A, nelim, m, small) ? 1 : 0;  // the first batch
      __syncthreads();
      if (wv < nc && base + wv < n)
        code = tpp_wave_test<NT>(A, pw, wv, sh, vc, nelim, m, u, small, tw, e0, e1, e3);
      if (lane == 0) {
        sh.code[wv] = code;
        sh.tt[wv] = tw;
        sh.dd[0][wv] = e0;
        sh.dd[1][wv] = e1;
        sh.dd[2][wv] = e3;
      }
      __syncthreads();
      const unsigned long long hit = __ballot(lane < NW && sh.code[lane & (NW - 1)] != 0);
      if (first && ((hit >> nc) & 1)) {
        c = 1;
        p = nelim;
        break;
      }
      const unsigned long long cand = hit & ((1ull << nc) - 1);
      if (cand != 0) {
        const int w = __builtin_ctzll(cand);
        p = base + w;
        c = sh.code[w];
        t = sh.tt[w];
        d0 = sh.dd[0][w];
        d1 = sh.dd[1][w];
        d3 = sh.dd[2][w];
        break;
      }
      base += nc;
      nc = NW;
      if (base >= n) break;
      __syncthreads();  // every thread has read the batch before it is reused
    }
    __syncthreads();  // (as above)
    if (c == 1) {  // a zero row/column: a zero pivot at nelim
      if (!fp.action) {
        if (tid == 0) N.flag = -5;
        failed = true;
        break;
      }
      swap(p, nelim);
      zero_pivot();
    } else if (c == 2) {
      swap(t, nelim);
      swap(p, nelim + 1);
      if (tid == 0) {
        D[2 * nelim] = d0;
        D[2 * nelim + 1] = d1;
        D[2 * nelim + 2] = INFINITY;
        D[2 * nelim + 3] = d3;
      }
      if (m - nelim - 2 <= TppShared<NT>::kCap)
        tpp_elim<NT, 2, true>(A, nelim, m, n, d0, d1, d3, sh, w0, w1);
      else
        tpp_elim<NT, 2, false>(A, nelim, m, n, d0, d1, d3, sh, w0, w1);
      nelim += 2;
    } else if (c == 3) {
      swap(p, nelim);
      pivot1();
    } else {  // no candidate: 1x1 on column nelim itself, or the end
      const double maxp = tpp_rc_max(A, nelim, nelim, m, sh);
      if (!(fabs(A(nelim, nelim)) >= u * maxp)) break;
      pivot1();
    }
  }
  if (defer && swapped) {
    if (cnt <= 64 * 4) tpp_rows<NT, 4>(A, sh.src, t0, cnt);
    else if (cnt <= 64 * 8) tpp_rows<NT, 2>(A, sh.src, t0, cnt);
    else tpp_rows<NT, 1>(A, sh.src, t0, cnt);
  }
  if (tid == 0 && !failed) N.nelim = nelim;
  return nelim;
}

// ---------------------------------------------------------------------------
// End of a level, one workgroup per front, in order:
//  * the APP result: nelim = p + npass of the last step (nelim_app);
//  * TPP on the columns APP failed (tpp_front);
//  * Dd: D per pivot in the (value, partner value, partner offset) form the
//    gather's L21 D operand uses;
//  * L21 D for the rows [n, m) and the TPP pivots (k_apply wrote it for the
//    APP pivots);
//  * ipos: pre-pivot -> post-pivot position of the fully-summed variables
//    (the variable-indexed scratch is conflict free: the fully-summed
//    variable sets of one level are disjoint).
// Values passed between the phases stay in registers; descriptor fields
// written here are re-read only after a barrier.
// ---------------------------------------------------------------------------
template <int NT>
__global__ __launch_bounds__(NT) void k_tail(NodeDev *nodes, int s0,
                                                   FactorParams fp, int *scratch) {
  __shared__ TppShared<NT> sh;
  NodeDev &N = nodes[s0 + blockIdx.x];
  const int tid = threadIdx.x;
  int nelim;
  {
    const int nsteps = N.nsteps, p = N.p, npass = N.npass, q = N.q, w = N.w;
    nelim = (nsteps > 0) ? p + npass : 0;
    __syncthreads();  // every thread has read the step state
    if (tid == 0) {
      if (nsteps > 0) {
        N.p = nelim;
        N.q = q - (w - npass);
      }
      N.nelim = nelim;
      N.nelim_app = nelim;
    }
    __syncthreads();
  }
  const int t0 = nelim;  // APP pivots end here
  nelim = tpp_front(N, fp, nelim, sh);
  __syncthreads();
  // Dd
  for (int k = tid; k < nelim; k += NT) {
    double e1, e2;
    int two;
    pivot_d(N.D, k, nelim, e1, e2, two);
    if (two == 0) {
      N.Dd[3 * k] = e1;
      N.Dd[3 * k + 1] = 0.0;
      N.Dd[3 * k + 2] = 0.0;
    } else if (two == 1) {
      N.Dd[3 * k] = e1;
      N.Dd[3 * k + 1] = e2;
      N.Dd[3 * k + 2] = 1.0;
    } else {
      N.Dd[3 * k] = e2;
      N.Dd[3 * k + 1] = e1;
      N.Dd[3 * k + 2] = -1.0;
    }
  }
  __syncthreads();
  // L21 D for the TPP pivots
  if (!N.skip && N.LD && t0 < nelim) {
    const int n = N.n, m = N.m, ldl = N.ldl;
    const double *L = N.L, *Dd = N.Dd;
    double *LD = N.LD;
    for (int i = n + tid; i < m; i += NT) {
      for (int t = t0; t < nelim; ++t) {
        const double e = Dd[3 * t], f = Dd[3 * t + 1];
        const int off = (int)Dd[3 * t + 2];
        double v = L[(size_t)t * ldl + i] * e;
        if (off != 0) v += L[(size_t)(t + off) * ldl + i] * f;
        LD[(size_t)t * ldl + i] = v;
      }
    }
  }
  // ipos
  const int n = N.n;
  for (int i = tid; i < n; i += NT) scratch[N.perm[i]] = i;
  __syncthreads();
  for (int j = tid; j < n; j += NT) N.ipos[j] = scratch[N.perm0[j]];
}

// inertia and delay counts over all fronts (integer atomics: deterministic)
constexpr int kStatsWaves = 16, kStatsGroups = 64;
__global__ __launch_bounds__(64 * kStatsWaves) void k_stats(const NodeDev *nodes, int nslots,
                                                            int *counters, int pivot_tpp,
                                                            int tpp_failed) {
  // a wave per front (fronts strided over the grid's waves), a lane per
  // pivot: pivot i is the second member of a 2x2 when its D^{-1} slot holds
  // infinity ([d11, d21 | inf, d22]), the first member when the next one is,
  // a 1x1 otherwise.  Sums go wave -> workgroup (LDS) -> 7 atomics per
  // workgroup (integer: deterministic).
  constexpr int kC = 8;
  __shared__ int red[kStatsWaves][kC];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int c[kC] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int s = blockIdx.x * kStatsWaves + wv; s < nslots; s += gridDim.x * kStatsWaves) {
    const NodeDev &N = nodes[s];
    const int ne = N.nelim;
    gcdouble *d = (gcdouble *)N.D;
    for (int i = lane; i < ne; i += 64) {
      const double a11 = d[2 * i];
      if (!isfinite(a11)) continue;
      if (i + 1 < ne && !isfinite(d[2 * i + 2])) {
        const double a21 = d[2 * i + 1], a22 = d[2 * i + 3];
        c[1]++;
        const double det = a11 * a22 - a21 * a21, tr = a11 + a22;
        if (det < 0) c[0]++;
        else if (tr < 0) c[0] += 2;
      } else {
        if (a11 == 0.0) c[2]++;
        if (a11 < 0.0) c[0]++;
      }
    }
    if (lane == 0) {
      c[3] += N.n - N.nelim;
      // not_first_pass / not_second_pass as src/ssids/cpu/factor.hxx:74-105:
      // the columns APP left (TPP pivoting: the columns TPP left), and the
      // columns a TPP pass over APP's failures left
      if (pivot_tpp) {
        c[4] += N.n - N.nelim;
      } else if (N.nelim_app < N.n) {
        c[4] += N.n - N.nelim_app;
        if (N.m == N.n || tpp_failed) c[7] += N.n - N.nelim;
      }
      c[5] += (N.flag == -5);
      c[6] += (N.flag == -6);
    }
  }
#pragma unroll
  for (int j = 0; j < kC; ++j) {
    int v = c[j];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (lane == 0) red[wv][j] = v;
  }
  __syncthreads();
  if (threadIdx.x < kC) {
    int v = 0;
    for (int q = 0; q < kStatsWaves; ++q) v += red[q][threadIdx.x];
    if (v) atomicAdd(&counters[threadIdx.x], v);
  }
}

// ---------------------------------------------------------------------------
// Level set-up for the static plan (one workgroup): sizes each front of the
// level from its children's results -- nd = sum of the children's failed
// columns, m = sm + nd, n = sn + nd -- and writes the level's launch tables
// (exclusive prefix sums of level_table_count).  A front whose delays exceed
// the capacity its buffers were planned with, or with a skipped child, is
// skipped (m = n = 0, no work) and counted in *overflow when it is the first
// on its path; the host then refactors with the per-level schedule.
// Thread tid sizes fronts tid, tid+1024, ...; after a workgroup barrier each
// wave scans its own share of the tables.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void k_level_setup(NodeDev *nodes, int s0, int nl,
                                                      const int *child_list, int pivot_tpp,
                                                      int S, int *tab, int *overflow) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  for (int li = tid; li < nl; li += 1024) {
    NodeDev &D = nodes[s0 + li];
    int nd = 0, poison = 0;
    for (int k = D.cbeg; k < D.cend; ++k) {
      const NodeDev &c = nodes[child_list[k]];
      nd += c.n - c.nelim;
      poison |= c.skip;
    }
    if (poison || nd > D.ndcap) {
      D.skip = 1;
      D.nd = 0;
      D.m = 0;
      D.n = 0;
      D.nsteps = 0;
      if (!poison) atomicAdd(overflow, 1);
    } else {
      D.skip = 0;
      D.nd = nd;
      D.m = D.sm + nd;
      D.n = D.sn + nd;
      D.nsteps = pivot_tpp ? 0 : (D.n + kBlk - 1) / kBlk;
    }
  }
  __syncthreads();  // the sizes above are visible to every wave
  // wave wv scans tables wv, wv + 16, ... over 64-front chunks, the running
  // sum in a register (no workgroup barrier per table)
  const int ntab = level_tables(S);
  for (int t = wv; t < ntab; t += 16) {
    int *out = tab + (size_t)t * (nl + 1);
    int carry = 0;
    for (int base = 0; base < nl; base += 64) {
      const int li = base + lane;
      int v = 0;
      if (li < nl) {
        const NodeDev &D = nodes[s0 + li];
        v = level_table_count(t, S, D.m, D.n, D.nsteps, D.is_root);
      }
      int x = v;  // inclusive scan within the wave
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
      }
      if (li < nl) out[li] = carry + x - v;
      carry += __shfl(x, 63);
    }
    if (lane == 0) out[nl] = carry;
  }
}

// the per-front results the host needs after a statically planned factor
__global__ void k_pack_nodes(const NodeDev *nodes, int nn, int *out) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nn) return;
  const NodeDev &D = nodes[s];
  int *o = out + 8 * (size_t)s;
  o[0] = D.nd;
  o[1] = D.m;
  o[2] = D.n;
  o[3] = D.nelim;
  o[4] = D.nelim_app;
  o[5] = D.flag;
  o[6] = D.skip;
  o[7] = D.nsteps;
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------
void launch_level_setup(hipStream_t st, NodeDev *nodes, int s0, int nl, const int *child_list,
                        int pivot_tpp, int S, int *tab, int *overflow) {
  if (nl > 0)
    hipLaunchKernelGGL(k_level_setup, dim3(1), dim3(1024), 0, st, nodes, s0, nl, child_list,
                       pivot_tpp, S, tab, overflow);
}
// D^{-1} (two per pivot) and the eliminated variables of every front, into
// contiguous arrays in node order: node i's pivots at [off[i], off[i+1]),
// with off from the host's read-back of each front's nelim
__global__ void k_pack_dperm(const NodeDev *nodes, const int *slot_of, const int64_t *off,
                             int nn, double *out_d, int *out_p) {
  for (int i = blockIdx.x; i < nn; i += gridDim.x) {
    const NodeDev &D = nodes[slot_of[i]];
    const int64_t o = off[i];
    const int ne = (int)(off[i + 1] - o);
    for (int k = threadIdx.x; k < 2 * ne; k += blockDim.x) out_d[2 * o + k] = D.D[k];
    for (int k = threadIdx.x; k < ne; k += blockDim.x) out_p[o + k] = D.perm[k];
  }
}
void launch_pack_dperm(hipStream_t st, const NodeDev *nodes, const int *slot_of,
                       const int64_t *off, int nn, double *out_d, int *out_p) {
  if (nn > 0)
    hipLaunchKernelGGL(k_pack_dperm, dim3(std::min(nn, 4096)), dim3(256), 0, st, nodes,
                       slot_of, off, nn, out_d, out_p);
}
void launch_pack_nodes(hipStream_t st, const NodeDev *nodes, int nn, int *out) {
  if (nn > 0)
    hipLaunchKernelGGL(k_pack_nodes, dim3((nn + 255) / 256), dim3(256), 0, st, nodes, nn, out);
}
void launch_gather_first(hipStream_t st, int nwg, NodeDev *nodes, int s0,
                         const int *wg_off, int nlvl, const int *child_list,
                         const double *aval, const int64_t *asrc, const int *arow,
                         const int *acix, const double *scaling, FactorParams fp) {
  const GatherArgs ga{wg_off, nlvl, child_list, aval, asrc, arow, acix, scaling};
  if (nwg <= 0) return;
  if (fp.c32)
    hipLaunchKernelGGL((k_diag<kDiagWaves, true, true>), dim3(nwg), dim3(64 * kDiagWaves), 0,
                       st, nodes, s0, 0, fp, ga);
  else
    hipLaunchKernelGGL((k_diag<kDiagWaves, true, false>), dim3(nwg), dim3(64 * kDiagWaves), 0,
                       st, nodes, s0, 0, fp, ga);
}
void launch_gather(hipStream_t st, int part, int nwg, NodeDev *nodes, int s0,
                   const int *wg_off, int nlvl, const int *child_list, const double *aval,
                   const int64_t *asrc, const int *arow, const int *acix,
                   const double *scaling, int c32) {
  if (nwg <= 0) return;
  auto kern = c32 ? ((part == 3)   ? k_gather<3, float>
                     : (part == 2) ? k_gather<2, float>
                                   : k_gather<0, float>)
                  : ((part == 3)   ? k_gather<3, double>
                     : (part == 2) ? k_gather<2, double>
                                   : k_gather<0, double>);
  hipLaunchKernelGGL(kern, dim3(nwg), dim3(kThreads), 0, st, nodes, s0, wg_off, nlvl,
                     child_list, aval, asrc, arow, acix, scaling);
}
void launch_maptab(hipStream_t st, int nlvl, NodeDev *nodes, int s0,
                   const int *child_list) {
  if (nlvl > 0)
    hipLaunchKernelGGL(k_maptab, dim3(nlvl, kMapParts), dim3(kThreads), 0, st, nodes, s0,
                       child_list);
}
void launch_tail(hipStream_t st, int nlvl, NodeDev *nodes, int s0, FactorParams fp,
                 int *scratch) {
  if (nlvl <= 0) return;
  if (nlvl < kTailWideMaxFronts)
    hipLaunchKernelGGL(k_tail<kTailWide>, dim3(nlvl), dim3(kTailWide), 0, st, nodes, s0, fp,
                       scratch);
  else
    hipLaunchKernelGGL(k_tail<kTailNarrow>, dim3(nlvl), dim3(kTailNarrow), 0, st, nodes, s0,
                       fp, scratch);
}
void launch_diag(hipStream_t st, int nlvl, NodeDev *nodes, int s0, int step,
                 FactorParams fp) {
  if (nlvl > 0)
    hipLaunchKernelGGL((k_diag<kDiagWaves, false, false>), dim3(nlvl), dim3(64 * kDiagWaves),
                       0, st,
                       nodes, s0, step, fp, GatherArgs{});
}
void launch_apply(hipStream_t st, int nwg, NodeDev *nodes, int s0,
                  const int *wg_off, int nlvl, int step, FactorParams fp) {
  if (nwg > 0)
    hipLaunchKernelGGL(k_apply, dim3(nwg), dim3(kThreads), 0, st, nodes, s0, wg_off,
                       nlvl, step, fp);
}
void launch_update(hipStream_t st, int nwg, NodeDev *nodes, int s0,
                   const int *wg_off, int nlvl, int step, int mode, int ahead,
                   FactorParams fp) {
  if (nwg <= 0) return;
  if (mode == 0)
    hipLaunchKernelGGL(k_update_panel, dim3(nwg), dim3(kThreads), 0, st, nodes, s0, wg_off,
                       nlvl, step, ahead, fp);
  else
    hipLaunchKernelGGL(k_update, dim3(nwg), dim3(kThreads), 0, st, nodes, s0, wg_off,
                       nlvl, step, mode, fp);
}
void launch_update_diag(hipStream_t st, int share, NodeDev *nodes, int s0, int nlvl, int step,
                        FactorParams fp) {
  // LDS past half a CU's: one workgroup a CU
  constexpr unsigned kAlone = 12 << 10;
  hipLaunchKernelGGL(k_update_diag, dim3(nlvl * (1 + share)), dim3(kThreads), kAlone, st,
                     nodes, s0, nlvl, share, step, fp);
}
void launch_swap(hipStream_t st, int nwg, NodeDev *nodes, int s0,
                 const int *wg_off, int nlvl, int step) {
  if (nwg > 0)
    hipLaunchKernelGGL(k_swap, dim3(nwg), dim3(kThreads), 0, st, nodes, s0, wg_off,
                       nlvl, step);
}
void launch_stats(hipStream_t st, const NodeDev *nodes, int nslots, int *counters,
                  const FactorParams &fp) {
  if (nslots > 0)
    hipLaunchKernelGGL(k_stats,
                       dim3(std::min(kStatsGroups, (nslots + kStatsWaves - 1) / kStatsWaves)),
                       dim3(64 * kStatsWaves), 0, st, nodes, nslots, counters, fp.pivot_tpp,
                       fp.tpp_failed);
}

}  // namespace ssids_hip
