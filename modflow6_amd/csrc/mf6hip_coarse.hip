// mf6hip_coarse.hip -- two-level preconditioner for the fused CG: the IMS
// ILU0 / MILU0 preconditioner plus an additive coarse-space correction on
// column aggregates (no counterpart in the reference, whose preconditioners
// are the one-level ILU0 / MILU0 / ILUT of ImsLinearBase.f90:761-1092).
//
//   M^-1 r = ILU0^-1 r + P Ac^-1 P^T r,   Ac = P^T A P
//
// P is piecewise constant: aggregate I holds every layer of an ha x ha block
// of grid columns, and P maps I to each of its cells that is coupled to a
// neighbour (a row with a nonzero off-diagonal).  Decoupled rows -- CHD and
// inactive cells after the sln_ls row fixes, identity rows -- stay with the
// ILU0 part alone, so their heads are left exactly as the one-level solve
// leaves them.  With A symmetric both parts are symmetric and the sum is a
// fixed linear operator: plain PCG applies.
//
// Setup (once per linear solve, the matrix changes every outer iteration):
//   k_tl_cmask     per column: bit k set when cell (k, column) is coupled
//   k_tl_build     one block per aggregate: its row of S = -Ac (diagonal,
//                  west and north couplings on the aggregate grid)
//   k_tl_chain, k_tl_diag, k_tl_prop  Ainv = -S^-1, FP64 or FP32, by block
//                  elimination over the aggregate rows
// (aggregate grids wider than 63 take rocSOLVER's dense dpotrf + dpotri)
// Per CG iteration (after the preconditioner kernels, before the round):
//   the black / red backward preconditioner kernels write each column's sum
//   of the residual over its coupled cells (colsum)
//   k_tl_gather   one block per aggregate: rc = P^T d from colsum
//   k_tl_gemv     one wavefront per coarse row: yc = Ainv rc, partial rc.yc
// and the direction update adds the prolongation: p = z + P yc + beta p.
// rho = d.(z + P yc) = d.z + rc.yc, so the round kernel adds the partials of
// rc.yc to those of d.z.
// Deflated form (preconditioner = 3): z = M^-1 (r - A P yc) + P yc with
// yc = Ac^-1 P^T r, the coarse solve before the sweeps.  P^T r of the
// iteration's new residual is P^T r_old - alpha P^T q: the sweeps' column
// sums of r_old and the SpMV's column sums of q (k_tl_gather with colsq).
// k_tl_defl_setup stores what A P yc needs per cell (the row sum over the
// coupled cells and the couplings across aggregate edges), k_tl_colsum the
// column sums of a replaced residual.
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <cmath>
#include <string>
#include <type_traits>
#include <vector>

#include "mf6hip_handle.h"

#define CK(x)                         \
  do {                                \
    int rc_ = (x);                    \
    if (rc_ != MF6HIP_OK) return rc_; \
  } while (0)

namespace {

__device__ inline double wsum64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// sum over the block (every thread gets it)
__device__ inline double block_sum(double v, double *lds) {
  v = wsum64(v);
  const int w = threadIdx.x >> 6, ln = threadIdx.x & 63;
  __syncthreads();
  if (ln == 0) lds[w] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < (int)(blockDim.x >> 6); i++) s = s + lds[i];
  return s;
}

// bit k of cmask[c * HP + h2]: cell (k, column) has a nonzero off-diagonal
__global__ void k_tl_cmask(Layout L, const double *__restrict__ A, unsigned *__restrict__ cmask) {
  const int NP = L.NP;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < 2 * L.HP;
       t += gridDim.x * blockDim.x) {
    const int c = t >= L.HP;
    const int h2 = t - c * L.HP;
    unsigned m = 0u;
    if (h2 < ncols_of(L, c)) {
      for (int k = 0; k < L.nlay; k++) {
        const int pos = c * L.H + k * L.HP + h2;
        bool cp = false;
        for (int s = S_UP; s <= S_DOWN; s++) cp = cp || A[(size_t)s * NP + pos] != 0.0;
        if (cp) m |= 1u << k;
      }
    }
    cmask[t] = m;
  }
}

// Row I of S = -Ac, compact: S3[3 I] = S(I, I) (cell diagonals plus the
// couplings inside the aggregate), S3[3 I + 1] = S(I, I - 1) (west),
// S3[3 I + 2] = S(I, I - naj) (north); zero where the neighbour does not
// exist.  An aggregate without a coupled cell gets a unit row (its
// restricted residual is always zero).
__global__ void __launch_bounds__(MF6_BLOCK) k_tl_build(Layout L, const double *__restrict__ A,
                                                       const unsigned *__restrict__ cmask,
                                                       TwoLevel T, double *__restrict__ S3) {
  __shared__ double lds[MF6_BLOCK / 64];
  const int I = blockIdx.x;
  if (I >= T.nc) return;
  const int ai = I / T.naj, aj = I - ai * T.naj;
  const int i0 = ai * T.ha, j0 = aj * T.ha;
  const int NP = L.NP;
  double sd = 0.0, sw = 0.0, se = 0.0, sn = 0.0, ss = 0.0, cnt = 0.0;
  for (int t = threadIdx.x; t < T.ha * T.ha; t += blockDim.x) {
    const int i = i0 + t / T.ha, j = j0 + t % T.ha;
    if (i >= L.nrow || j >= L.ncol) continue;
    const int l = i * L.ncol + j, c = (i + j) & 1, h2 = l >> 1;
    const unsigned m = cmask[c * L.HP + h2];
    for (int k = 0; k < L.nlay; k++) {
      if (!((m >> k) & 1u)) continue;
      const int pos = c * L.H + k * L.HP + h2;
      cnt = cnt + 1.0;
      // up / down stay in the column, hence in the aggregate
      sd = sd + A[pos] + A[(size_t)S_UP * NP + pos] + A[(size_t)S_DOWN * NP + pos];
      const double ab = A[(size_t)S_BACK * NP + pos], al = A[(size_t)S_LEFT * NP + pos];
      const double ar = A[(size_t)S_RIGHT * NP + pos], af = A[(size_t)S_FRONT * NP + pos];
      if (i > i0) sd = sd + ab; else sn = sn + ab;
      if (i < i0 + T.ha - 1) sd = sd + af; else ss = ss + af;
      if (j > j0) sd = sd + al; else sw = sw + al;
      if (j < j0 + T.ha - 1) sd = sd + ar; else se = se + ar;
    }
  }
  sd = block_sum(sd, lds);
  sw = block_sum(sw, lds);
  se = block_sum(se, lds);
  sn = block_sum(sn, lds);
  ss = block_sum(ss, lds);
  cnt = block_sum(cnt, lds);
  if (threadIdx.x != 0) return;
  (void)se;
  (void)ss;
  S3[3 * I] = cnt == 0.0 ? 1.0 : -sd;
  S3[3 * I + 1] = (cnt != 0.0 && aj > 0) ? -sw : 0.0;
  S3[3 * I + 2] = (cnt != 0.0 && ai > 0) ? -sn : 0.0;
}

// dense symmetric S (row-major, leading dimension ld; zeroed beforehand),
// for rocSOLVER
__global__ void k_tl_expand(TwoLevel T, const double *__restrict__ S3, double *__restrict__ G) {
  const size_t ld = (size_t)T.ld;
  for (int I = blockIdx.x * blockDim.x + threadIdx.x; I < T.nc; I += gridDim.x * blockDim.x) {
    G[(size_t)I * ld + I] = S3[3 * I];
    if (I % T.naj > 0) {
      G[(size_t)I * ld + I - 1] = S3[3 * I + 1];
      G[(size_t)(I - 1) * ld + I] = S3[3 * I + 1];
    }
    if (I >= T.naj) {
      G[(size_t)I * ld + I - T.naj] = S3[3 * I + 2];
      G[(size_t)(I - T.naj) * ld + I] = S3[3 * I + 2];
    }
  }
}

// ---------------------------------------------------------------------------
// Inverse of S for aggregate grids at most 63 wide.  With the aggregate rows
// as blocks of b = naj unknowns S is block tridiagonal: D_i (tridiagonal) on
// the diagonal and the diagonal matrix E_i between rows i - 1 and i.  With
// the Schur complements from the top and from the bottom
//   F_i = D_i - E_i F_{i-1}^-1 E_i,   G_i = D_i - E_{i+1} G_{i+1}^-1 E_{i+1}
// the blocks of X = S^-1 are
//   X_ii = (F_i + G_i - D_i)^-1,
//   X_ij = -G_i^-1 E_i X_{i-1,j} (i > j),  X_ij = -F_i^-1 E_{i+1} X_{i+1,j} (i < j).
// Only the two chains of b x b inverses are sequential, one workgroup each
// (k_tl_chain); the diagonal blocks invert in parallel (k_tl_diag), and every
// 16 columns of X follow from theirs by nai products with b x b matrices on
// the FP64 matrix cores (k_tl_prop).  S is definite and diagonally dominant
// by construction, so no pivoting is needed.  The banded Cholesky
// factorisation and substitutions that this replaces (one workgroup, then one
// wavefront per column of X, each nai b steps long) took 3.45 + 2.35 ms at
// 63 x 63 aggregates and 0.77 + 0.42 ms at 28 x 37; the four kernels here take
// 1.05 and 0.34 ms.
// ---------------------------------------------------------------------------

constexpr int TL_B = 64;   // padded block

// S3 with every unknown scaled by a power of two sc (exact) that brings its
// diagonal into [1, 4): S3s[3 I ..] as S3, X = sc X_scaled sc.  A diagonal that
// is not positive keeps its value (and is found as a pivot).
__global__ void k_tl_scale(TwoLevel T, const double *__restrict__ S3, double *__restrict__ S3s,
                           double *__restrict__ sc) {
  auto scale = [&](int I) {
    const double d = S3[3 * I];
    return d > 0.0 && d <= 1.7976931348623157e308 ? ldexp(1.0, -(ilogb(d) >> 1)) : 1.0;
  };
  for (int I = blockIdx.x * blockDim.x + threadIdx.x; I < T.nc; I += gridDim.x * blockDim.x) {
    const double s = scale(I);
    sc[I] = s;
    S3s[3 * I] = S3[3 * I] * s * s;
    S3s[3 * I + 1] = I > 0 ? S3[3 * I + 1] * s * scale(I - 1) : 0.0;
    S3s[3 * I + 2] = I >= T.naj ? S3[3 * I + 2] * s * scale(I - T.naj) : 0.0;
  }
}

typedef double d4 __attribute__((ext_vector_type(4)));

// In-place Gauss-Jordan inverse of a b x b symmetric positive definite block
// (identity beyond b) in four waves, four pivots a step on the FP64 matrix
// cores.  Wave w holds rows 16 w .., tile t columns 16 t .., in the layout of
// the matrix results: row 4 e + lane / 16 and column lane % 16 in a[t][e].
// With K the first pivot of a step, P its 4 x 4 block and rows K .. K + 3
// published in rowbuf by their owner (two in turn, one barrier a step):
//   X = rows K .. K + 3 with the identity in the pivot columns   (4 x 64)
//   a(i, :) -= a(i, K ..) P^-1 X, the pivot columns of a taken as zero
//   a(K .., :) = P^-1 X.
// A lane's row value is its operand B as it stands, and by symmetry (a(i, k) =
// a(k, i) for rows still to come, -a(k, i) for rows done) the first element
// of P^-1 times it is its operand A of the update.  P^-1 comes from the LDL^T
// factors of P, which every lane computes, and the solve for the lane's own
// column of the identity.  The owner forms its rows P^-1 X after the next
// pivots are published, beside the next step's factors.  Returns 1 + the first
// pivot that is not positive (0: none); such a pivot is taken as 1.
//
// One pivot at a time (a row through LDS, 16 multiply-adds a lane and a
// barrier) took 0.39 us a pivot, a step here 0.85 us.
__device__ inline int tl_invert(d4 (&a)[4], int b, double (*rowbuf)[4][TL_B]) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, k4 = lane >> 4;
  int first = 0;
  __syncthreads();
  if (wv == 0)
#pragma unroll
    for (int t = 0; t < 4; t++) rowbuf[0][t][lane] = a[t][0];
  __syncthreads();
  auto step = [&](auto KK) {
    constexpr int K = decltype(KK)::value, tk = K / 16, ek = (K / 4) & 3;
    const double(*buf)[TL_B] = rowbuf[(K / 4) & 1];
    double x[4], P[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = i; j < 4; j++) P[i][j] = buf[tk][16 * i + 4 * ek + j];
#pragma unroll
    for (int t = 0; t < 4; t++) x[t] = buf[t][lane];
    const double xw = buf[wv][lane];
    // P = L D L^T: L in the lower part of P, the reciprocals of D in id
    double id[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      double p = P[k][k];
      const bool bad = !(p > 0.0);
      first = bad && first == 0 ? K + k + 1 : first;
      p = bad ? 1.0 : p;
      // 1 / p: the hardware's estimate and two Newton steps
      double ip = __builtin_amdgcn_rcp(p);
      ip = fma(fma(-p, ip, 1.0), ip, ip);
      ip = fma(fma(-p, ip, 1.0), ip, ip);
      id[k] = ip;
#pragma unroll
      for (int i = k + 1; i < 4; i++) P[i][k] = P[k][i] * ip;
#pragma unroll
      for (int i = k + 1; i < 4; i++)
#pragma unroll
        for (int j = i; j < 4; j++) P[i][j] = fma(-P[i][k], P[k][j], P[i][j]);
    }
    // column k4 of P^-1
    double y[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      y[i] = k4 == i ? 1.0 : 0.0;
#pragma unroll
      for (int j = 0; j < i; j++) y[i] = fma(-P[i][j], y[j], y[i]);
    }
#pragma unroll
    for (int i = 3; i >= 0; i--) {
      y[i] = y[i] * id[i];
#pragma unroll
      for (int j = i + 1; j < 4; j++) y[i] = fma(-P[j][i], y[j], y[i]);
    }
    const double pa = c16 == 0 ? y[0] : c16 == 1 ? y[1] : c16 == 2 ? y[2] : c16 == 3 ? y[3] : 0.0;
    const bool pc = (c16 >> 2) == ek;   // a pivot column of tile tk
    const d4 zero = {0.0, 0.0, 0.0, 0.0};
    const double w = __builtin_amdgcn_mfma_f64_16x16x4f64(pa, xw, zero, 0, 0, 0)[0];
    const double f = 16 * wv + c16 < K ? w : -w;
    x[tk] = pc ? (k4 == (c16 & 3) ? 1.0 : 0.0) : x[tk];
#pragma unroll
    for (int e = 0; e < 4; e++) a[tk][e] = pc ? 0.0 : a[tk][e];
#pragma unroll
    for (int t = 0; t < 4; t++)
      a[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(f, x[t], a[t], 0, 0, 0);
    constexpr int K1 = K + 4;
    if (K1 < TL_B && wv == K1 / 16)
#pragma unroll
      for (int t = 0; t < 4; t++) rowbuf[(K1 / 4) & 1][t][lane] = a[t][(K1 / 4) & 3];
    __syncthreads();
    if (wv == tk)
#pragma unroll
      for (int t = 0; t < 4; t++)
        a[t][ek] = __builtin_amdgcn_mfma_f64_16x16x4f64(pa, x[t], zero, 0, 0, 0)[0];
  };
#define MF6_PIV(K) if (K < b) step(std::integral_constant<int, K>{});
  MF6_PIV(0) MF6_PIV(4) MF6_PIV(8) MF6_PIV(12) MF6_PIV(16) MF6_PIV(20) MF6_PIV(24) MF6_PIV(28)
  MF6_PIV(32) MF6_PIV(36) MF6_PIV(40) MF6_PIV(44) MF6_PIV(48) MF6_PIV(52) MF6_PIV(56) MF6_PIV(60)
#undef MF6_PIV
  return first;
}

// column c of the padded diagonal block of aggregate row i: its diagonal and
// the couplings to c - 1 and c + 1 (no branch: a wave that loads ahead must not
// wait at one)
struct TlCol {
  double d, lo, hi;
};
__device__ inline TlCol tl_dcol(const double *__restrict__ S3, int b, int i, int c) {
  const int I = i * b + (c < b ? c : 0), J = i * b + (c + 1 < b ? c + 1 : 0);
  const double d = S3[3 * I], lo = S3[3 * I + 1], hi = S3[3 * J + 1];
  return TlCol{c < b ? d : 1.0, c > 0 && c < b ? lo : 0.0, c + 1 < b ? hi : 0.0};
}
__device__ inline double tl_dentry(const TlCol &v, int r, int c) {
  return r == c ? v.d : r == c - 1 ? v.lo : r == c + 1 ? v.hi : 0.0;
}

// coupling of aggregate (i, r) to (i - 1, r)
__device__ inline double tl_eentry(const double *__restrict__ S3, int b, int nai, int i, int r) {
  const bool in = r < b && i > 0 && i < nai;
  const double v = S3[in ? 3 * (i * b + r) + 2 : 2];
  return in ? v : 0.0;
}

// The two chains: workgroup 0 F_i^-1 for i = 0 .. nai - 1 into Fi, workgroup 1
// G_i^-1 for i = nai - 1 .. 0 into Gi (blocks of b x b, rows b apart).  Bound
// by the dependent latency of the steps (nai b / 4 of them): 0.85 ms at 63 x 63,
// 0.27 at 28 x 37.  info[0] = 1 + the first
// unknown whose pivot is not positive (in the order of the unknowns), else 0.
__global__ void __launch_bounds__(256) k_tl_chain(TwoLevel T, const double *__restrict__ S3,
                                                  double *__restrict__ Fi, double *__restrict__ Gi,
                                                  int *info) {
  __shared__ double rowbuf[2][4][TL_B];
  const int lane = threadIdx.x & 63, c0 = lane & 15;
  const int r0 = 16 * (int)(threadIdx.x >> 6) + (lane >> 4);
  const int b = T.naj, n = T.nai, down = blockIdx.x == 0;
  double *out = down ? Fi : Gi;
  d4 a[4];
  TlCol dn[4];
  double en[4], ec[4];
  int first = 0;
  // the next block's entries are loaded while this one is inverted
  auto load = [&](int s) {
    const int i = down ? s : n - 1 - s, e = down ? i : i + 1;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      ec[t] = tl_eentry(S3, b, n, e, 16 * t + c0);
      en[t] = tl_eentry(S3, b, n, e, r0 + 4 * t);
      dn[t] = tl_dcol(S3, b, i, 16 * t + c0);
    }
  };
  load(0);
#pragma unroll
  for (int t = 0; t < 4; t++) a[t] = d4{0.0, 0.0, 0.0, 0.0};
  for (int s = 0; s < n; s++) {
    const int i = down ? s : n - 1 - s;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        a[t][q] = fma(-en[q] * ec[t], a[t][q], tl_dentry(dn[t], r0 + 4 * q, 16 * t + c0));
    if (s + 1 < n) load(s + 1);
    const int bd = tl_invert(a, b, rowbuf);
    if (bd && !first) first = i * b + bd;
    double *o = out + (size_t)i * b * b;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (r0 + 4 * q < b && 16 * t + c0 < b) o[(r0 + 4 * q) * b + 16 * t + c0] = a[t][q];
  }
  if (down && threadIdx.x == 0) info[0] = first;
}

// X_ii = (D_i - E_i F_{i-1}^-1 E_i - E_{i+1} G_{i+1}^-1 E_{i+1})^-1, one workgroup per i
__global__ void __launch_bounds__(256) k_tl_diag(TwoLevel T, const double *__restrict__ S3,
                                                 const double *__restrict__ Fi,
                                                 const double *__restrict__ Gi,
                                                 double *__restrict__ Xd) {
  __shared__ double rowbuf[2][4][TL_B];
  const int lane = threadIdx.x & 63, c0 = lane & 15;
  const int r0 = 16 * (int)(threadIdx.x >> 6) + (lane >> 4);
  const int b = T.naj, n = T.nai, i = blockIdx.x;
  d4 a[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const int c = 16 * t + c0;
    const TlCol dc = tl_dcol(S3, b, i, c);
    const double ecu = tl_eentry(S3, b, n, i, c), ecd = tl_eentry(S3, b, n, i + 1, c);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int r = r0 + 4 * q;
      const bool in = r < b && c < b;
      const double f = in && i > 0 ? Fi[(size_t)(i - 1) * b * b + r * b + c] : 0.0;
      const double g = in && i + 1 < n ? Gi[(size_t)(i + 1) * b * b + r * b + c] : 0.0;
      double v = tl_dentry(dc, r, c);
      v = fma(-tl_eentry(S3, b, n, i, r) * ecu, f, v);
      a[t][q] = fma(-tl_eentry(S3, b, n, i + 1, r) * ecd, g, v);
    }
  }
  (void)tl_invert(a, b, rowbuf);
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (r0 + 4 * q < b && 16 * t + c0 < b)
        Xd[(size_t)i * b * b + (r0 + 4 * q) * b + 16 * t + c0] = a[t][q];
}

// 16 columns of X below (blockIdx.z = 0, with the diagonal block) or above
// the diagonal block of aggregate row j = blockIdx.x, written as Ainv = -X in
// FP64 or FP32.  Per row block one 64 x 64 by 64 x 16 product on
// v_mfma_f64_16x16x4_f64: wave w takes rows 16 w .., operand A (lane: row
// l % 16, k = l / 16) from the symmetric inverse read by columns, operand B
// (k = l / 16, column l % 16) from LDS, result rows 4 e + l / 16.  The next
// inverse is loaded while the product runs.
template <typename TA>
__global__ void __launch_bounds__(256) k_tl_prop(TwoLevel T, const double *__restrict__ S3,
                                                 const double *__restrict__ Fi,
                                                 const double *__restrict__ Gi,
                                                 const double *__restrict__ Xd,
                                                 const double *__restrict__ sc,
                                                 TA *__restrict__ Ainv) {
  __shared__ double V[2][TL_B][16];
  const int b = T.naj, n = T.nai, j = blockIdx.x, c0 = 16 * (int)blockIdx.y;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & 15, kq = lane >> 4, row = 16 * wv + col;
  const bool low = blockIdx.z == 0, colok = c0 + col < b;
  const int step = low ? 1 : -1;
  TA *oc = Ainv + (size_t)j * b + c0 + col;   // this lane's column
  // columns past the last unknown are zero
  if (low && blockIdx.y == 0)
    for (int e = threadIdx.x; e < b * (T.ld - T.nc); e += 256) {
      const int r = e / (T.ld - T.nc);
      Ainv[(size_t)(j * b + r) * T.ld + T.nc + (e - r * (T.ld - T.nc))] = (TA)0;
    }
  const double *inv = low ? Gi : Fi;
  double an[16], es[4], so[4];
  const double sj = colok ? sc[j * b + c0 + col] : 0.0;
  auto load = [&](int i) {                     // the inverse of block i
#pragma unroll
    for (int t = 0; t < 16; t++) {
      const int k = 4 * t + kq;
      an[t] = (i >= 0 && i < n && k < b && row < b) ? inv[(size_t)i * b * b + k * b + row] : 0.0;
    }
  };
  // rows 16 wv + 4 e + kq of block i: the couplings that multiply them on the
  // way to the next block, and the scales of their results
  auto scale = [&](int i) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = 16 * wv + 4 * e + kq;
      es[e] = tl_eentry(S3, b, n, low ? i + 1 : i, r);
      so[e] = r < b ? sj * sc[i * b + r] : 0.0;
    }
  };
  load(j + step);
  scale(j);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int r = 16 * wv + 4 * e + kq;
    const double x = (r < b && colok) ? Xd[(size_t)j * b * b + r * b + c0 + col] : 0.0;
    V[0][r][col] = es[e] * x;
    if (low && r < b && colok) oc[(size_t)(j * b + r) * T.ld] = (TA)(-x * so[e]);
  }
  __syncthreads();
  int p = 0;
  for (int i = j + step; i >= 0 && i < n; i += step, p ^= 1) {
    double a[16];
#pragma unroll
    for (int t = 0; t < 16; t++) a[t] = an[t];
    load(i + step);
    scale(i);
    d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < 16; t++)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], V[p][4 * t + kq][col], acc, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = 16 * wv + 4 * e + kq;
      V[p ^ 1][r][col] = -es[e] * acc[e];
      if (r < b && colok) oc[(size_t)(i * b + r) * T.ld] = (TA)(acc[e] * so[e]);   // -X
    }
    __syncthreads();
  }
}

// Ainv = -(G^-1) from the lower triangle potri left in G (column-major:
// element (r, c), r >= c, at G[r + c ld]); written in full, FP64 and FP32.
__global__ void k_tl_finish(TwoLevel T, const double *__restrict__ G, double *__restrict__ A64,
                            float *__restrict__ A32) {
  const size_t n = (size_t)T.nc * T.ld;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (size_t)gridDim.x * blockDim.x) {
    const int r = (int)(e / T.ld), c = (int)(e - (size_t)r * T.ld);
    double v = 0.0;
    if (c < T.nc) v = -(r >= c ? G[r + (size_t)c * T.ld] : G[c + (size_t)r * T.ld]);
    if (A64) A64[e] = v;
    if (A32) A32[e] = (float)v;
  }
}

// rc[I] = sum of d over the coupled cells of aggregate I
template <typename TV>
__global__ void __launch_bounds__(MF6_BLOCK) k_tl_restrict(Layout L, const TV *__restrict__ d,
                                                          const unsigned *__restrict__ cmask,
                                                          TwoLevel T, double *__restrict__ rc,
                                                          const KState *st) {
  __shared__ double lds[MF6_BLOCK / 64];
  if (st && st->stop) return;
  for (int I = blockIdx.x; I < T.nc; I += gridDim.x) {
    const int ai = I / T.naj, aj = I - ai * T.naj;
    double s = 0.0;
    for (int t = threadIdx.x; t < T.ha * T.ha; t += blockDim.x) {
      const int i = ai * T.ha + t / T.ha, j = aj * T.ha + t % T.ha;
      if (i >= L.nrow || j >= L.ncol) continue;
      const int l = i * L.ncol + j, c = (i + j) & 1, h2 = l >> 1;
      const unsigned m = cmask[c * L.HP + h2];
      const int base = c * L.H + h2;
      for (int k = 0; k < L.nlay; k++)
        if ((m >> k) & 1u) s = s + (double)d[base + k * L.HP];
    }
    s = block_sum(s, lds);
    if (threadIdx.x == 0) rc[I] = s;
  }
}

// rc[I] = sum of colsum over the columns of aggregate I (fixed order)
__global__ void __launch_bounds__(MF6_BLOCK) k_tl_gather(Layout L, const double *__restrict__ colsum,
                                                        TwoLevel T, double *__restrict__ rc,
                                                        const KState *st,
                                                        const double *__restrict__ colsq = nullptr,
                                                        const double *alpha = nullptr) {
  __shared__ double lds[MF6_BLOCK / 64];
  if (st && st->stop) return;
  // colsq given (colour layout, c HP + l / 2): P^T (r - alpha q); alpha = 0
  // leaves colsq unread
  const double a = colsq ? *alpha : 0.0;
  for (int I = blockIdx.x; I < T.nc; I += gridDim.x) {
    const int ai = I / T.naj, aj = I - ai * T.naj;
    double s = 0.0;
    for (int t = threadIdx.x; t < T.ha * T.ha; t += blockDim.x) {
      const int i = ai * T.ha + t / T.ha, j = aj * T.ha + t % T.ha;
      if (i < L.nrow && j < L.ncol) {
        const int l = i * L.ncol + j;
        double v = colsum[l];
        if (a != 0.0) v = v - a * colsq[((i + j) & 1) * L.HP + (l >> 1)];
        s = s + v;
      }
    }
    s = block_sum(s, lds);
    if (threadIdx.x == 0) rc[I] = s;
  }
}

// The same sums by aggregate-row strips: block (ai, chunk) takes TL_GCH
// consecutive grid columns (whole aggregates) of the strip's ha grid rows,
// one column per lane and every fourth row per wavefront, so each grid
// row's sums are read as whole 64-column segments (and each colour's as two
// interleaved ones) rather than as ha-wide pieces.  Each lane adds its rows
// in order, the four wavefronts' column totals are added in order, and the
// aggregate sums add ha consecutive column totals (fixed order).
constexpr int TL_GCH = 64;
__global__ void __launch_bounds__(4 * TL_GCH) k_tl_gather_rows(Layout L,
                                                              const double *__restrict__ colsum,
                                                              TwoLevel T, double *__restrict__ rc,
                                                              const KState *st,
                                                              const double *__restrict__ colsq,
                                                              const double *alpha) {
  __shared__ double acc[4][TL_GCH];
  if (st && st->stop) return;
  const double a = colsq ? *alpha : 0.0;
  const int per = (TL_GCH / T.ha) * T.ha;   // columns of whole aggregates per block
  const int nag = per / T.ha;
  const int nchunk = (L.ncol + per - 1) / per;
  const int w = threadIdx.x >> 6, ln = threadIdx.x & 63;
  for (int blk = blockIdx.x; blk < T.nai * nchunk; blk += gridDim.x) {
    const int ai = blk / nchunk, ch = blk - ai * nchunk;
    const int j = ch * per + ln;
    const int i0 = ai * T.ha;
    const int i1 = i0 + T.ha < L.nrow ? i0 + T.ha : L.nrow;
    double sum = 0.0;
    if (ln < per && j < L.ncol) {
#pragma unroll 4
      for (int i = i0 + w; i < i1; i += 4) {
        const int l = i * L.ncol + j;
        double v = colsum[l];
        if (a != 0.0) v = v - a * colsq[((i + j) & 1) * L.HP + (l >> 1)];
        sum = sum + v;
      }
    }
    acc[w][ln] = sum;
    __syncthreads();
    if ((int)threadIdx.x < nag) {
      const int aj = ch * nag + (int)threadIdx.x;
      if (aj < T.naj) {
        double t = 0.0;
        for (int q = 0; q < T.ha; q++) {
          const int cq = threadIdx.x * T.ha + q;
          t = t + (((acc[0][cq] + acc[1][cq]) + acc[2][cq]) + acc[3][cq]);
        }
        rc[ai * T.naj + aj] = t;
      }
    }
    __syncthreads();
  }
}

template <typename TA> struct Row4;
template <> struct Row4<float> {
  float4 v;
  __device__ static Row4 load(const float *p) { return Row4{*reinterpret_cast<const float4 *>(p)}; }
  __device__ double dot(const double *x) const {
    return (double)v.x * x[0] + (double)v.y * x[1] + (double)v.z * x[2] + (double)v.w * x[3];
  }
};
template <> struct Row4<double> {
  double2 a, b;
  __device__ static Row4 load(const double *p) {
    return Row4{reinterpret_cast<const double2 *>(p)[0], reinterpret_cast<const double2 *>(p)[1]};
  }
  __device__ double dot(const double *x) const {
    return a.x * x[0] + a.y * x[1] + b.x * x[2] + b.y * x[3];
  }
};

// yc = Ainv rc, one wavefront per row with 16-byte (FP32) / 32-byte (FP64)
// row loads; rc is staged in LDS (ld doubles, zero beyond nc; the row
// entries beyond nc are zero as well).  part[b] = this block's sum of
// rc[I] yc[I]; slots gridDim.x .. nslot-1 are cleared.
constexpr int TL_GEMV_THREADS = MF6_BLOCK;
template <typename TA, typename TV>
__global__ void __launch_bounds__(MF6_BLOCK) k_tl_gemv(TwoLevel T, const TA *__restrict__ Ainv,
                                                      const double *__restrict__ rc,
                                                      TV *__restrict__ yc, double *part,
                                                      int nslot, const KState *st) {
  extern __shared__ double xs[];
  __shared__ double lds[MF6_BLOCK / 64];
  if (st && st->stop) return;
  for (int c = threadIdx.x; c < T.ld; c += blockDim.x) xs[c] = c < T.nc ? rc[c] : 0.0;
  __syncthreads();
  const int w = threadIdx.x >> 6, ln = threadIdx.x & 63;
  const int wpb = blockDim.x >> 6;
  double acc = 0.0;
  for (int I = blockIdx.x * wpb + w; I < T.nc; I += gridDim.x * wpb) {
    const TA *row = Ainv + (size_t)I * T.ld;
    double s0 = 0.0, s1 = 0.0;
    int c = 4 * ln;
    for (; c + 256 < T.ld; c += 512) {
      const Row4<TA> r0 = Row4<TA>::load(row + c);
      const Row4<TA> r1 = Row4<TA>::load(row + c + 256);
      s0 = s0 + r0.dot(xs + c);
      s1 = s1 + r1.dot(xs + c + 256);
    }
    if (c < T.ld) s0 = s0 + Row4<TA>::load(row + c).dot(xs + c);
    const double sr = wsum64(s0 + s1);
    if (ln == 0) {
      yc[I] = (TV)sr;
      acc = acc + xs[I] * (double)(TV)sr;
    }
  }
  acc = block_sum(acc, lds);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = acc;
    for (int e = (int)gridDim.x + blockIdx.x; e < nslot; e += (int)gridDim.x) part[e] = 0.0;
  }
}

// z += P yc (coupled cells)
template <typename TV>
__global__ void k_tl_prolong(Layout L, const unsigned *__restrict__ cmask, TwoLevel T,
                             const TV *__restrict__ yc, TV *__restrict__ z) {
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < 2 * L.HP;
       t += gridDim.x * blockDim.x) {
    const int c = t >= L.HP;
    const int h2 = t - c * L.HP;
    if (h2 >= ncols_of(L, c)) continue;
    const unsigned m = cmask[t];
    if (!m) continue;
    const int l = col_l(L, c, h2);
    const TV y = yc[tl_agg(T, L, l)];
    for (int k = 0; k < L.nlay; k++)
      if ((m >> k) & 1u) {
        const int pos = c * L.H + k * L.HP + h2;
        z[pos] = z[pos] + y;
      }
  }
}

// colsum[l] = sum of d over the coupled cells of grid column l
template <typename TV>
__global__ void k_tl_colsum(Layout L, const TV *__restrict__ d, const unsigned *__restrict__ cmask,
                            double *__restrict__ colsum) {
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < L.HP0 + L.HP1;
       t += gridDim.x * blockDim.x) {
    const int c = t >= L.HP0;
    const int h2 = t - c * L.HP0;
    const unsigned m = cmask[c * L.HP + h2];
    double sum = 0.0;
    for (int k = 0; k < L.nlay; k++)
      if ((m >> k) & 1u) sum = sum + (double)d[c * L.H + k * L.HP + h2];
    colsum[col_l(L, c, h2)] = sum;
  }
}

// the same column sums in the colour layout (c HP + l / 2) the SpMV writes
// the column sums of q in, for the gather check of mf6hip_apply_op
template <typename TV>
__global__ void k_tl_colsum_colour(Layout L, const TV *__restrict__ d,
                                   const unsigned *__restrict__ cmask,
                                   double *__restrict__ colsq) {
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < L.HP0 + L.HP1;
       t += gridDim.x * blockDim.x) {
    const int c = t >= L.HP0;
    const int h2 = t - c * L.HP0;
    const unsigned m = cmask[c * L.HP + h2];
    double sum = 0.0;
    for (int k = 0; k < L.nlay; k++)
      if ((m >> k) & 1u) sum = sum + (double)d[c * L.H + k * L.HP + h2];
    colsq[c * L.HP + h2] = sum;
  }
}

// Position of grid column (i, j) in a row of ns: colour by colour within the
// row (the row's colour-0 cells first), so the lanes of one colour kernel
// read consecutive words.
__host__ __device__ inline int ns_col(const Layout &L, int i, int j) {
  if (((i + j) & 1) == 0) return j >> 1;
  return ((i & 1) ? (L.ncol >> 1) : ((L.ncol + 1) >> 1)) + (j >> 1);
}

// Per cell n (FP64 planes A): s[n] = A(n, n) + sum of A(n, m) over the
// coupled neighbours m (0 on decoupled cells), and the couplings A(n, m) to
// coupled neighbours across aggregate edges into ew / ns (layouts as the
// fused CG reads them: ew [(k nrow + i) 2 naj + 2 aj + e], e = 0 to j - 1
// at the aggregate's first column, 1 to j + 1 at its last; ns [(k 2 nai +
// 2 ai + e) ncol + ns_col(i, j)], the same in i).
__global__ void k_tl_defl_setup(Layout L, const double *__restrict__ A,
                                const unsigned *__restrict__ cmask, TwoLevel T,
                                float *__restrict__ sdiag, float *__restrict__ ew,
                                float *__restrict__ ns) {
  const size_t NP = (size_t)L.NP;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < L.HP0 + L.HP1;
       t += gridDim.x * blockDim.x) {
    const int c = t >= L.HP0;
    const int h2 = t - c * L.HP0;
    const int l = col_l(L, c, h2);
    const int i = l / L.ncol, j = l - i * L.ncol;
    const int ai = i / T.ha, aj = j / T.ha;
    const int ri = i - ai * T.ha, rj = j - aj * T.ha;
    const bool hb = i > 0, hf = i < L.nrow - 1, hl = j > 0, hr = j < L.ncol - 1;
    const unsigned m = cmask[c * L.HP + h2];
    const unsigned *om = cmask + (1 - c) * L.HP;
    const unsigned mb = hb ? om[hn(l, -L.ncol)] : 0u, mf = hf ? om[hn(l, L.ncol)] : 0u;
    const unsigned ml = hl ? om[hn(l, -1)] : 0u, mr = hr ? om[hn(l, 1)] : 0u;
    for (int k = 0; k < L.nlay; k++) {
      const size_t pos = (size_t)c * L.H + (size_t)k * L.HP + h2;
      const bool own = (m >> k) & 1u;
      const double ab = ((mb >> k) & 1u) ? A[2 * NP + pos] : 0.0;
      const double al = ((ml >> k) & 1u) ? A[3 * NP + pos] : 0.0;
      const double ar = ((mr >> k) & 1u) ? A[4 * NP + pos] : 0.0;
      const double af = ((mf >> k) & 1u) ? A[5 * NP + pos] : 0.0;
      const double au = (k > 0 && ((m >> (k - 1)) & 1u)) ? A[1 * NP + pos] : 0.0;
      const double ad = (k + 1 < L.nlay && ((m >> (k + 1)) & 1u)) ? A[6 * NP + pos] : 0.0;
      double sum = A[pos];
      sum = sum + au;
      sum = sum + ab;
      sum = sum + al;
      sum = sum + ar;
      sum = sum + af;
      sum = sum + ad;
      sdiag[pos] = own ? (float)sum : 0.0f;
      const size_t e0 = ((size_t)k * L.nrow + i) * 2 * T.naj + 2 * aj;
      const size_t n0 = ((size_t)k * 2 * T.nai + 2 * ai) * L.ncol + ns_col(L, i, j);
      if (rj == 0 && hl) ew[e0] = own ? (float)al : 0.0f;
      if (rj == T.ha - 1 && hr) ew[e0 + 1] = own ? (float)ar : 0.0f;
      if (ri == 0 && hb) ns[n0] = own ? (float)ab : 0.0f;
      if (ri == T.ha - 1 && hf) ns[n0 + L.ncol] = own ? (float)af : 0.0f;
    }
  }
}

inline int tl_grid(size_t n) {
  size_t g = (n + MF6_BLOCK - 1) / MF6_BLOCK;
  if (g > 65535) g = 65535;
  return g < 1 ? 1 : (int)g;
}

}  // namespace

// Aggregate width and grid: the smallest ha whose aggregate grid has at most
// target coarse unknowns and, where that costs at most a doubling of ha, at
// most 63 aggregates per row (the block that the elimination handles).  The
// default target, sqrt(2 N) within [16, 4096], keeps the coarse GEMV (nc^2
// values per iteration) well below the fine iteration's bytes (~24 N).
TwoLevel mf6hip_tl_shape(const Layout &L, int target) {
  if (target <= 0) {
    target = (int)std::sqrt(2.0 * (double)L.N);
    if (target < 16) target = 16;
    if (target > 4096) target = 4096;
  }
  TwoLevel T{};
  int ha = (int)std::ceil(std::sqrt((double)L.NRC / (double)target));
  if (ha < 1) ha = 1;
  while (((L.nrow + ha - 1) / ha) * ((L.ncol + ha - 1) / ha) > target) ha++;
  const int ha0 = ha;
  while ((L.ncol + ha - 1) / ha > 63 && ha < 2 * ha0) ha++;
  T.ha = ha;
  T.nai = (L.nrow + ha - 1) / ha;
  T.naj = (L.ncol + ha - 1) / ha;
  T.nc = T.nai * T.naj;
  T.ld = (T.nc + 63) / 64 * 64;
  return T;
}

// Allocates every buffer of the two-level preconditioner; tl_ready is set
// only once all of them exist, and a failure frees what was allocated, so
// the next call starts over instead of running on missing buffers.
static int tl_alloc_all(Mf6Handle *h);

int mf6hip_tl_alloc(Mf6Handle *h) {
  if (h->tl_ready) return MF6HIP_OK;
  mf6hip_tl_free(h);
  const int rc = tl_alloc_all(h);
  if (rc != MF6HIP_OK) {
    mf6hip_tl_free(h);
    return rc;
  }
  h->tl_ready = true;
  return MF6HIP_OK;
}

static int tl_alloc_all(Mf6Handle *h) {
  const Layout &L = h->L;
  h->tl = mf6hip_tl_shape(L, h->s.coarse_size);
  const size_t nn = (size_t)h->tl.nc * h->tl.ld;
  // b x b blocks for the block inverse; the dense matrix for rocSOLVER
  const size_t nb = (size_t)h->tl.nc * h->tl.naj;
  const bool wide = h->tl.naj > 63;
  if (hipMalloc((void **)&h->tl_cmask, sizeof(unsigned) * 2 * (size_t)L.HP) != hipSuccess ||
      hipMalloc((void **)&h->tl_G, sizeof(double) * (wide ? nn : nb)) != hipSuccess ||
      hipMalloc((void **)&h->tl_rc, sizeof(double) * h->tl.ld) != hipSuccess ||
      hipMalloc((void **)&h->tl_yc64, sizeof(double) * h->tl.ld) != hipSuccess ||
      hipMalloc((void **)&h->tl_yc32, sizeof(float) * h->tl.ld) != hipSuccess ||
      hipMalloc((void **)&h->tl_info, sizeof(int)) != hipSuccess ||
      hipMalloc((void **)&h->tl_colsum, sizeof(double) * (size_t)L.NRC) != hipSuccess ||
      hipMalloc((void **)&h->tl_S3, sizeof(double) * 7 * (size_t)h->tl.nc) != hipSuccess ||
      (!wide && hipMalloc((void **)&h->tl_Fi, sizeof(double) * nb) != hipSuccess) ||
      (!wide && hipMalloc((void **)&h->tl_Gi, sizeof(double) * nb) != hipSuccess)) {
    mf6hip_set_error("hipMalloc failed (two-level preconditioner)");
    return MF6HIP_EHIP;
  }
  if (h->s.precision == MF6HIP_FP64) {
    if (hipMalloc((void **)&h->tl_A64, sizeof(double) * nn) != hipSuccess) {
      mf6hip_set_error("hipMalloc failed (two-level preconditioner)");
      return MF6HIP_EHIP;
    }
  } else if (hipMalloc((void **)&h->tl_A32, sizeof(float) * nn) != hipSuccess) {
    mf6hip_set_error("hipMalloc failed (two-level preconditioner)");
    return MF6HIP_EHIP;
  }
  if (h->s.preconditioner == 3) {
    const TwoLevel &T = h->tl;
    const size_t new_ = (size_t)L.nlay * L.nrow * 2 * T.naj;
    const size_t nns = (size_t)L.nlay * 2 * T.nai * L.ncol;
    if (hipMalloc((void **)&h->tl_s32, sizeof(float) * (size_t)L.NP) != hipSuccess ||
        hipMalloc((void **)&h->tl_ew, sizeof(float) * new_) != hipSuccess ||
        hipMalloc((void **)&h->tl_ns, sizeof(float) * nns) != hipSuccess ||
        hipMalloc((void **)&h->tl_colsq, sizeof(double) * 2 * (size_t)L.HP) != hipSuccess) {
      mf6hip_set_error("hipMalloc failed (two-level preconditioner)");
      return MF6HIP_EHIP;
    }
    HIPCHK(hipMemsetAsync(h->tl_s32, 0, sizeof(float) * (size_t)L.NP, h->stream));
    HIPCHK(hipMemsetAsync(h->tl_ew, 0, sizeof(float) * new_, h->stream));
    HIPCHK(hipMemsetAsync(h->tl_ns, 0, sizeof(float) * nns, h->stream));
    HIPCHK(hipMemsetAsync(h->tl_colsq, 0, sizeof(double) * 2 * (size_t)L.HP, h->stream));
  }
  rocblas_handle rb = nullptr;
  if (rocblas_create_handle(&rb) != rocblas_status_success) {
    mf6hip_set_error("rocblas_create_handle failed");
    return MF6HIP_EHIP;
  }
  h->tl_blas = rb;
  if (rocblas_set_stream(rb, h->stream) != rocblas_status_success) {
    mf6hip_set_error("rocblas_set_stream failed");
    return MF6HIP_EHIP;
  }
  return MF6HIP_OK;
}

void mf6hip_tl_free(Mf6Handle *h) {
  h->tl_ready = false;
  if (h->tl_blas) rocblas_destroy_handle((rocblas_handle)h->tl_blas);
  h->tl_blas = nullptr;
  void *bufs[] = {h->tl_cmask, h->tl_G, h->tl_rc, h->tl_yc64, h->tl_yc32, h->tl_info,
                  h->tl_A64, h->tl_A32, h->tl_colsum, h->tl_S3, h->tl_Fi, h->tl_Gi,
                  h->tl_s32, h->tl_ew, h->tl_ns, h->tl_colsq};
  for (void *b : bufs)
    if (b) (void)hipFree(b);
  h->tl_cmask = nullptr;
  h->tl_G = h->tl_A64 = h->tl_rc = h->tl_yc64 = nullptr;
  h->tl_A32 = h->tl_yc32 = nullptr;
  h->tl_info = nullptr;
  h->tl_colsum = nullptr;
  h->tl_S3 = h->tl_Fi = h->tl_Gi = nullptr;
  h->tl_s32 = h->tl_ew = h->tl_ns = nullptr;
  h->tl_colsq = nullptr;
}

// Ainv = -S^-1 of the compact rows S3 (aggregate grid at most 63 wide), FP64
// or FP32; Fi, Gi and Xd hold nc naj doubles each, S3 7 nc (the rows, then
// their scaled copy and the scales).
static int tl_block_inverse(const TwoLevel &T, double *S3, double *Fi, double *Gi,
                            double *Xd, double *A64, float *A32, int *dinfo, hipStream_t s) {
  const dim3 grid(T.nai, (T.naj + 15) / 16, 2);
  double *S = S3 + 3 * (size_t)T.nc, *sc = S3 + 6 * (size_t)T.nc;   // scaled rows, scales
  k_tl_scale<<<tl_grid(T.nc), MF6_BLOCK, 0, s>>>(T, S3, S, sc);
  k_tl_chain<<<2, 256, 0, s>>>(T, S, Fi, Gi, dinfo);
  k_tl_diag<<<T.nai, 256, 0, s>>>(T, S, Fi, Gi, Xd);
  if (A64) k_tl_prop<double><<<grid, 256, 0, s>>>(T, S, Fi, Gi, Xd, sc, A64);
  if (A32) k_tl_prop<float><<<grid, 256, 0, s>>>(T, S, Fi, Gi, Xd, sc, A32);
  HIPCHK(hipGetLastError());
  return MF6HIP_OK;
}

// Coarse operator of the current FP64 planes: mask, S = -Ac, its inverse.
int mf6hip_tl_setup(Mf6Handle *h) {
  CK(mf6hip_tl_alloc(h));
  const Layout &L = h->L;
  const TwoLevel &T = h->tl;
  hipStream_t s = h->stream;
  k_tl_cmask<<<tl_grid(2 * (size_t)L.HP), MF6_BLOCK, 0, s>>>(L, h->A, h->tl_cmask);
  k_tl_build<<<T.nc, MF6_BLOCK, 0, s>>>(L, h->A, h->tl_cmask, T, h->tl_S3);
  if (h->s.preconditioner == 3)
    k_tl_defl_setup<<<tl_grid((size_t)L.HP0 + L.HP1), MF6_BLOCK, 0, s>>>(
        L, h->A, h->tl_cmask, T, h->tl_s32, h->tl_ew, h->tl_ns);
  HIPCHK(hipGetLastError());
  int info = 0;
  if (T.naj <= 63) {
    CK(tl_block_inverse(T, h->tl_S3, h->tl_Fi, h->tl_Gi, h->tl_G, h->tl_A64, h->tl_A32,
                        h->tl_info, s));
    HIPCHK(hipMemcpyAsync(&info, h->tl_info, sizeof(int), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
  } else {
    HIPCHK(hipMemsetAsync(h->tl_G, 0, sizeof(double) * (size_t)T.nc * T.ld, s));
    k_tl_expand<<<tl_grid(T.nc), MF6_BLOCK, 0, s>>>(T, h->tl_S3, h->tl_G);
    HIPCHK(hipGetLastError());
    rocblas_handle rb = (rocblas_handle)h->tl_blas;
    if (rocsolver_dpotrf(rb, rocblas_fill_lower, T.nc, h->tl_G, T.ld, h->tl_info) !=
        rocblas_status_success) {
      mf6hip_set_error("rocsolver_dpotrf failed");
      return MF6HIP_EHIP;
    }
    HIPCHK(hipMemcpyAsync(&info, h->tl_info, sizeof(int), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if (info == 0) {
      if (rocsolver_dpotri(rb, rocblas_fill_lower, T.nc, h->tl_G, T.ld, h->tl_info) !=
          rocblas_status_success) {
        mf6hip_set_error("rocsolver_dpotri failed");
        return MF6HIP_EHIP;
      }
      k_tl_finish<<<tl_grid((size_t)T.nc * T.ld), MF6_BLOCK, 0, s>>>(T, h->tl_G, h->tl_A64,
                                                                    h->tl_A32);
      HIPCHK(hipGetLastError());
    }
  }
  if (info != 0) {
    mf6hip_set_error("two-level preconditioner: the coarse matrix is not definite (leading minor " +
                     std::to_string(info) + "); the system must be symmetric definite");
    return MF6HIP_EINVAL;
  }
  return MF6HIP_OK;
}

// The coarse setup of one system whose FP64 planes are A (layout L), into
// caller-owned arrays: cmask (2 HP), S3 (7 nc), Fi / Gi / Xd (nc naj each)
// and the FP32 inverse A32 (nc ld).  For the ensemble solver; aggregate grids
// wider than 63 are not supported there.  Returns the info code of the
// factorisation through *info (0: definite).
int mf6hip_tl_setup_slice(const Layout &L, const double *A, const TwoLevel &T,
                          unsigned *cmask, double *S3, double *Fi, double *Gi, double *Xd,
                          float *A32, int *dinfo, int *info, hipStream_t s) {
  if (T.naj > 63) {
    mf6hip_set_error("ensemble two-level: aggregate grid wider than 63");
    return MF6HIP_EUNSUPPORTED;
  }
  k_tl_cmask<<<tl_grid(2 * (size_t)L.HP), MF6_BLOCK, 0, s>>>(L, A, cmask);
  k_tl_build<<<T.nc, MF6_BLOCK, 0, s>>>(L, A, cmask, T, S3);
  CK(tl_block_inverse(T, S3, Fi, Gi, Xd, nullptr, A32, dinfo, s));
  HIPCHK(hipMemcpyAsync(info, dinfo, sizeof(int), hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  return MF6HIP_OK;
}

// blocks of the coarse GEMV (each writes one partial of rc.yc)
static int tl_gemv_grid(const TwoLevel &T, int nslot) {
  const int rows = TL_GEMV_THREADS / 64;
  int gg = (T.nc + rows - 1) / rows;
  if (gg > nslot) gg = nslot;
  return gg < 1 ? 1 : gg;
}

int mf6hip_tl_nslot(const Mf6Handle *h, int nslot) { return tl_gemv_grid(h->tl, nslot); }

// rc = P^T (colsum - alpha colsq) into tl_rc (alpha null: P^T colsum)
static void launch_tl_gather(Mf6Handle *h, const KState *st, const double *alpha) {
  const TwoLevel &T = h->tl;
  const Layout &L = h->L;
  const double *cq = alpha ? h->tl_colsq : nullptr;
  if (T.ha <= TL_GCH) {
    const int per = (TL_GCH / T.ha) * T.ha;
    int gr = T.nai * ((L.ncol + per - 1) / per);
    if (gr > 4096) gr = 4096;
    k_tl_gather_rows<<<gr, 4 * TL_GCH, 0, h->stream>>>(L, h->tl_colsum, T, h->tl_rc, st, cq,
                                                       alpha);
  } else {
    const int gr = T.nc < 4096 ? T.nc : 4096;
    k_tl_gather<<<gr, MF6_BLOCK, 0, h->stream>>>(L, h->tl_colsum, T, h->tl_rc, st, cq, alpha);
  }
}

// rc = P^T d (from the preconditioner kernels' column sums when d is null,
// else from d itself) ; yc = Ainv rc ; partial rc.yc into part[0 .. nslot)
// With alpha (a device pointer, the deflated form): rc = P^T (d - alpha q)
// from the column sums of d and of q.
template <typename TV>
void mf6hip_tl_enqueue(Mf6Handle *h, const TV *d, TV *yc, double *part, int nslot,
                       const KState *st, const double *alpha) {
  const TwoLevel &T = h->tl;
  hipStream_t s = h->stream;
  int gr = T.nc < 4096 ? T.nc : 4096;
  if (d)
    k_tl_restrict<TV><<<gr, MF6_BLOCK, 0, s>>>(h->L, d, h->tl_cmask, T, h->tl_rc, st);
  else
    launch_tl_gather(h, st, alpha);
  const int gg = tl_gemv_grid(T, nslot);
  const size_t shm = sizeof(double) * (size_t)T.ld;
  if (sizeof(TV) == sizeof(double))
    k_tl_gemv<double, TV><<<gg, TL_GEMV_THREADS, shm, s>>>(T, h->tl_A64, h->tl_rc, yc, part,
                                                           nslot, st);
  else
    k_tl_gemv<float, TV><<<gg, TL_GEMV_THREADS, shm, s>>>(T, h->tl_A32, h->tl_rc, yc, part,
                                                          nslot, st);
}

template void mf6hip_tl_enqueue<double>(Mf6Handle *, const double *, double *, double *, int,
                                        const KState *, const double *);
template void mf6hip_tl_enqueue<float>(Mf6Handle *, const float *, float *, double *, int,
                                       const KState *, const double *);

// column sums of a (replaced) residual d over the coupled cells, for the
// deflated form's first coarse solve after it
template <typename TV>
void mf6hip_tl_colsum(Mf6Handle *h, const TV *d) {
  const Layout &L = h->L;
  k_tl_colsum<TV><<<tl_grid((size_t)L.HP0 + L.HP1), MF6_BLOCK, 0, h->stream>>>(
      L, d, h->tl_cmask, h->tl_colsum);
}

template void mf6hip_tl_colsum<double>(Mf6Handle *, const double *);
template void mf6hip_tl_colsum<float>(Mf6Handle *, const float *);

// z += P yc (the FP64 coarse correction of the last mf6hip_tl_enqueue)
int mf6hip_tl_prolong64(Mf6Handle *h, double *z) {
  k_tl_prolong<double><<<tl_grid(2 * (size_t)h->L.HP), MF6_BLOCK, 0, h->stream>>>(
      h->L, h->tl_cmask, h->tl, h->tl_yc64, z);
  HIPCHK(hipGetLastError());
  return MF6HIP_OK;
}

// Restriction P^T x over the coupled cells two ways, for the parity helper
// mf6hip_apply_op (op 9): out[0, nc) by the deflated iteration's route, the
// gather of column sums with the colour-layout column sums of x as q and
// alpha = 0.75 (so P^T (x - 0.75 x)); out[nc, 2 nc) by k_tl_restrict.  x is
// a device vector in the position layout; out a device array of 2 nc.
int mf6hip_tl_gather_check(Mf6Handle *h, const double *x, double *out) {
  if (!h->tl_cmask || !h->tl_colsq || !h->tl_colsum) {
    mf6hip_set_error("op 9 needs preconditioner = 3 and a loaded system");
    return MF6HIP_EINVAL;
  }
  const Layout &L = h->L;
  const TwoLevel &T = h->tl;
  hipStream_t s = h->stream;
  static const double alpha_host = 0.75;
  double *alpha = h->d_part + 7 * (size_t)MF6_MAXBLK + 16;
  HIPCHK(hipMemcpyAsync(alpha, &alpha_host, sizeof(double), hipMemcpyHostToDevice, s));
  mf6hip_tl_colsum<double>(h, x);
  k_tl_colsum_colour<double><<<tl_grid((size_t)L.HP0 + L.HP1), MF6_BLOCK, 0, s>>>(
      L, x, h->tl_cmask, h->tl_colsq);
  launch_tl_gather(h, nullptr, alpha);
  HIPCHK(hipMemcpyAsync(out, h->tl_rc, sizeof(double) * T.nc, hipMemcpyDeviceToDevice, s));
  const int gr = T.nc < 4096 ? T.nc : 4096;
  k_tl_restrict<double><<<gr, MF6_BLOCK, 0, s>>>(L, x, h->tl_cmask, T, out + T.nc, nullptr);
  HIPCHK(hipGetLastError());
  return MF6HIP_OK;
}

// z += P Ainv P^T r on device vectors (FP64): the coarse part of M^-1 r for
// the parity helper mf6hip_apply_op
int mf6hip_tl_apply64(Mf6Handle *h, const double *r, double *z) {
  if (!h->tl_A64) {
    mf6hip_set_error("the FP64 coarse inverse exists for precision FP64 only");
    return MF6HIP_EINVAL;
  }
  double *part = h->d_part + 5 * (size_t)MF6_MAXBLK;
  mf6hip_tl_enqueue<double>(h, r, h->tl_yc64, part, MF6_MAXBLK, nullptr);
  k_tl_prolong<double><<<tl_grid(2 * (size_t)h->L.HP), MF6_BLOCK, 0, h->stream>>>(
      h->L, h->tl_cmask, h->tl, h->tl_yc64, z);
  HIPCHK(hipGetLastError());
  return MF6HIP_OK;
}
