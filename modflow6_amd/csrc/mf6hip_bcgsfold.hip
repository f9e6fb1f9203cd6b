// mf6hip_bcgsfold.hip -- BiCGSTAB (ims_base_bcgs, src/Solution/LinearMethods/
// ImsLinearBase.f90:249-549) with the ILU0 sweeps, one column or one chunk of
// a column per thread: the FP64 solve, and the FP32 inner solves of the mixed
// one.
//
// One kernel per reference vector pass (run_bcgs) is eighteen launches an
// iteration, one cell per thread with its index arithmetic, and four
// one-block reductions over thousands of partials (5 to 16 us each).  Here an
// iteration is nine kernels:
//
//   k_b_red    p = d + beta (p - omega v) (red cells), forward sweep of the red
//              columns; beta from the partials of dhat.d
//   k_b_black  the same of the black columns, forward and backward sweep
//   k_b_bwd    backward sweep of the red columns: phat
//   k_b_mv     v = A phat, partials of dhat.v
//   k_b_red, k_b_black, k_b_bwd   q = d - alpha v, qhat; alpha from the partials
//   k_b_mv     t = A qhat, partials of t.q and t.t
//   k_b_upd    omega from the partials; x += alpha phat + omega qhat,
//              d = q - omega t; partials of the maxima, d.d and dhat.d
//
// Every workgroup of a kernel that needs a scalar adds the partials itself, in
// the same order (the same bits everywhere); on grids with many partials a
// squeeze to 256 comes first.  Extra workgroups of k_b_red reduce what the
// convergence test needs, one of k_b_black runs it; on the largest grids, where the
// two sweeps before that answer cost more than a launch, k_b_test ends the
// iteration with it.  The arithmetic of every
// vector element is that of the one-pass kernels, in the same order.
//
// Measured (us per iteration, one-pass -> folded), FP64: 1x100x100 63.5 -> 29.0,
// 3x100x100 76.6 -> 32.1, 4x187x251 99.9 -> 44.5, 5x500x500 207.7 -> 125.7,
// 10x500x500 386 -> 235, 10x1000x1000 1085 -> 1015; FP32 inner solves:
// 3x100x100 73 -> 37, 5x500x500 172 -> 92, 10x300x300 195 -> 83.  The small grids
// are bound by nine dependent launches of 2.5 to 5 us, the large ones by memory.
#include <cstring>
#include <string>

#include <hip/hip_fp16.h>

#include "mf6hip_fold.h"

#define CK(x)                         \
  do {                                \
    int rc_ = (x);                    \
    if (rc_ != MF6HIP_OK) return rc_; \
  } while (0)

namespace {

// what the kernels of an iteration leave for the later ones; two values by
// round parity.  No kernel reads a field that it writes (stop excepted, see
// the flags' comments).
struct BState {
  double rho[2], alpha[2], omega[2];
  double beta;
  int have;        // an iteration was completed (written by k_b_upd)
  int stop;        // the test's result (k_b_black); read from k_b_bwd on
  int stop_seen;   // its copy (k_b_bwd, k_b_test); read by k_b_red and k_b_black
  double ss;       // reduced for the test (k_b_red, k_b_test)
  MaxLoc mx, mr;
};

constexpr int B_SQ = 256;                // partials after a squeeze
constexpr int B_RAW = 2048;              // most partials read without one (512 with 64 threads)
enum { BP_DV = 0, BP_TQ = 1, BP_TT = 2, BP_SS = 3, BP_RHO = 4 };   // sums
enum { BM_X = 0, BM_R = 1 };                                       // maxima
// squeezed copies sit behind the raw partials
constexpr size_t B_SQP = 6 * (size_t)MF6_MAXBLK, B_SQM = 3 * (size_t)MF6_MAXBLK;

// Grids of at most B_THIN layers have kernels of their own (THIN) that load the
// layers which exist; the others load whole chunks of C_CH, clamped to the last
// layer, so that no branch stands between the loads.  us per iteration, clamped ->
// own: FP64 1x700x700 109 -> 71, 1x1000x1000 224 -> 126, 2x1000x1000 266 -> 208, FP16
// factor 1x1000x1000 152 -> 113, 2x1000x1000 174 -> 157.  With three layers or more
// the branches cost more than the loads: 3x1000x1000 FP16 185 -> 187, 7x300x300 80 ->
// 87, 32x200x200 142 -> 176.
constexpr int B_THIN = 2;

template <int BS>
constexpr int NI_B = BS == 64 ? 512 / 64 : B_RAW / BS;

// pivots as FP64, FP32 or FP16 bits
template <typename TP>
__device__ inline double bpiv(const TP *p, int e) { return (double)p[e]; }
template <>
__device__ inline double bpiv<unsigned short>(const unsigned short *p, int e) {
  const unsigned short u = p[e];
  const __half h = *reinterpret_cast<const __half *>(&u);
  return (double)__half2float(h);
}

// the partials a kernel reads: raw or squeezed
struct BPart {
  const double *s;
  const MaxLoc *m;
  size_t ld;   // slots per quantity
  int n;
};

// partials of quantities slot .. slot + ns - 1 (and, from the first block on,
// both maxima) summed into B_SQ slots each, block b taking every B_SQ-th
__global__ void __launch_bounds__(64) k_b_squeeze(double *part, MaxLoc *mpart, int n, int slot,
                                                  int ns, int maxima) {
  const int b = blockIdx.x;
  for (int q = 0; q < ns; q++) {
    const double *s = part + (size_t)(slot + q) * MF6_MAXBLK;
    double v = 0.0;
    for (int i = b + (int)threadIdx.x * B_SQ; i < n; i += 64 * B_SQ) v = v + s[i];
    v = csum(v);
    if (threadIdx.x == 0) part[B_SQP + (slot + q) * B_SQ + b] = v;
  }
  if (!maxima) return;
  for (int q = 0; q < 2; q++) {
    const MaxLoc *s = mpart + (size_t)q * MF6_MAXBLK;
    MaxLoc v{0.0, -1};
    for (int i = b + (int)threadIdx.x * B_SQ; i < n; i += 64 * B_SQ) v = maxloc_pick(v, s[i]);
    v = cmax(v);
    if (threadIdx.x == 0) mpart[B_SQM + q * B_SQ + b] = v;
  }
}

// Q false: w = p = d + beta (p - omega v); Q true: w = q = d - alpha v; then the
// forward sweep of the red columns into zf.  Q false: three more blocks reduce
// the maxima and d.d of the last iteration for the test.
template <int BS, bool Q, bool THIN, typename TM, typename TV, typename TP>
__global__ void __launch_bounds__(BS, 2) k_b_red(Layout L, const TM *__restrict__ A,
                                                 const TP *__restrict__ piv,
                                                 const TV *__restrict__ d,
                                                 const TV *__restrict__ v, TV *__restrict__ w,
                                                 TV *__restrict__ zf, BPart pt, BState *bs, int nc,
                                                 int par) {
  constexpr int CH = THIN ? B_THIN : C_CH;
  __shared__ double lds[4];
  __shared__ MaxLoc mlds[4];
  if (!Q && (int)blockIdx.x >= nc) {
    const int e = (int)blockIdx.x - nc;
    if (e < 2) {
      const MaxLoc m = call_max<BS>(cmpart<BS, NI_B<BS>>(pt.m + e * pt.ld, pt.n), mlds);
      if (threadIdx.x == 0) (e == 0 ? bs->mx : bs->mr) = m;
    } else {
      const double s = call_sum<BS>(cpart<BS, NI_B<BS>>(pt.s + BP_SS * pt.ld, pt.n), lds);
      if (threadIdx.x == 0) bs->ss = s;
    }
    return;
  }
  const int lb = cblock(blockIdx.x, nc);
  const int NP = L.NP, HP = L.HP;
  const int stop = Q ? bs->stop : bs->stop_seen, have = bs->have;
  const double rho = bs->rho[par], rho0 = bs->rho[1 - par];
  const double alpha0 = bs->alpha[1 - par], omega0 = bs->omega[1 - par];
  double s = cpart<BS, NI_B<BS>>(pt.s + (Q ? BP_DV : BP_RHO) * pt.ld, pt.n);
  const int h2 = lb * BS + threadIdx.x;
  const bool in = h2 < L.HP0;
  const int h = in ? h2 : 0;
  TV dv[CH], vv[CH], wv[CH];
  TM a1[CH];
  TV pv[CH];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < CH; u++) {
      if (THIN && u > 0 && k0 + u >= L.nlay) break;
      const int p = (k0 + u < L.nlay ? k0 + u : L.nlay - 1) * HP + h;
      dv[u] = d[p];
      vv[u] = v[p];
      if (!Q) wv[u] = w[p];
      a1[u] = A[NP + p];
      pv[u] = (TV)bpiv(piv, p);
    }
  };
  load(0);
  if (stop) return;
  s = call_sum<BS>(s, lds);
  TV c0, c1 = (TV)0;
  if (Q) {
    const double alpha = rho / (s + copysign(DPREC_C, s));
    if (blockIdx.x == 0 && threadIdx.x == 0) bs->alpha[par] = alpha;
    c0 = (TV)alpha;
  } else {
    const double beta = have ? (s / rho0) * (alpha0 / omega0) : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      bs->rho[par] = s;
      bs->beta = beta;
    }
    c0 = (TV)beta;
    c1 = (TV)omega0;
  }
  if (!in) return;
  TV zup = (TV)0, pup = (TV)0;
  for (int k0 = 0; k0 < L.nlay; k0 += C_CH) {
    if (k0) load(k0);
#pragma unroll
    for (int u = 0; u < CH; u++) {
      const int k = k0 + u;
      if (k < L.nlay) {
        const int p = k * HP + h;
        TV x;
        if (Q) x = dv[u] - c0 * vv[u];
        else x = have ? dv[u] + c0 * (wv[u] - c1 * vv[u]) : dv[u];
        w[p] = x;
        TV tv = x;
        if (k > 0) tv = tv - (TV)((TV)a1[u] * pup) * zup;
        zf[p] = tv;
        zup = tv;
        pup = pv[u];
      }
    }
  }
}

// convergence test of the last iteration (FP64: ImsLinearBase.f90:475-505;
// mixed: the inner solve's max |r| against its target, and the breakdowns)
__device__ inline void b_test(KState *st, BState *bs, int mixed, int par, double *hist, int *hloc,
                              FoldHost *hf) {
  if (bs->stop_seen || !bs->have) return;
  // the current rho is in slot par, the tested iteration's in 1 - par; the
  // iteration before it left rho0 .. in the state
  const double rho = bs->rho[1 - par], alpha = bs->alpha[1 - par], omega = bs->omega[1 - par];
  const double ss = bs->ss;
  const MaxLoc mx = bs->mx, mr = bs->mr;
  const int it = st->iter + 1;
  st->iter = it;
  st->rho = rho;
  st->alpha = alpha;
  st->omega = omega;
  st->deltax = mx.v;
  st->xloc = mx.loc;
  st->rmax = mr.v;
  st->rloc = mr.loc;
  const double rho0 = st->rho0, alpha0 = st->alpha0, omega0 = st->omega0;
  int icnvg = st->icnvg;
  if (mixed) {
    if (fabs(mr.v) <= st->rclose) icnvg = 1;
  } else {
    const double l2norm = sqrt(ss);
    st->l2norm = l2norm;
    if (it <= st->hist_cap) {
      const int cap = st->hist_cap;
      hist[it - 1] = mx.v;
      hist[cap + it - 1] = mr.v;
      hist[2 * cap + it - 1] = alpha;
      hist[3 * cap + it - 1] = omega;
      hloc[it - 1] = mx.loc;
      hloc[cap + it - 1] = mr.loc;
    }
    const int o = st->icnvgopt;
    const double rcnvg = (o == 2 || o == 3 || o == 4) ? l2norm : mr.v;
    c_testcnvg(o, &icnvg, it, mx.v, rcnvg, st->l2norm0, st->epfact, st->dvclose, st->rclose);
    if (rcnvg == 0.0) icnvg = 1;
  }
  st->icnvg = icnvg;
  int stop = 0;
  if (icnvg != 0) stop = 1;
  else if (c_close(rho, rho0) || c_close(alpha, alpha0) || c_close(omega, omega0) ||
           rho * omega == 0.0)
    stop = 2;
  else if (it >= st->itmax) stop = 3;
  if (stop != 2 && icnvg == 0) {
    st->rho0 = rho;
    st->alpha0 = alpha;
    st->omega0 = omega;
  }
  if (stop) {
    bs->stop = stop;
    c_publish(hf, st, stop);
  }
}

// NL bounds the layers at compile time (a column's values stay in registers).
// Q false: the last block runs the convergence test.
template <int BS, bool Q, int NL, typename TM, typename TV, typename TP>
__global__ void __launch_bounds__(BS, NL <= 16 ? 2 : 1) k_b_black(
    Layout L, const TM *__restrict__ A, const TP *__restrict__ piv, const TV *__restrict__ d,
    const TV *__restrict__ v, TV *__restrict__ w, const TV *__restrict__ zf, TV *__restrict__ z,
    KState *st, BState *bs, int nc, int par, int mixed, double *hist, int *hloc,
    FoldHost *hf) {
  constexpr bool THIN = NL <= B_THIN;
  constexpr int CH = THIN ? B_THIN : C_CH;
  if (!Q && (int)blockIdx.x == nc) {
    if (threadIdx.x == 0) b_test(st, bs, mixed, par, hist, hloc, hf);
    return;
  }
  const int lb = cblock(blockIdx.x, nc);
  const int NP = L.NP, HP = L.HP;
  const int stop = Q ? bs->stop : bs->stop_seen, have = bs->have;
  const TV c0 = (TV)(Q ? bs->alpha[par] : bs->beta), c1 = (TV)(Q ? 0.0 : bs->omega[1 - par]);
  const int h = lb * BS + threadIdx.x;
  if (h >= L.HP1) return;
  const CGeo G(L, 1, h);
  TV zup = (TV)0, pup = (TV)0;
  TV zc[NL], pc[NL];
  TM ac[NL];
#pragma unroll
  for (int k0 = 0; k0 < NL; k0 += C_CH) {
    if (k0 >= L.nlay) break;
    TM a1[CH], ab[CH], al[CH], ar[CH], af[CH];
    TV pb[CH], zb[CH], pl[CH], zl[CH], pr[CH], zr[CH], pf[CH], zf_[CH], dv[CH], vv[CH], wv[CH];
#pragma unroll
    for (int u = 0; u < CH; u++) {
      if (THIN && u > 0 && k0 + u >= L.nlay) break;
      const int k = k0 + u < L.nlay ? k0 + u : L.nlay - 1;
      const int pos = L.H + k * HP + h, rb = k * HP;
      dv[u] = d[pos];
      vv[u] = v[pos];
      if (!Q) wv[u] = w[pos];
      a1[u] = A[NP + pos];
      ab[u] = A[2 * NP + pos];
      al[u] = A[3 * NP + pos];
      ar[u] = A[4 * NP + pos];
      af[u] = A[5 * NP + pos];
      ac[k0 + u] = A[6 * NP + pos];
      pb[u] = (TV)bpiv(piv, rb + G.ib);
      zb[u] = zf[rb + G.ib];
      pl[u] = (TV)bpiv(piv, rb + G.il);
      zl[u] = zf[rb + G.il];
      pr[u] = (TV)bpiv(piv, rb + G.ir);
      zr[u] = zf[rb + G.ir];
      pf[u] = (TV)bpiv(piv, rb + G.ifr);
      zf_[u] = zf[rb + G.ifr];
      pc[k0 + u] = (TV)bpiv(piv, pos);
    }
    if (stop) return;
#pragma unroll
    for (int u = 0; u < CH; u++) {
      const int k = k0 + u;
      if (k < L.nlay) {
        TV x;
        if (Q) x = dv[u] - c0 * vv[u];
        else x = have ? dv[u] + c0 * (wv[u] - c1 * vv[u]) : dv[u];
        w[L.H + k * HP + h] = x;
        TV tv = x;
        tv = G.hb ? tv - (TV)((TV)ab[u] * pb[u]) * zb[u] : tv;
        tv = G.hl ? tv - (TV)((TV)al[u] * pl[u]) * zl[u] : tv;
        tv = G.hr ? tv - (TV)((TV)ar[u] * pr[u]) * zr[u] : tv;
        tv = G.hf ? tv - (TV)((TV)af[u] * pf[u]) * zf_[u] : tv;
        if (k > 0) tv = tv - (TV)((TV)a1[u] * pup) * zup;
        zc[k] = tv;
        zup = tv;
        pup = pc[k];
      }
    }
  }
  TV zdn = (TV)0;
#pragma unroll
  for (int k = NL - 1; k >= 0; k--) {
    if (k < L.nlay) {
      TV tv = zc[k];
      if (k < L.nlay - 1) tv = tv - (TV)ac[k] * zdn;
      tv = tv * pc[k];
      z[L.H + k * HP + h] = tv;
      zdn = tv;
    }
  }
}

// backward sweep of the red columns: cell below, then the black neighbours
template <int BS, bool Q, bool THIN, typename TM, typename TV, typename TP>
__global__ void __launch_bounds__(BS, 2) k_b_bwd(Layout L, const TM *__restrict__ A,
                                                 const TP *__restrict__ piv,
                                                 const TV *__restrict__ zf, TV *__restrict__ z,
                                                 BState *bs, int nc) {
  constexpr int CH = THIN ? B_THIN : C_CH;
  const int lb = cblock(blockIdx.x, nc);
  const int NP = L.NP, HP = L.HP;
  const int stop = bs->stop;
  const int h = lb * BS + threadIdx.x;
  if (!Q && blockIdx.x == 0 && threadIdx.x == 0) bs->stop_seen = stop;
  if (h >= L.HP0) return;
  const CGeo G(L, 0, h);
  TV zdn = (TV)0;
  for (int k0 = L.nlay - 1; k0 >= 0; k0 -= CH) {
    TV zv[CH], zb[CH], zl[CH], zr[CH], zq[CH], pv[CH];
    TM a6[CH], ab[CH], al[CH], ar[CH], af[CH];
#pragma unroll
    for (int u = 0; u < CH; u++) {
      if (THIN && u > k0) break;
      const int k = k0 - u > 0 ? k0 - u : 0;
      const int pos = k * HP + h, bb = L.H + k * HP;
      zv[u] = zf[pos];
      a6[u] = A[6 * NP + pos];
      ab[u] = A[2 * NP + pos];
      al[u] = A[3 * NP + pos];
      ar[u] = A[4 * NP + pos];
      af[u] = A[5 * NP + pos];
      zb[u] = z[bb + G.ib];
      zl[u] = z[bb + G.il];
      zr[u] = z[bb + G.ir];
      zq[u] = z[bb + G.ifr];
      pv[u] = (TV)bpiv(piv, pos);
    }
    if (stop) return;
#pragma unroll
    for (int u = 0; u < CH; u++) {
      const int k = k0 - u;
      if (k >= 0) {
        TV tv = zv[u];
        if (k < L.nlay - 1) tv = tv - (TV)a6[u] * zdn;
        tv = G.hb ? tv - (TV)ab[u] * zb[u] : tv;
        tv = G.hl ? tv - (TV)al[u] * zl[u] : tv;
        tv = G.hr ? tv - (TV)ar[u] * zr[u] : tv;
        tv = G.hf ? tv - (TV)af[u] * zq[u] : tv;
        tv = tv * pv[u];
        z[k * HP + h] = tv;
        zdn = tv;
      }
    }
  }
}

// y = A x (amux order); T false: partials of w.y (dhat.v); T true: of y.w and
// y.y (t.q and t.t).  One thread per column and ny-th of its layers.
template <int BS, bool T, bool THIN, typename TM, typename TV>
__global__ void __launch_bounds__(BS, 2) k_b_mv(Layout L, const TM *__restrict__ A,
                                                const TV *__restrict__ x, TV *__restrict__ y,
                                                const TV *__restrict__ w, double *part,
                                                const BState *bs, int nq, int ny) {
  constexpr int CH = THIN ? B_THIN : C_CH;
  __shared__ double lds[4], lds2[4];
  const int lb = cblock(blockIdx.x, nq);
  const int NP = L.NP, HP = L.HP;
  const int stop = bs->stop;
  const int t = (lb / ny) * BS + threadIdx.x;
  const int c = t & 1, h2 = t >> 1;
  const bool in = h2 < ncols_of(L, c);
  const int h = in ? h2 : 0;
  const int chunks = (L.nlay + C_CH - 1) / C_CH, cy = lb % ny;
  const int ka = chunks * cy / ny * C_CH, kb = chunks * (cy + 1) / ny * C_CH;
  double s1 = 0.0, s2 = 0.0;
  if (in) {
    const CGeo G(L, c, h);
    const int own = c * L.H + h, oth = (1 - c) * L.H;
    for (int k0 = ka; k0 < kb; k0 += C_CH) {
      TV xo[CH + 2], xb[CH], xl[CH], xr[CH], xf[CH], wv[CH];
      TM a0[CH], a1[CH], ab[CH], al[CH], ar[CH], af[CH], a6[CH];
#pragma unroll
      for (int u = 0; u < CH + 2; u++) {
        if (THIN && u > 1 && k0 + u > L.nlay) break;
        int k = k0 + u - 1;
        k = k < 0 ? 0 : (k < L.nlay ? k : L.nlay - 1);
        xo[u] = x[own + k * HP];
      }
#pragma unroll
      for (int u = 0; u < CH; u++) {
        if (THIN && u > 0 && k0 + u >= L.nlay) break;
        const int k = k0 + u < L.nlay ? k0 + u : L.nlay - 1;
        const int pos = own + k * HP, ob = oth + k * HP;
        a0[u] = A[pos];
        a1[u] = A[NP + pos];
        ab[u] = A[2 * NP + pos];
        al[u] = A[3 * NP + pos];
        ar[u] = A[4 * NP + pos];
        af[u] = A[5 * NP + pos];
        a6[u] = A[6 * NP + pos];
        xb[u] = x[ob + G.ib];
        xl[u] = x[ob + G.il];
        xr[u] = x[ob + G.ir];
        xf[u] = x[ob + G.ifr];
        wv[u] = w[pos];
      }
      if (stop) return;
#pragma unroll
      for (int u = 0; u < CH; u++) {
        const int k = k0 + u;
        if (k < L.nlay) {
          TV q = (TV)0;
          q = q + (TV)a0[u] * xo[u + 1];
          if (k > 0) q = q + (TV)a1[u] * xo[u];
          if (G.hb) q = q + (TV)ab[u] * xb[u];
          if (G.hl) q = q + (TV)al[u] * xl[u];
          if (G.hr) q = q + (TV)ar[u] * xr[u];
          if (G.hf) q = q + (TV)af[u] * xf[u];
          if (k < L.nlay - 1) q = q + (TV)a6[u] * xo[u + 2];
          y[own + k * HP] = q;
          s1 = s1 + (double)wv[u] * (double)q;
          if (T) s2 = s2 + (double)q * (double)q;
        }
      }
    }
  }
  if (stop) return;
  s1 = call_sum<BS>(s1, lds);
  if (T) s2 = call_sum<BS>(s2, lds2);
  if (threadIdx.x == 0) {
    part[(size_t)(T ? BP_TQ : BP_DV) * MF6_MAXBLK + lb] = s1;
    if (T) part[(size_t)BP_TT * MF6_MAXBLK + lb] = s2;
  }
}

// INIT: dhat = d and the partials of dhat.d; else the end of an iteration (see
// the file's head)
template <int BS, bool INIT, bool THIN, typename TV, typename TX>
__global__ void __launch_bounds__(BS) k_b_upd(Layout L, TX *__restrict__ x,
                                              const TV *__restrict__ phat,
                                              const TV *__restrict__ qhat, TV *__restrict__ d,
                                              const TV *__restrict__ q, const TV *__restrict__ t_,
                                              TV *__restrict__ dhat, BPart pt, double *part,
                                              MaxLoc *mpart, BState *bs, int nq, int ny, int par) {
  constexpr int CH = THIN ? B_THIN : C_CH;
  __shared__ double lds[4][4];
  __shared__ MaxLoc mlds[2][4];
  const int lb = cblock(blockIdx.x, nq);
  const int HP = L.HP;
  const int stop = INIT ? 0 : bs->stop;
  const double alpha = INIT ? 0.0 : bs->alpha[par];
  double tq = 0.0, tt = 0.0;
  if (!INIT) {
    tq = cpart<BS, NI_B<BS>>(pt.s + BP_TQ * pt.ld, pt.n);
    tt = cpart<BS, NI_B<BS>>(pt.s + BP_TT * pt.ld, pt.n);
  }
  const int t = (lb / ny) * BS + threadIdx.x;
  const int c = t >= HP, h2 = t - c * HP;
  const bool in = c < 2 && h2 < ncols_of(L, c);
  const int own = c * L.H + (in ? h2 : 0);
  const int chunks = (L.nlay + C_CH - 1) / C_CH, cy = lb % ny;
  const int ka = chunks * cy / ny * C_CH, kb = chunks * (cy + 1) / ny * C_CH;
  TV ph[CH], qh[CH], qv[CH], tv_[CH], dh[CH];
  TX xv[CH];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < CH; u++) {
      if (THIN && u > 0 && k0 + u >= L.nlay) break;
      const int pos = own + (k0 + u < L.nlay ? k0 + u : L.nlay - 1) * HP;
      if (INIT) {
        dh[u] = d[pos];
      } else {
        ph[u] = phat[pos];
        qh[u] = qhat[pos];
        qv[u] = q[pos];
        tv_[u] = t_[pos];
        dh[u] = dhat[pos];
        xv[u] = x[pos];
      }
    }
  };
  load(ka < L.nlay ? ka : 0);
  if (stop) return;
  TV ca = (TV)0, co = (TV)0;
  if (!INIT) {
    tq = call_sum<BS>(tq, lds[0]);
    tt = call_sum<BS>(tt, lds[1]);
    const double omega = tq / (tt + copysign(DPREC_C, tt));
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      bs->omega[par] = omega;
      bs->have = 1;
    }
    ca = (TV)alpha;
    co = (TV)omega;
  }
  double ss = 0.0, rho = 0.0;
  MaxLoc mx{0.0, -1}, mr{0.0, -1};
  if (in) {
    const int l = col_l(L, c, h2);
    for (int k0 = ka; k0 < kb; k0 += C_CH) {
      if (k0 != ka) load(k0);
#pragma unroll
      for (int u = 0; u < CH; u++) {
        const int k = k0 + u;
        if (k < L.nlay) {
          const int pos = own + k * HP;
          if (INIT) {
            dhat[pos] = dh[u];
            rho = rho + (double)dh[u] * (double)dh[u];
          } else {
            const TV tv = ca * ph[u] + co * qh[u];
            x[pos] = (TX)(xv[u] + (TX)tv);
            mx = maxloc_pick(mx, MaxLoc{(double)tv, k * L.NRC + l});
            const TV r = qv[u] - co * tv_[u];
            d[pos] = r;
            mr = maxloc_pick(mr, MaxLoc{(double)r, k * L.NRC + l});
            ss = ss + (double)r * (double)r;
            rho = rho + (double)dh[u] * (double)r;
          }
        }
      }
    }
  }
  rho = call_sum<BS>(rho, lds[2]);
  if (!INIT) {
    ss = call_sum<BS>(ss, lds[3]);
    mx = call_max<BS>(mx, mlds[0]);
    mr = call_max<BS>(mr, mlds[1]);
  }
  if (threadIdx.x == 0) {
    part[(size_t)BP_RHO * MF6_MAXBLK + lb] = rho;
    if (!INIT) {
      part[(size_t)BP_SS * MF6_MAXBLK + lb] = ss;
      mpart[(size_t)BM_X * MF6_MAXBLK + lb] = mx;
      mpart[(size_t)BM_R * MF6_MAXBLK + lb] = mr;
    }
  }
}

// the convergence test of iteration r = 2 m + par, at its end (one block)
__global__ void __launch_bounds__(64) k_b_test(BPart pt, KState *st, BState *bs, int mixed, int par,
                                               double *hist, int *hloc, FoldHost *hf) {
  const MaxLoc mx = cmax(cmpart<64, B_SQ / 64>(pt.m + BM_X * pt.ld, B_SQ));
  const MaxLoc mr = cmax(cmpart<64, B_SQ / 64>(pt.m + BM_R * pt.ld, B_SQ));
  const double ss = csum(cpart<64, B_SQ / 64>(pt.s + BP_SS * pt.ld, B_SQ));
  if (threadIdx.x != 0) return;
  bs->mx = mx;
  bs->mr = mr;
  bs->ss = ss;
  b_test(st, bs, mixed, 1 - par, hist, hloc, hf);
  bs->stop_seen = bs->stop;
}

// Positions above which k_b_test runs: its launch takes about 4 us an iteration, the
// red and black sweeps that otherwise run for nothing at the end of a solve 160 us at
// 10x1000x1000 (a solve of one iteration 1933 -> 1773 us, of twenty 21.1 -> 21.0 ms) and in
// proportion to the cells, so that at four million a solve of some twenty iterations
// breaks even.
constexpr int B_TEST_NP = 1 << 22;

struct BGrid {
  int bs, nc, ny, nq;   // threads; blocks of one colour; chunks a column; blocks of all
  bool squeeze, test;   // test: k_b_test
};

// 64 threads a block where 512 blocks hold every chunk, else 256; a chunk of
// layers per thread while that leaves at most 2048 blocks, else a column
BGrid b_grid(const Layout &L) {
  BGrid g{};
  g.ny = (L.nlay + C_CH - 1) / C_CH;
  g.bs = (2 * L.HP0 + 63) / 64 * g.ny <= 512 ? 64 : 256;
  if ((2 * L.HP0 + g.bs - 1) / g.bs * g.ny > 2048) g.ny = 1;
  g.nc = (L.HP0 + g.bs - 1) / g.bs;
  g.nq = (2 * L.HP0 + g.bs - 1) / g.bs * g.ny;
  g.squeeze = g.nq > B_RAW;
  g.test = g.squeeze && L.NP > B_TEST_NP;
  return g;
}

// the vectors of one solve
template <typename TM, typename TV, typename TP, typename TX>
struct BVec {
  const TM *A;
  const TP *piv;
  TX *x;
  TV *d, *p, *v, *q, *phat, *qhat, *t, *dhat, *zf;
  KState *st;
  int mixed;
};

template <int BS, int NL, typename B>
void enqueue_b(Mf6Handle *h, const BGrid &g, const B &b, int n) {
  constexpr bool THIN = NL <= B_THIN;
  const Layout &L = h->L;
  hipStream_t s = h->stream;
  BState *bs = reinterpret_cast<BState *>(h->d_state + 2);
  double *part = h->d_part;
  MaxLoc *mpart = h->d_mpart;
  const BPart pt = g.squeeze ? BPart{part + B_SQP, mpart + B_SQM, (size_t)B_SQ, B_SQ}
                             : BPart{part, mpart, (size_t)MF6_MAXBLK, g.nq};
  auto squeeze = [&](int slot, int ns, int maxima) {
    if (g.squeeze) k_b_squeeze<<<B_SQ, 64, 0, s>>>(part, mpart, g.nq, slot, ns, maxima);
  };
  for (int r = 0; r < n; r++) {
    const int par = r & 1;
    k_b_red<BS, false, THIN><<<g.nc + (g.test ? 0 : 3), BS, 0, s>>>(L, b.A, b.piv, b.d, b.v, b.p,
                                                                    b.zf, pt, bs, g.nc, par);
    k_b_black<BS, false, NL><<<g.nc + (g.test ? 0 : 1), BS, 0, s>>>(
        L, b.A, b.piv, b.d, b.v, b.p, b.zf, b.phat, b.st, bs, g.nc, par, b.mixed, h->d_hist,
        h->d_hloc, h->h_fold);
    k_b_bwd<BS, false, THIN><<<g.nc, BS, 0, s>>>(L, b.A, b.piv, b.zf, b.phat, bs, g.nc);
    hipEvent_t e1 = nullptr;
    if (h->timing && (h->spmv_calls++ % h->spmv_sample) == 0 &&
        2 * (h->last_spmv_n + 1) <= (int)h->spmv_ev.size()) {
      const int slot = h->last_spmv_n++;
      (void)hipEventRecord(h->spmv_ev[2 * slot], s);
      e1 = h->spmv_ev[2 * slot + 1];
    }
    k_b_mv<BS, false, THIN><<<g.nq, BS, 0, s>>>(L, b.A, b.phat, b.v, b.dhat, part, bs, g.nq, g.ny);
    if (e1) (void)hipEventRecord(e1, s);
    squeeze(BP_DV, 1, 0);
    k_b_red<BS, true, THIN><<<g.nc, BS, 0, s>>>(L, b.A, b.piv, b.d, b.v, b.q, b.zf, pt, bs, g.nc,
                                                par);
    k_b_black<BS, true, NL><<<g.nc, BS, 0, s>>>(L, b.A, b.piv, b.d, b.v, b.q, b.zf, b.qhat, b.st,
                                                bs, g.nc, par, b.mixed, h->d_hist, h->d_hloc,
                                                h->h_fold);
    k_b_bwd<BS, true, THIN><<<g.nc, BS, 0, s>>>(L, b.A, b.piv, b.zf, b.qhat, bs, g.nc);
    k_b_mv<BS, true, THIN><<<g.nq, BS, 0, s>>>(L, b.A, b.qhat, b.t, b.q, part, bs, g.nq, g.ny);
    squeeze(BP_TQ, 2, 0);
    k_b_upd<BS, false, THIN><<<g.nq, BS, 0, s>>>(L, b.x, b.phat, b.qhat, b.d, b.q, b.t, b.dhat, pt,
                                                 part, mpart, bs, g.nq, g.ny, par);
    squeeze(BP_SS, 2, 1);
    if (g.test)
      k_b_test<<<1, 64, 0, s>>>(pt, b.st, bs, b.mixed, par, h->d_hist, h->d_hloc, h->h_fold);
  }
}

// iterations of one graph (even: the parities alternate); with 4 the short solves of a
// Newton step run more for nothing (mixed 4x187x251 3.08 -> 3.31 ms a step, 5x500x500 5.34
// -> 5.75; FP64 up to 2 % more)
constexpr int B_ITERS = 2;

template <typename B>
void enqueue_b(Mf6Handle *h, const BGrid &g, const B &b, int n) {
  const int nl = h->L.nlay;
#define MF6_B(N) (g.bs == 64 ? enqueue_b<64, N>(h, g, b, n) : enqueue_b<256, N>(h, g, b, n))
  if (nl <= B_THIN) MF6_B(B_THIN);
  else if (nl <= 4) MF6_B(4);
  else if (nl <= 8) MF6_B(8);
  else if (nl <= 16) MF6_B(16);
  else MF6_B(32);
#undef MF6_B
}

template <typename B>
bool b_graph(Mf6Handle *h, const BGrid &g, const B &b) {
  if (h->cg_graph) return true;
  if (h->cg_graph_failed) return false;
  hipStream_t s = h->stream;
  hipGraph_t gr = nullptr;
  bool ok = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) == hipSuccess;
  if (ok) {
    enqueue_b(h, g, b, B_ITERS);
    ok = hipStreamEndCapture(s, &gr) == hipSuccess && gr != nullptr;
  }
  if (ok) ok = hipGraphInstantiate(&h->cg_graph, gr, nullptr, nullptr, 0) == hipSuccess;
  if (gr) (void)hipGraphDestroy(gr);
  if (!ok) {
    h->cg_graph = nullptr;
    h->cg_graph_failed = true;
    (void)hipGetLastError();
  }
  return ok;
}

// BiCGSTAB from the residual in b.d (b.st initialised, its slot si of the
// device states); on return h_state[si] holds the final state.
template <typename B>
int run_b(Mf6Handle *h, const B &b, int si) {
  const Layout &L = h->L;
  hipStream_t s = h->stream;
  const BGrid g = b_grid(L);
  BState *bs = reinterpret_cast<BState *>(h->d_state + 2);
  static_assert(sizeof(BState) <= sizeof(KState), "BState fits its slot");
  HIPCHK(hipMemsetAsync(bs, 0, sizeof(BState), s));
  const BPart none{};
  if (g.bs == 64)
    k_b_upd<64, true, false><<<g.nq, 64, 0, s>>>(L, b.x, b.phat, b.qhat, b.d, b.q, b.t, b.dhat, none,
                                          h->d_part, h->d_mpart, bs, g.nq, g.ny, 0);
  else
    k_b_upd<256, true, false><<<g.nq, 256, 0, s>>>(L, b.x, b.phat, b.qhat, b.d, b.q, b.t, b.dhat, none,
                                            h->d_part, h->d_mpart, bs, g.nq, g.ny, 0);
  if (g.squeeze) k_b_squeeze<<<B_SQ, 64, 0, s>>>(h->d_part, h->d_mpart, g.nq, BP_RHO, 1, 0);
  h->h_fold->stop = 0;
  const bool graph = !h->timing && b_graph(h, g, b);
  CK(fold_batches(h, B_ITERS, [&]() -> int {
    if (graph) HIPCHK(hipGraphLaunch(h->cg_graph, s));
    else enqueue_b(h, g, b, B_ITERS);
    HIPCHK(hipGetLastError());
    return MF6HIP_OK;
  }));
  h->h_state[si] = h->h_fold->st;
  return MF6HIP_OK;
}

}  // namespace

// Whether the folded BiCGSTAB takes a handle's solves: no reorthogonalisation
// and no scaling (their extra passes stay with the one-pass kernels), and
// partials that fit their arrays.
bool mf6hip_bcgs_fold_takes(const Mf6Handle *h) {
  return h->s.kernel_variant == 0 && h->s.north == 0 && h->s.iscl == 0 &&
         b_grid(h->L).nq <= MF6_MAXBLK;
}

int mf6hip_run_bcgs_fold(Mf6Handle *h) {
  // INNER_MAXIMUM 0: the state stays as initialised.  (An iteration is tested by the
  // kernels of the next one, so the first would run.)
  if (h->s.iter1 == 0) return MF6HIP_OK;
  const BVec<double, double, double, double> b{h->A, h->invpiv, h->x, h->d, h->p, h->v, h->q,
                                               h->phat, h->qhat, h->t, h->dhat, h->zf,
                                               h->d_state, 0};
  return run_b(h, b, 0);
}

// the FP32 inner solve of the mixed BiCGSTAB on h->r32 (state 1, initialised)
int mf6hip_run_bcgs_fold_inner(Mf6Handle *h) {
  if (h->s.precision == MF6HIP_MIXED) {
    const BVec<float, float, float, float> b{h->A32, h->invpiv32, h->e32, h->r32, h->p32, h->p232,
                                             h->q32, h->z32, h->qhat32, h->t32, h->dhat32,
                                             h->zf32, h->d_state + 1, 1};
    return run_b(h, b, 1);
  }
  const BVec<float, float, unsigned short, float> b{
      h->A32, h->invpiv16, h->e32, h->r32, h->p32, h->p232, h->q32, h->z32, h->qhat32, h->t32,
      h->dhat32, h->zf32, h->d_state + 1, 1};
  return run_b(h, b, 1);
}
