// mf6hip_fcg.hip -- flexible preconditioned CG with the learned correction.
//
// Preconditioner (variable, hence flexible CG), a two-level cycle with the
// network as the coarse correction:
//   z  = ILU0(r)                      pre-smoothing: the device ILU0
//   t  = r - A z                      what the ILU0 step leaves
//   y  = s * net([t / s, features])   s = rms(t): the network sees unit-scale
//                                     residuals; its output is rescaled
//   z += w y,  w = y.t / y.A y        energy-optimal step along y
//   z += ILU0(r - A z)                post-smoothing: damps the rough part of
//                                     the correction (BF16 noise of y)
// FCG(m) (Notay 2000): p = z - sum_j (z.q_j / p_j.q_j) p_j over the last m
// directions, alpha = p.r / p.q, x += alpha p, r -= alpha q.  The IMS
// convergence test (ImsLinearBase.f90:1101-1146) is applied to every
// iteration with the signed largest head change alpha p and residual; when
// it passes, the FP64 true residual b - A x is recomputed and must pass it
// too (else the iteration continues from the true residual).  The network
// runs on every nn_every-th iteration (ILU0 alone on the others).
// Fallback: the ILU0-only step replaces the learned one for the rest of the
// solve when z.r changes sign against the ILU0 step (not a descent
// direction) or when ten applications of the network (10 nn_every
// iterations) reduce ||r||_2 by less than 10 %.
//
// Every scalar of the iteration lives in a device FcgState: the host
// enqueues the kernels of a group of iterations without waiting, one group
// ahead of the one it waits for; once the solve has stopped (converged) the
// state-changing kernels of the rest of the queue return at once.
//
// On the grids that a network takes (tens of thousands to a few million
// cells) an iteration is bound by the latency of its launches, so the kernels
// carry their neighbours' work: the SpMV forms the residual or the network's
// step, the sweeps form their operand, every block of a consumer adds the
// partials of a dot product in the same order.  At 6x96x112 an iteration without
// the network takes 42 us in nine launches (68 in thirteen when every vector pass,
// sum and ILU0 sweep was a kernel of its own), with it nineteen launches and the
// network's (thirty-two before).  A chunk of layers loads those that exist only: with
// the loads clamped to the last layer instead (no branch between them) a single
// layer's cost as much as four's, 132 against 82 us an iteration at 1x1000x1000 with
// one direction, 437 against 231 at 1x2000x2000, and 296 against 282 at 10x700x700.
#include <cmath>
#include <vector>

#include "mf6hip_fold.h"

namespace {

constexpr int FCG_MAXM = 64;   // directions kept, at most
constexpr int FCG_NDOT = 8;    // dot products per pass
constexpr int FCG_GROUP = 4;   // iterations between looks at the state

struct FcgState {
  double tt, zr_ilu, yt, yay, yr, w;   // learned step
  double zr_l;                         // z.r of the smoothed learned step
  double pr;                           // p.r
  double rnorm, dvmax, rmax;
  double rn_window;
  double c[FCG_MAXM];                  // z.q_j, by ring slot
  double pqs[FCG_MAXM];                // p_j.q_j, by ring slot
  int learned;                         // network steps still allowed
  int acc;                             // the last learned step was accepted
  int cand;                            // the IMS test passed: check b - A x
  int stop;                            // converged: k_g_red's answer, which k_g_bwd copies to
                                       // KState::stop (no kernel reads the flag that it writes)
  int icnvg, iter, learned_iters, window;
};

struct FcgSlots {
  int n;
  int slot[FCG_MAXM];
};

struct FcgTest {
  double dvclose, rclose;
  int icnvgopt, nn_every;
};

constexpr int G_MAXB = 2048;   // blocks of a kernel whose partials are added by its consumers
constexpr int G_NI = 8;        // partials a thread adds (512 blocks of 64 threads, else 2048)
constexpr int G_RB = 256;      // blocks of the true residual
// partial sums, G_MAXB slots each: the dots with the stored directions, then
enum { G_D0 = FCG_NDOT, G_D1, G_ZR, G_SS, G_NSLOT };
// maxima: the changes, the residual; the true residual's (values only)
enum { GM_X = 0, GM_R = 1, GM_T = 2 };

__global__ void k_fcg_init(FcgState *fs, KState *ks, int learned) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  fs->learned = learned;
  fs->acc = 0;
  fs->cand = 0;
  fs->stop = 0;
  fs->icnvg = 0;
  fs->iter = 0;
  fs->learned_iters = 0;
  fs->window = 0;
  fs->rn_window = -1.0;
  for (int j = 0; j < FCG_MAXM; j++) { fs->c[j] = 0.0; fs->pqs[j] = 0.0; }
  ks->stop = 0;
}

// the true residual decides a candidate: max |b - A x| <= rclose (or a test that
// ignores the residual); the same answer in every thread and block of BS threads
template <int BS>
__device__ inline bool g_final(const MaxLoc *mpart, int nr, const FcgTest &tst, MaxLoc *mlds) {
  const MaxLoc m = call_max<BS>(cmpart<BS, G_RB / BS>(mpart + GM_T * G_MAXB, nr), mlds);
  return fabs(m.v) <= tst.rclose || tst.icnvgopt == 3;
}

__device__ inline void g_stop(FcgState *fs, const KState *ks, FoldHost *hf) {
  fs->icnvg = 1;
  fs->stop = 1;
  c_publish(hf, ks, 1);
}

// no network steps for the rest of the solve; the host, which reads the flag
// without waiting, stops enqueuing them
__device__ inline void g_off(FcgState *fs, FoldHost *hf) {
  fs->learned = 0;
  __hip_atomic_store(&hf->off, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// the last iteration's candidate, after the last one allowed
__global__ void __launch_bounds__(64) k_g_last(const MaxLoc *mpart, int nr, FcgTest tst,
                                               FcgState *fs, const KState *ks, FoldHost *hf) {
  if (ks->stop || !fs->cand) return;
  if (g_final<64>(mpart, nr, tst, nullptr) && threadIdx.x == 0) g_stop(fs, ks, hf);
}

// forward sweep of the red columns.  LEARNED false: of r, after the decision on
// the last iteration's candidate; true: of t - w A y, w = y.t / y.A y the weight
// of the learned step, or 0 when the network is off or the step degenerate
template <int BS, bool LEARNED>
__global__ void __launch_bounds__(BS, 2) k_g_red(Layout L, const double *__restrict__ A,
                                                 const double *__restrict__ piv,
                                                 const double *__restrict__ x,
                                                 const double *__restrict__ ay,
                                                 double *__restrict__ zf, const double *part,
                                                 const MaxLoc *mpart, int nq, int nr, FcgTest tst,
                                                 FcgState *fs, const KState *ks, FoldHost *hf) {
  __shared__ double lds[2][4];
  __shared__ MaxLoc mlds[4];
  const int NP = L.NP, HP = L.HP;
  const int stop = ks->stop, cand = fs->cand;
  const int h2 = cblock(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  const bool in = h2 < L.HP0;
  const int h = in ? h2 : 0;
  double xv[C_CH], yv[C_CH], a1[C_CH], pv[C_CH];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < C_CH; u++) {
      if (u > 0 && k0 + u >= L.nlay) break;
      const int p = (k0 + u) * HP + h;
      xv[u] = x[p];
      if (LEARNED) yv[u] = ay[p];
      a1[u] = A[NP + p];
      pv[u] = piv[p];
    }
  };
  load(0);
  if (stop) return;
  double w = 0.0;
  if (LEARNED) {
    const int on = fs->learned;
    const double tt = fs->tt;
    const double yt = call_sum<BS>(cpart<BS, G_NI>(part + G_D0 * G_MAXB, nq), lds[0]);
    const double yay = call_sum<BS>(cpart<BS, G_NI>(part + G_D1 * G_MAXB, nq), lds[1]);
    if (on && tt > 0.0 && yay != 0.0 && isfinite(yt) && isfinite(yay)) w = yt / yay;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      fs->yt = yt;
      fs->yay = yay;
      fs->w = w;
    }
  } else if (cand) {
    if (g_final<BS>(mpart, nr, tst, mlds)) {
      if (blockIdx.x == 0 && threadIdx.x == 0) g_stop(fs, ks, hf);
      return;
    }
  }
  if (!in) return;
  double zup = 0.0, pup = 0.0;
  for (int k0 = 0; k0 < L.nlay; k0 += C_CH) {
    if (k0) load(k0);
#pragma unroll
    for (int u = 0; u < C_CH; u++) {
      const int k = k0 + u;
      if (k < L.nlay) {
        double tv = xv[u];
        if (LEARNED) tv = w == 0.0 ? tv : tv - w * yv[u];
        if (k > 0) tv = tv - (a1[u] * pup) * zup;
        zf[k * HP + h] = tv;
        zup = tv;
        pup = pv[u];
      }
    }
  }
}

// forward and backward sweep of the black columns; NL bounds the layers at
// compile time, so that a column's values stay in registers.  fs->stop: set by
// k_g_red just before, or since an earlier iteration
template <int BS, bool LEARNED, int NL>
__global__ void __launch_bounds__(BS, NL <= 16 ? 2 : 1) k_g_black(
    Layout L, const double *__restrict__ A, const double *__restrict__ piv,
    const double *__restrict__ x, const double *__restrict__ ay, const double *__restrict__ zf,
    double *__restrict__ z, const FcgState *fs) {
  const int NP = L.NP, HP = L.HP;
  const int stop = fs->stop;
  const double w = LEARNED ? fs->w : 0.0;
  const int h = cblock(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (h >= L.HP1) return;
  const CGeo G(L, 1, h);
  double zup = 0.0, pup = 0.0;
  double zc[NL], pc[NL], ac[NL];
#pragma unroll
  for (int k0 = 0; k0 < NL; k0 += C_CH) {
    if (k0 >= L.nlay) break;
    double a1[C_CH], ab[C_CH], al[C_CH], ar[C_CH], af[C_CH], xv[C_CH], yv[C_CH];
    double pb[C_CH], zb[C_CH], pl[C_CH], zl[C_CH], pr[C_CH], zr[C_CH], pf[C_CH], zq[C_CH];
#pragma unroll
    for (int u = 0; u < C_CH; u++) {
      if (u > 0 && k0 + u >= L.nlay) break;
      const int k = k0 + u;
      const int pos = L.H + k * HP + h, rb = k * HP;
      xv[u] = x[pos];
      if (LEARNED) yv[u] = ay[pos];
      a1[u] = A[NP + pos];
      ab[u] = A[2 * NP + pos];
      al[u] = A[3 * NP + pos];
      ar[u] = A[4 * NP + pos];
      af[u] = A[5 * NP + pos];
      ac[k0 + u] = A[6 * NP + pos];
      pb[u] = piv[rb + G.ib];
      zb[u] = zf[rb + G.ib];
      pl[u] = piv[rb + G.il];
      zl[u] = zf[rb + G.il];
      pr[u] = piv[rb + G.ir];
      zr[u] = zf[rb + G.ir];
      pf[u] = piv[rb + G.ifr];
      zq[u] = zf[rb + G.ifr];
      pc[k0 + u] = piv[pos];
    }
    if (stop) return;
#pragma unroll
    for (int u = 0; u < C_CH; u++) {
      const int k = k0 + u;
      if (k < L.nlay) {
        double tv = xv[u];
        if (LEARNED) tv = w == 0.0 ? tv : tv - w * yv[u];
        tv = G.hb ? tv - (ab[u] * pb[u]) * zb[u] : tv;
        tv = G.hl ? tv - (al[u] * pl[u]) * zl[u] : tv;
        tv = G.hr ? tv - (ar[u] * pr[u]) * zr[u] : tv;
        tv = G.hf ? tv - (af[u] * pf[u]) * zq[u] : tv;
        if (k > 0) tv = tv - (a1[u] * pup) * zup;
        zc[k] = tv;
        zup = tv;
        pup = pc[k];
      }
    }
  }
  double zdn = 0.0;
#pragma unroll
  for (int k = NL - 1; k >= 0; k--) {
    if (k < L.nlay) {
      double tv = zc[k];
      if (k < L.nlay - 1) tv = tv - ac[k] * zdn;
      tv = tv * pc[k];
      z[L.H + k * HP + h] = tv;
      zdn = tv;
    }
  }
}

// backward sweep of the red columns: cell below, then the black neighbours
template <int BS>
__global__ void __launch_bounds__(BS, 2) k_g_bwd(Layout L, const double *__restrict__ A,
                                                 const double *__restrict__ piv,
                                                 const double *__restrict__ zf,
                                                 double *__restrict__ z, const FcgState *fs,
                                                 KState *ks) {
  const int NP = L.NP, HP = L.HP;
  const int stop = fs->stop;
  if (stop && blockIdx.x == 0 && threadIdx.x == 0) ks->stop = 1;
  const int h = cblock(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (h >= L.HP0) return;
  const CGeo G(L, 0, h);
  double zdn = 0.0;
  for (int k0 = L.nlay - 1; k0 >= 0; k0 -= C_CH) {
    double zv[C_CH], zb[C_CH], zl[C_CH], zr[C_CH], zq[C_CH], pv[C_CH];
    double a6[C_CH], ab[C_CH], al[C_CH], ar[C_CH], af[C_CH];
#pragma unroll
    for (int u = 0; u < C_CH; u++) {
      if (u > k0) break;
      const int k = k0 - u;
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
      pv[u] = piv[pos];
    }
    if (stop) return;
#pragma unroll
    for (int u = 0; u < C_CH; u++) {
      const int k = k0 - u;
      if (k >= 0) {
        double tv = zv[u];
        if (k < L.nlay - 1) tv = tv - a6[u] * zdn;
        tv = G.hb ? tv - ab[u] * zb[u] : tv;
        tv = G.hl ? tv - al[u] * zl[u] : tv;
        tv = G.hr ? tv - ar[u] * zr[u] : tv;
        tv = G.hf ? tv - af[u] * zq[u] : tv;
        tv = tv * pv[u];
        z[k * HP + h] = tv;
        zdn = tv;
      }
    }
  }
}

// A v (amux order), one thread per column and ny-th of its layers
enum { G_RES = 0,   // out = aux - A x; partials of out.out and x.aux
       G_NET = 1,   // x = s net (natural order), stored; out = A x; of x.aux and x.out
       G_DIR = 2 }; // out = A x; of x.out and x.aux
template <int BS, int MODE>
__global__ void __launch_bounds__(BS, 2) k_g_mv(Layout L, const double *__restrict__ A,
                                                const double *__restrict__ x,
                                                const float *__restrict__ net,
                                                double *__restrict__ xs,
                                                const double *__restrict__ aux,
                                                double *__restrict__ out, double *part,
                                                const FcgState *fs, const KState *ks, int nq,
                                                int ny) {
  __shared__ double lds[2][4];
  const int NP = L.NP, HP = L.HP, NRC = L.NRC;
  const int stop = ks->stop;
  double sc = 0.0;
  if (MODE == G_NET) {
    const double tt = fs->tt;
    sc = tt > 0.0 ? sqrt(tt / (double)L.N) : 0.0;
  }
  double s0 = 0.0, s1 = 0.0;
  const int chunks = (L.nlay + C_CH - 1) / C_CH;
  for (int lb = cblock(blockIdx.x, gridDim.x); lb < nq; lb += gridDim.x) {
    const int t = (lb / ny) * BS + threadIdx.x;
    const int c = t & 1, h = t >> 1;
    if (h >= ncols_of(L, c)) continue;
    const int cy = lb % ny;
    const int ka = chunks * cy / ny * C_CH, kb = chunks * (cy + 1) / ny * C_CH;
    const CGeo G(L, c, h);
    const int own = c * L.H + h, oth = (1 - c) * L.H;
    const int nb = G.hb ? G.l - L.ncol : G.l, nl = G.hl ? G.l - 1 : G.l;
    const int nr = G.hr ? G.l + 1 : G.l, nf = G.hf ? G.l + L.ncol : G.l;
    for (int k0 = ka; k0 < kb; k0 += C_CH) {
      double xo[C_CH + 2], xb[C_CH], xl[C_CH], xr[C_CH], xf[C_CH], av[C_CH];
      double a0[C_CH], a1[C_CH], ab[C_CH], al[C_CH], ar[C_CH], af[C_CH], a6[C_CH];
#pragma unroll
      for (int u = 0; u < C_CH + 2; u++) {
        if (u > 1 && k0 + u > L.nlay) break;
        const int k = k0 + u > 0 ? k0 + u - 1 : 0;
        xo[u] = MODE == G_NET ? sc * (double)net[k * NRC + G.l] : x[own + k * HP];
      }
#pragma unroll
      for (int u = 0; u < C_CH; u++) {
        if (u > 0 && k0 + u >= L.nlay) break;
        const int k = k0 + u;
        const int pos = own + k * HP, ob = oth + k * HP;
        a0[u] = A[pos];
        a1[u] = A[NP + pos];
        ab[u] = A[2 * NP + pos];
        al[u] = A[3 * NP + pos];
        ar[u] = A[4 * NP + pos];
        af[u] = A[5 * NP + pos];
        a6[u] = A[6 * NP + pos];
        if (MODE == G_NET) {
          xb[u] = sc * (double)net[k * NRC + nb];
          xl[u] = sc * (double)net[k * NRC + nl];
          xr[u] = sc * (double)net[k * NRC + nr];
          xf[u] = sc * (double)net[k * NRC + nf];
        } else {
          xb[u] = x[ob + G.ib];
          xl[u] = x[ob + G.il];
          xr[u] = x[ob + G.ir];
          xf[u] = x[ob + G.ifr];
        }
        av[u] = aux[pos];
      }
      if (stop) return;
#pragma unroll
      for (int u = 0; u < C_CH; u++) {
        const int k = k0 + u;
        if (k < L.nlay) {
          const int pos = own + k * HP;
          const double xv = xo[u + 1];
          double q = 0.0;
          q = q + a0[u] * xv;
          if (k > 0) q = q + a1[u] * xo[u];
          if (G.hb) q = q + ab[u] * xb[u];
          if (G.hl) q = q + al[u] * xl[u];
          if (G.hr) q = q + ar[u] * xr[u];
          if (G.hf) q = q + af[u] * xf[u];
          if (k < L.nlay - 1) q = q + a6[u] * xo[u + 2];
          if (MODE == G_RES) q = av[u] - q;
          out[pos] = q;
          if (MODE == G_NET) xs[pos] = xv;
          s0 = s0 + (MODE == G_RES ? q * q : (MODE == G_NET ? xv * av[u] : xv * q));
          s1 = s1 + (MODE == G_NET ? xv * q : xv * av[u]);
        }
      }
    }
  }
  if (stop) return;
  s0 = call_sum<BS>(s0, lds[0]);
  s1 = call_sum<BS>(s1, lds[1]);
  if (threadIdx.x == 0) {
    part[G_D0 * G_MAXB + blockIdx.x] = s0;
    part[G_D1 * G_MAXB + blockIdx.x] = s1;
  }
}

__device__ inline unsigned bf16_bits(float v) {
  const unsigned u = __float_as_uint(v);
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// network input (BF16, 16 channels, natural order): ch0 = t / s with
// s = rms(t) = sqrt(tt / N), ch1..2 = features, ch3..15 = 0; a cell's 32 bytes
// per thread
__global__ void __launch_bounds__(MF6_BLOCK) k_fcg_nn_input(Layout L, const double *__restrict__ t,
                                                            const double *part, int nq,
                                                            FcgState *fs, const KState *ks,
                                                            const float *__restrict__ feat,
                                                            uint4 *__restrict__ in0) {
  __shared__ double lds[2][4];
  const int stop = ks->stop;
  const double tt = call_sum<MF6_BLOCK>(cpart<MF6_BLOCK, G_NI>(part + G_D0 * G_MAXB, nq), lds[0]);
  const double zr = call_sum<MF6_BLOCK>(cpart<MF6_BLOCK, G_NI>(part + G_D1 * G_MAXB, nq), lds[1]);
  if (stop) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    fs->tt = tt;
    fs->zr_ilu = zr;
  }
  const double inv_s = tt > 0.0 ? sqrt((double)L.N / tt) : 0.0;
  for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < L.N; n += gridDim.x * blockDim.x) {
    const unsigned c0 = bf16_bits((float)(t[pos_of_natural(L, n)] * inv_s));
    const unsigned c1 = bf16_bits(feat[n]), c2 = bf16_bits(feat[(size_t)L.N + n]);
    in0[2 * (size_t)n] = make_uint4(c0 | (c1 << 16), c2, 0u, 0u);
    in0[2 * (size_t)n + 1] = make_uint4(0u, 0u, 0u, 0u);
  }
}

// zl = z + w y + zs (zs the post-smoothing correction; zl = z when the step was
// declined); partials of zl.r
__global__ void __launch_bounds__(MF6_BLOCK) k_g_comb(int n, const FcgState *fs, const KState *ks,
                                                      const double *__restrict__ z,
                                                      const double *__restrict__ y,
                                                      const double *__restrict__ zs,
                                                      const double *__restrict__ r,
                                                      double *__restrict__ zl, double *part) {
  __shared__ double lds[4];
  if (ks->stop) return;
  const double w = fs->w;
  double s = 0.0;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
    const double v = w == 0.0 ? z[e] : (z[e] + w * y[e]) + zs[e];
    zl[e] = v;
    s = s + v * r[e];
  }
  s = call_sum<MF6_BLOCK>(s, lds);
  if (threadIdx.x == 0) part[G_ZR * G_MAXB + blockIdx.x] = s;
}

// up to FCG_NDOT dot products z . b_k in one pass; z is the ILU0 step, or the
// learned one where it is accepted: zl.r has the sign of the ILU0 step's z.r (a
// descent direction), else the ILU0 step stays for the rest of the solve.
// mode 0: z; 1: decide; 2: as decided
struct DotArgs {
  int n;
  const double *b[FCG_NDOT];
};

__global__ void __launch_bounds__(MF6_BLOCK) k_g_mdots(int n, int mode, DotArgs d,
                                                       const double *__restrict__ z,
                                                       const double *__restrict__ zl,
                                                       double *part, FcgState *fs,
                                                       const KState *ks, FoldHost *hf) {
  if (ks->stop) return;
  __shared__ double lds[FCG_NDOT][MF6_BLOCK / 64], lds2[4];
  const double *a = z;
  if (mode == 1) {
    const double w = fs->w, zri = fs->zr_ilu;
    const double zr =
        call_sum<MF6_BLOCK>(cpart<MF6_BLOCK, G_NI>(part + G_ZR * G_MAXB, gridDim.x), lds2);
    const bool acc = w != 0.0 && zr * zri > 0.0 && isfinite(zr);
    if (acc) a = zl;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      fs->zr_l = zr;
      fs->acc = acc ? 1 : 0;
      if (acc) fs->learned_iters++;
      else if (w != 0.0) g_off(fs, hf);
    }
  } else if (mode == 2 && fs->acc) {
    a = zl;
  }
  double s[FCG_NDOT];
#pragma unroll
  for (int k = 0; k < FCG_NDOT; k++) s[k] = 0.0;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
    const double av = a[e];
#pragma unroll
    for (int k = 0; k < FCG_NDOT; k++)
      if (k < d.n) s[k] = s[k] + av * d.b[k][e];
  }
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < FCG_NDOT; k++) {
    const double t = csum(s[k]);
    if ((threadIdx.x & 63) == 0) lds[k][w] = t;
  }
  __syncthreads();
  if (threadIdx.x < d.n) {
    double t = 0.0;
#pragma unroll
    for (int v = 0; v < MF6_BLOCK / 64; v++) t = t + lds[threadIdx.x][v];
    part[threadIdx.x * G_MAXB + blockIdx.x] = t;
  }
}

// dot k's nb partials (fixed order) by block k
struct SumOut {
  double *o[FCG_NDOT];
};

__global__ void __launch_bounds__(MF6_BLOCK) k_fcg_sum(const double *part, int nb, SumOut out,
                                                       const KState *ks) {
  __shared__ double lds[MF6_BLOCK / 64];
  const int stop = ks->stop;
  const double s = call_sum<MF6_BLOCK>(
      cpart<MF6_BLOCK, G_NI>(part + blockIdx.x * G_MAXB, nb), lds);
  if (threadIdx.x == 0 && !stop) *out.o[blockIdx.x] = s;
}

// p = z - sum_j (c_j / pq_j) P_j over the stored slots
__global__ void __launch_bounds__(MF6_BLOCK) k_fcg_dir(int n, int learned,
                                                       const double *__restrict__ z,
                                                       const double *__restrict__ zl,
                                                       const double *__restrict__ P, size_t ld,
                                                       FcgSlots sl, const FcgState *fs,
                                                       double *__restrict__ p, const KState *ks) {
  if (ks->stop) return;
  __shared__ double cf[FCG_MAXM];
  const double *a = learned && fs->acc ? zl : z;
  if (threadIdx.x < sl.n) {
    const int k = sl.slot[threadIdx.x];
    const double pq = fs->pqs[k];
    // a direction without length is left out
    cf[threadIdx.x] = pq != 0.0 ? fs->c[k] / pq : 0.0;
  }
  __syncthreads();
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
    double v = a[e];
    for (int j0 = 0; j0 < sl.n; j0 += FCG_NDOT) {
      double pv[FCG_NDOT];
#pragma unroll
      for (int j = 0; j < FCG_NDOT; j++)
        if (j0 + j < sl.n) pv[j] = P[(size_t)sl.slot[j0 + j] * ld + e];
#pragma unroll
      for (int j = 0; j < FCG_NDOT; j++)
        if (j0 + j < sl.n && cf[j0 + j] != 0.0) v = v - cf[j0 + j] * pv[j];
    }
    p[e] = v;
  }
}

// x += alpha p ; r -= alpha q with alpha = p.r / p.q ; partials: sum r^2,
// signed max |alpha p| and max |r| with natural locations (first occurrence
// on ties)
template <int BS>
__global__ void __launch_bounds__(BS) k_g_update(Layout L, FcgState *fs, int head,
                                                 double *__restrict__ x,
                                                 const double *__restrict__ p,
                                                 double *__restrict__ r,
                                                 const double *__restrict__ q, double *part,
                                                 MaxLoc *mpart, const KState *ks, int nq, int ny) {
  __shared__ double lds[3][4];
  __shared__ MaxLoc ml[2][4];
  const int HP = L.HP;
  const int stop = ks->stop;
  double pq = cpart<BS, G_NI>(part + G_D0 * G_MAXB, gridDim.x);
  double pr = cpart<BS, G_NI>(part + G_D1 * G_MAXB, gridDim.x);
  if (stop) return;
  pq = call_sum<BS>(pq, lds[0]);
  pr = call_sum<BS>(pr, lds[1]);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    fs->pqs[head] = pq;
    fs->pr = pr;
  }
  const double alpha = pr / (pq + copysign(DPREC_C, pq));
  double ss = 0.0;
  MaxLoc mx{0.0, -1}, mr{0.0, -1};
  const int chunks = (L.nlay + C_CH - 1) / C_CH;
  for (int lb = cblock(blockIdx.x, gridDim.x); lb < nq; lb += gridDim.x) {
    const int t = (lb / ny) * BS + threadIdx.x;
    const int c = t & 1, h = t >> 1;
    if (h >= ncols_of(L, c)) continue;
    const int cy = lb % ny;
    const int ka = chunks * cy / ny * C_CH, kb = chunks * (cy + 1) / ny * C_CH;
    const int own = c * L.H + h, l = col_l(L, c, h);
    for (int k0 = ka; k0 < kb; k0 += C_CH) {
      double xv[C_CH], pv[C_CH], rv[C_CH], qv[C_CH];
#pragma unroll
      for (int u = 0; u < C_CH; u++) {
        if (u > 0 && k0 + u >= L.nlay) break;
        const int pos = own + (k0 + u) * HP;
        xv[u] = x[pos];
        pv[u] = p[pos];
        rv[u] = r[pos];
        qv[u] = q[pos];
      }
#pragma unroll
      for (int u = 0; u < C_CH; u++) {
        const int k = k0 + u;
        if (k < L.nlay) {
          const int pos = own + k * HP, nat = k * L.NRC + l;
          const double dx = alpha * pv[u];
          x[pos] = xv[u] + dx;
          const double v = rv[u] - alpha * qv[u];
          r[pos] = v;
          ss = ss + v * v;
          mx = maxloc_pick(mx, MaxLoc{dx, nat});
          mr = maxloc_pick(mr, MaxLoc{v, nat});
        }
      }
    }
  }
  ss = call_sum<BS>(ss, lds[2]);
  mx = call_max<BS>(mx, ml[0]);
  mr = call_max<BS>(mr, ml[1]);
  if (threadIdx.x == 0) {
    part[G_SS * G_MAXB + blockIdx.x] = ss;
    mpart[GM_X * G_MAXB + blockIdx.x] = mx;
    mpart[GM_R * G_MAXB + blockIdx.x] = mr;
  }
}

// End of an iteration: norms, the IMS test, the stall check of the learned step.
// When the test passes, r = b - A x (amux order), the FP64 true residual, and
// partials of max |r|: the next sweep decides on them.
__global__ void __launch_bounds__(MF6_BLOCK) k_g_test(Layout L, const double *__restrict__ A,
                                                      const double *__restrict__ x,
                                                      const double *__restrict__ b,
                                                      double *__restrict__ r, const double *part,
                                                      MaxLoc *mpart, int nb, FcgState *fs,
                                                      const KState *ks, FcgTest tst,
                                                      FoldHost *hf) {
  __shared__ double lds[4];
  __shared__ MaxLoc ml[3][4];
  const int stop = ks->stop;
  double s = cpart<MF6_BLOCK, G_NI>(part + G_SS * G_MAXB, nb);
  MaxLoc ra = cmpart<MF6_BLOCK, G_NI>(mpart + GM_X * G_MAXB, nb);
  MaxLoc rb = cmpart<MF6_BLOCK, G_NI>(mpart + GM_R * G_MAXB, nb);
  if (stop) return;
  s = call_sum<MF6_BLOCK>(s, lds);
  ra = call_max<MF6_BLOCK>(ra, ml[0]);
  rb = call_max<MF6_BLOCK>(rb, ml[1]);
  const double rnorm = sqrt(s), dvmax = ra.v, rmax = rb.v;
  // IMS test on the signed maxima (ICNVGOPT 0 / 1), or with the L2 norm
  bool conv = fabs(dvmax) <= tst.dvclose && fabs(rmax) <= tst.rclose;
  if (tst.icnvgopt == 2 || tst.icnvgopt == 3 || tst.icnvgopt == 4)
    conv = fabs(dvmax) <= tst.dvclose && (tst.icnvgopt == 3 || rnorm <= tst.rclose);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    fs->rnorm = rnorm;
    fs->dvmax = dvmax;
    fs->rmax = rmax;
    fs->iter++;
    fs->cand = conv ? 1 : 0;
    // stall check of the learned step over windows of ten applications
    if (fs->learned) {
      if (fs->window == 0) fs->rn_window = rnorm;
      if (++fs->window == 10 * tst.nn_every) {
        if (!(rnorm < 0.9 * fs->rn_window)) g_off(fs, hf);
        fs->window = 0;
      }
    }
  }
  if (!conv) return;
  const int NP = L.NP;
  MaxLoc m{0.0, -1};
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < NP; e += gridDim.x * blockDim.x) {
    int c, k, i, j, l;
    if (!pos_to_cell(L, e, c, k, i, j, l)) { r[e] = 0.0; continue; }
    const int ob = (1 - c) * L.H + k * L.HP;
    double t = 0.0;
    t = t + A[e] * x[e];
    if (k > 0) t = t + A[NP + e] * x[e - L.HP];
    if (i > 0) t = t + A[2 * NP + e] * x[ob + hn(l, -L.ncol)];
    if (j > 0) t = t + A[3 * NP + e] * x[ob + hn(l, -1)];
    if (j < L.ncol - 1) t = t + A[4 * NP + e] * x[ob + hn(l, 1)];
    if (i < L.nrow - 1) t = t + A[5 * NP + e] * x[ob + hn(l, L.ncol)];
    if (k < L.nlay - 1) t = t + A[6 * NP + e] * x[e + L.HP];
    const double rv = b[e] - t;
    r[e] = rv;
    m = maxloc_pick(m, MaxLoc{rv, e});
  }
  m = call_max<MF6_BLOCK>(m, ml[2]);
  if (threadIdx.x == 0) mpart[GM_T * G_MAXB + blockIdx.x] = m;
}

inline int gsz(int n) {
  int g = (n + MF6_BLOCK - 1) / MF6_BLOCK;
  if (g > 2048) g = 2048;
  return g < 1 ? 1 : g;
}

}  // namespace

#define FCK(x)                        \
  do {                                \
    int rc_ = (x);                    \
    if (rc_ != MF6HIP_OK) return rc_; \
  } while (0)

namespace {

// 64 threads a block where 512 blocks hold every chunk of four layers, else 256;
// a chunk per thread while that leaves at most G_MAXB blocks, else a column
// (above G_MAXB blocks of columns each takes several)
struct GGrid {
  int bs, nc, ny, nq, nb;   // threads; blocks of one colour; chunks a column; of all; launched
};

GGrid g_grid(const Layout &L) {
  GGrid g{};
  g.ny = (L.nlay + C_CH - 1) / C_CH;
  g.bs = (2 * L.HP0 + 63) / 64 * g.ny <= 512 ? 64 : 256;
  const int n = (2 * L.HP0 + g.bs - 1) / g.bs;
  if (n * g.ny > G_MAXB) g.ny = 1;
  g.nc = (L.HP0 + g.bs - 1) / g.bs;
  g.nq = n * g.ny;
  g.nb = g.nq < G_MAXB ? g.nq : G_MAXB;
  return g;
}

// one solve's kernels
struct Fcg {
  Mf6Handle *h;
  GGrid g;
  FcgState *fs;
  double *part;
  FcgTest tst;
  int nr;   // blocks of the true residual
};

template <int BS, bool LEARNED>
void g_ilu(const Fcg &c, const double *x, const double *ay, double *z) {
  Mf6Handle *h = c.h;
  const Layout &L = h->L;
  hipStream_t s = h->stream;
  const double *A = h->A, *piv = h->invpiv;
  k_g_red<BS, LEARNED><<<c.g.nc, BS, 0, s>>>(L, A, piv, x, ay, h->zf, c.part, h->d_mpart, c.g.nb,
                                             c.nr, c.tst, c.fs, h->d_state, h->h_fold);
#define MF6_G(N) \
  k_g_black<BS, LEARNED, N><<<c.g.nc, BS, 0, s>>>(L, A, piv, x, ay, h->zf, z, c.fs)
  if (L.nlay <= 4) MF6_G(4);
  else if (L.nlay <= 8) MF6_G(8);
  else if (L.nlay <= 16) MF6_G(16);
  else MF6_G(32);
#undef MF6_G
  k_g_bwd<BS><<<c.g.nc, BS, 0, s>>>(L, A, piv, h->zf, z, c.fs, h->d_state);
}

template <int BS, int MODE>
void g_mv(const Fcg &c, const double *x, const float *net, double *xs, const double *aux,
          double *out) {
  k_g_mv<BS, MODE><<<c.g.nb, BS, 0, c.h->stream>>>(c.h->L, c.h->A, x, net, xs, aux, out, c.part,
                                                   c.fs, c.h->d_state, c.g.nq, c.g.ny);
}

// z = ILU0(r), plus the learned step into zl when `learned` (enqueued only; the
// weight is decided on the device)
template <int BS>
int precondition(const Fcg &c, const double *r, double *z, double *zl, bool learned) {
  Mf6Handle *h = c.h;
  const Layout &L = h->L;
  hipStream_t s = h->stream;
  g_ilu<BS, false>(c, r, nullptr, z);
  if (!learned) return MF6HIP_OK;
  double *t = h->v, *yv = h->dhat, *ay = h->phat, *zs = h->p;
  g_mv<BS, G_RES>(c, z, nullptr, nullptr, r, t);
  k_fcg_nn_input<<<gsz(L.N), MF6_BLOCK, 0, s>>>(L, t, c.part, c.g.nb, c.fs, h->d_state,
                                                h->unet_feat, (uint4 *)mf6hip_unet_input(h->unet));
  FCK(mf6hip_unet_apply_device(h->unet, s));
  g_mv<BS, G_NET>(c, nullptr, mf6hip_unet_output(h->unet), yv, t, ay);
  // post-smoothing of r - A (z + w y) = t - w A y
  g_ilu<BS, true>(c, t, ay, zs);
  k_g_comb<<<gsz(L.NP), MF6_BLOCK, 0, s>>>(L.NP, c.fs, h->d_state, z, yv, zs, r, zl, c.part);
  return MF6HIP_OK;
}

template <int BS>
int run_fcg(Fcg c, double *P, double *Q) {
  Mf6Handle *h = c.h;
  const Layout &L = h->L;
  hipStream_t s = h->stream;
  KState *hs = h->h_state;
  const int m = h->fcg_m, nb = gsz(L.NP), itmax = h->s.iter1;
  double *r = h->d, *z = h->z, *zl = h->qhat;
  const bool net = h->unet != nullptr;
  k_fcg_init<<<1, 64, 0, s>>>(c.fs, h->d_state, net ? 1 : 0);
  HIPCHK(hipGetLastError());
  int nstored = 0, head = 0, it = 0;
  auto group = [&](int ev) -> int {
    for (int g = 0; g < FCG_GROUP && it < itmax; g++) {
      it++;
      const bool use_net = net && ((it - 1) % h->nn_every == 0) &&
                           __atomic_load_n(&h->h_fold->off, __ATOMIC_RELAXED) == 0;
      FCK(precondition<BS>(c, r, z, zl, use_net));
      // c_j = z.q_j over the stored slots (newest first), FCG_NDOT a pass
      FcgSlots sl{};
      sl.n = nstored;
      for (int j = 0; j < nstored; j++) sl.slot[j] = (head - 1 - j + 2 * m) % m;
      for (int j0 = 0; j0 < nstored || (j0 == 0 && use_net); j0 += FCG_NDOT) {
        const int nd = nstored - j0 < FCG_NDOT ? nstored - j0 : FCG_NDOT;
        DotArgs da{};
        da.n = nd;
        SumOut so{};
        for (int k = 0; k < nd; k++) {
          da.b[k] = Q + (size_t)sl.slot[j0 + k] * L.NP;
          so.o[k] = &c.fs->c[sl.slot[j0 + k]];
        }
        k_g_mdots<<<nb, MF6_BLOCK, 0, s>>>(L.NP, use_net ? (j0 == 0 ? 1 : 2) : 0, da, z, zl,
                                           c.part, c.fs, h->d_state, h->h_fold);
        if (nd > 0) k_fcg_sum<<<nd, MF6_BLOCK, 0, s>>>(c.part, nb, so, h->d_state);
      }
      // the new direction goes straight into the ring slot `head`
      double *p = P + (size_t)head * L.NP, *q = Q + (size_t)head * L.NP;
      k_fcg_dir<<<nb, MF6_BLOCK, 0, s>>>(L.NP, use_net ? 1 : 0, z, zl, P, (size_t)L.NP, sl, c.fs,
                                         p, h->d_state);
      g_mv<BS, G_DIR>(c, p, nullptr, nullptr, r, q);
      k_g_update<BS><<<c.g.nb, BS, 0, s>>>(L, c.fs, head, h->x, p, r, q, c.part, h->d_mpart,
                                           h->d_state, c.g.nq, c.g.ny);
      k_g_test<<<c.nr, MF6_BLOCK, 0, s>>>(L, h->A, h->x, h->b, r, c.part, h->d_mpart, c.g.nb, c.fs,
                                          h->d_state, c.tst, h->h_fold);
      HIPCHK(hipGetLastError());
      head = (head + 1) % m;
      if (nstored < m) nstored++;
    }
    if (it >= itmax)
      k_g_last<<<1, 64, 0, s>>>(h->d_mpart, c.nr, c.tst, c.fs, h->d_state, h->h_fold);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(h->ev_batch[ev], s));
    return MF6HIP_OK;
  };
  h->h_fold->stop = h->h_fold->off = 0;   // nothing of an earlier solve is still running
  FCK(group(0));
  for (int ev = 0;; ev ^= 1) {
    const bool more = it < itmax;
    if (more) FCK(group(ev ^ 1));
    HIPCHK(hipEventSynchronize(h->ev_batch[ev]));
    if (!more || __atomic_load_n(&h->h_fold->stop, __ATOMIC_ACQUIRE) != 0) break;
  }
  FcgState hf{};
  HIPCHK(hipMemcpyAsync(&hf, c.fs, sizeof(FcgState), hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  hs->icnvg = hf.icnvg;
  hs->iter = hf.iter;
  hs->deltax = hf.dvmax;
  hs->rmax = hf.rmax;
  hs->l2norm = hf.rnorm;
  hs->stop = 1;
  h->learned_iters = hf.learned_iters;
  HIPCHK(hipMemcpyAsync(h->d_state, hs, sizeof(KState), hipMemcpyHostToDevice, s));
  return MF6HIP_OK;
}

}  // namespace

// Flexible CG on the device system; h->d = b - A x, the ILU0 factor and
// the initial state (l2norm0, settings) are in place.  The new direction is
// A-orthogonalised against the last fcg_m directions (FCG(m)).
int mf6hip_run_fcg(Mf6Handle *h) {
  const Layout &L = h->L;
  const int m = h->fcg_m;
  const size_t vec = sizeof(double) * 2 * (size_t)m * L.NP;
  if (!h->fcg_store) {
    const size_t bytes = vec + sizeof(FcgState) + sizeof(double) * G_NSLOT * G_MAXB;
    if (hipMalloc((void **)&h->fcg_store, bytes) != hipSuccess) {
      mf6hip_set_error("hipMalloc failed (flexible CG directions)");
      return MF6HIP_EHIP;
    }
    // the SpMV leaves the padding of A p_j alone
    HIPCHK(hipMemsetAsync(h->fcg_store, 0, vec, h->stream));
  }
  static_assert(3 * G_MAXB <= 4 * MF6_MAXBLK, "maxima fit their array");
  Fcg c{};
  c.h = h;
  c.g = g_grid(L);
  c.fs = (FcgState *)(h->fcg_store + 2 * (size_t)m * L.NP);
  c.part = (double *)(c.fs + 1);
  c.tst = FcgTest{h->s.dvclose, h->s.rclose, h->s.icnvgopt, h->nn_every};
  c.nr = gsz(L.NP) < G_RB ? gsz(L.NP) : G_RB;
  double *P = h->fcg_store, *Q = h->fcg_store + (size_t)m * L.NP;
  return c.g.bs == 64 ? run_fcg<64>(c, P, Q) : run_fcg<256>(c, P, Q);
}

extern "C" int mf6hip_attach_unet(void *handle, void *net, const float *features, int fcg_m,
                                  int nn_every) {
  Mf6Handle *h = (Mf6Handle *)handle;
  if (!h) { mf6hip_set_error("null handle"); return MF6HIP_EINVAL; }
  if (fcg_m < 1 || fcg_m > 64) { mf6hip_set_error("fcg_m must be 1..64"); return MF6HIP_EINVAL; }
  if (nn_every < 1) { mf6hip_set_error("nn_every must be >= 1"); return MF6HIP_EINVAL; }
  h->nn_every = nn_every;
  if (fcg_m != h->fcg_m && h->fcg_store) {
    hipFree(h->fcg_store);
    h->fcg_store = nullptr;
  }
  h->fcg_m = fcg_m;
  if (!net) { h->unet = nullptr; return MF6HIP_OK; }
  if (!features) { mf6hip_set_error("features required"); return MF6HIP_EINVAL; }
  int nl, nr, nc, nin;
  FCK(mf6hip_unet_dims(net, &nl, &nr, &nc, &nin));
  if (nl != h->L.nlay || nr != h->L.nrow || nc != h->L.ncol || nin != 3) {
    mf6hip_set_error("network grid or inputs do not match the solver");
    return MF6HIP_EINVAL;
  }
  if (!h->unet_feat) {
    if (hipMalloc((void **)&h->unet_feat, sizeof(float) * 2 * (size_t)h->L.N) != hipSuccess) {
      mf6hip_set_error("hipMalloc failed");
      return MF6HIP_EHIP;
    }
  }
  HIPCHK(hipMemcpy(h->unet_feat, features, sizeof(float) * 2 * (size_t)h->L.N, hipMemcpyHostToDevice));
  h->unet = net;
  return MF6HIP_OK;
}

extern "C" int mf6hip_last_learned_iterations(void *handle, int *n) {
  Mf6Handle *h = (Mf6Handle *)handle;
  if (!h || !n) { mf6hip_set_error("null argument"); return MF6HIP_EINVAL; }
  *n = h->learned_iters;
  return MF6HIP_OK;
}
