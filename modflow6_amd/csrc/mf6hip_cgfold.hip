// mf6hip_cgfold.hip -- the FP64 CG of symmetric systems (ims_base_cg,
// src/Solution/LinearMethods/ImsLinearBase.f90:30-240) for grids whose
// iteration is bound by kernel latency, not by memory bandwidth.
//
// The fused CG (mf6hip_cgfused.hip) runs an iteration in seven kernels, two of
// them one-block reductions.  On a few hundred thousand cells each of them is
// a chain of memory latencies (the solve state, then layer after layer, then
// the partial sums) on a few dozen workgroups: 4 to 9 us a kernel where an
// empty one takes 1.9 us in a graph.  Here an iteration is four kernels:
//
//   k_c_red    alpha from the partials of p.q (every workgroup adds them in the
//              same order, so all get the same bits); d -= alpha q (red cells);
//              forward ILU0 sweep of the red columns
//   k_c_black  d -= alpha q (black); forward and backward sweep; partial rho
//   k_c_bwd    backward sweep of the red columns; partial rho
//   k_c_spmv   rho and beta from the partials, likewise; p = z + beta p at the
//              cell and, again, at its neighbours; x += alpha p_prev; q = A p;
//              partials of p.q and max |p|.  One workgroup more than the columns
//              need runs the convergence test of the finished iteration (the
//              sums and maxima it needs are reduced by extra workgroups of the
//              kernels before it).
//
// One column per thread (k_c_spmv: per chunk of four layers); the loads of a
// chunk and of the solve state are all issued before anything waits for them,
// and a column's sweep values stay in registers.  Per cell the arithmetic and its order are those
// of the fused kernels; the head update of the last iteration is applied by
// the same k_c_spmv that finds it converged.
//
// Measured (FP64 ILU0, us per iteration, fused -> folded): 3 x 100 x 100
// 47.4 -> 19.5, 4 x 256 x 256 54.7 -> 28.0, 10 x 300 x 300 87.0 -> 56.8,
// 10 x 350 x 350 94.5 -> 59.3, 30 x 200 x 200 172 -> 84.
#include <cstring>
#include <string>

#include "mf6hip_fold.h"

#define CK(x)                         \
  do {                                \
    int rc_ = (x);                    \
    if (rc_ != MF6HIP_OK) return rc_; \
  } while (0)

namespace {

// state beyond KState: what one kernel of an iteration leaves for the next
// ones (no kernel reads a field that it writes itself)
struct CState {
  double rho[2];   // rho of the last two iterations, by round parity
  int have;        // a direction exists: alpha is defined
  int stop;        // the test's result; k_c_red copies it to KState::stop
  double ss;       // sum of squares and maximum of the residual, max |p|
  MaxLoc md, mp;
};

// slots of the partial arrays (C_MAXPART each)
enum { CP_SSR = 0, CP_SSB = 1, CP_RHOB = 2, CP_RHOR = 3, CP_PQ = 4 };
enum { CM_DR = 0, CM_DB = 1, CM_P = 2 };   // CM_P, CM_P + 1: by round parity

// partials per thread of the colour kernels (at most 256 blocks) and of
// k_c_spmv (at most C_MAXPART)
template <int BS>
constexpr int NI_C = 256 / BS;
template <int BS>
constexpr int NI_Q = BS == 64 ? 512 / 64 : C_MAXPART / BS;

// NL bounds the layers at compile time: the chunks' loads are double-buffered
// and a column's values stay in registers.  (At most FOLD_MAXCOL / 2 columns of
// a colour are at most one wave per SIMD, so registers cost no occupancy.)
// The last block reduces max |p| of the last direction for the test.
template <int BS, int NL>
__global__ void __launch_bounds__(BS) k_c_red(Layout L, const double *__restrict__ A,
                                              const double *__restrict__ piv,
                                              double *__restrict__ d,
                                              const double *__restrict__ q,
                                              double *__restrict__ zf, double *part,
                                              MaxLoc *mpart, KState *st, CState *cs, int nc,
                                              int nq, int par) {
  __shared__ double lds[4], lds2[4];
  __shared__ MaxLoc mlds[4];
  if ((int)blockIdx.x == nc) {
    const MaxLoc mp = call_max<BS>(cmpart<BS, NI_Q<BS>>(mpart + (CM_P + 1 - par) * C_MAXPART, nq), mlds);
    if (threadIdx.x == 0) cs->mp = mp;
    return;
  }
  const int lb = cblock(blockIdx.x, nc);
  const int NP = L.NP, HP = L.HP;
  const int stop = cs->stop, have = cs->have, iter = st->iter;
  const double rho = cs->rho[1 - par];
  double pq = cpart<BS, NI_Q<BS>>(part + CP_PQ * C_MAXPART, nq);
  const int h2 = lb * BS + threadIdx.x;
  const bool in = h2 < L.HP0;
  const int h = in ? h2 : 0;
  double dv[2][C_CH], qv[2][C_CH], a6[2][C_CH], pv[2][C_CH];
  auto load = [&](int k0, int b) {
#pragma unroll
    for (int u = 0; u < C_CH; u++) {
      const int p = (k0 + u < L.nlay ? k0 + u : L.nlay - 1) * HP + h;
      dv[b][u] = d[p];
      qv[b][u] = q[p];
      a6[b][u] = A[6 * NP + p];
      pv[b][u] = piv[p];
    }
  };
  load(0, 0);
  pq = call_sum<BS>(pq, lds);
  const double alpha = have ? rho / (pq + copysign(DPREC_C, pq)) : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (stop) st->stop = stop;
    else if (have) {
      st->pq = pq;
      st->alpha = alpha;
      st->iter = iter + 1;
    }
  }
  if (stop) return;
  double ss = 0.0, zup = 0.0, lup = 0.0;
  MaxLoc md{0.0, -1};
  if (in) {
    const int l = col_l(L, 0, h2);
#pragma unroll
    for (int k0 = 0; k0 < NL; k0 += C_CH) {
      if (k0 >= L.nlay) break;
      const int b = (k0 / C_CH) & 1;
      if (k0 + C_CH < NL) load(k0 + C_CH, 1 - b);
#pragma unroll
      for (int u = 0; u < C_CH; u++) {
        const int k = k0 + u;
        if (k < L.nlay) {
          const int p = k * HP + h2;
          const double x = dv[b][u] - alpha * qv[b][u];
          double tv = x;
          d[p] = x;
          md = maxloc_pick(md, MaxLoc{x, k * L.NRC + l});
          ss = ss + x * x;
          if (k > 0) tv = tv - lup * zup;
          zf[p] = tv;
          zup = tv;
          lup = a6[b][u] * pv[b][u];
        }
      }
    }
  }
  ss = call_sum<BS>(ss, lds2);
  md = call_max<BS>(md, mlds);
  if (threadIdx.x == 0) {
    part[CP_SSR * C_MAXPART + lb] = ss;
    mpart[CM_DR * C_MAXPART + lb] = md;
  }
}

template <int BS, int NL>
__global__ void __launch_bounds__(BS) k_c_black(Layout L, const double *__restrict__ A,
                                                const double *__restrict__ piv,
                                                double *__restrict__ d,
                                                const double *__restrict__ q,
                                                const double *__restrict__ zf,
                                                double *__restrict__ z, double *part,
                                                MaxLoc *mpart, const KState *st) {
  __shared__ double lds[4], lds2[4];
  __shared__ MaxLoc mlds[4];
  const int lb = xcd_block();
  const int NP = L.NP, HP = L.HP;
  const int stop = st->stop;
  const double alpha = st->iter > 0 ? st->alpha : 0.0;
  const int h2 = lb * BS + threadIdx.x;
  const bool in = h2 < L.HP1;
  const int h = in ? h2 : 0;
  double ss = 0.0, rho = 0.0, zup = 0.0, lup = 0.0;
  MaxLoc md{0.0, -1};
  double zc[NL], dc[NL], ac[NL], pc[NL];
  if (in) {
    const CGeo G(L, 1, h);
    double ab[2][C_CH], pb[2][C_CH], zb[2][C_CH], al[2][C_CH], pl[2][C_CH], zl[2][C_CH],
        ar[2][C_CH], pr[2][C_CH], zr[2][C_CH], af[2][C_CH], pf[2][C_CH], zf_[2][C_CH], qv[2][C_CH];
    auto load = [&](int k0, int b) {
#pragma unroll
      for (int u = 0; u < C_CH; u++) {
        const int k = k0 + u < L.nlay ? k0 + u : L.nlay - 1;
        const int pos = L.H + k * HP + h, rb = k * HP;
        ab[b][u] = A[5 * NP + rb + G.ib];
        pb[b][u] = piv[rb + G.ib];
        zb[b][u] = zf[rb + G.ib];
        al[b][u] = A[4 * NP + rb + G.il];
        pl[b][u] = piv[rb + G.il];
        zl[b][u] = zf[rb + G.il];
        ar[b][u] = A[4 * NP + pos];
        pr[b][u] = piv[rb + G.ir];
        zr[b][u] = zf[rb + G.ir];
        af[b][u] = A[5 * NP + pos];
        pf[b][u] = piv[rb + G.ifr];
        zf_[b][u] = zf[rb + G.ifr];
        ac[k0 + u] = A[6 * NP + pos];
        pc[k0 + u] = piv[pos];
        dc[k0 + u] = d[pos];
        qv[b][u] = q[pos];
      }
    };
    load(0, 0);
    if (stop) return;
#pragma unroll
    for (int k0 = 0; k0 < NL; k0 += C_CH) {
      if (k0 >= L.nlay) break;
      const int b = (k0 / C_CH) & 1;
      if (k0 + C_CH < NL) load(k0 + C_CH, 1 - b);
#pragma unroll
      for (int u = 0; u < C_CH; u++) {
        const int k = k0 + u;
        if (k < L.nlay) {
          const double x = dc[k] - alpha * qv[b][u];
          double tv = x;
          d[L.H + k * HP + h] = x;
          dc[k] = x;
          md = maxloc_pick(md, MaxLoc{x, k * L.NRC + G.l});
          ss = ss + x * x;
          tv = G.hb ? tv - ab[b][u] * pb[b][u] * zb[b][u] : tv;
          tv = G.hl ? tv - al[b][u] * pl[b][u] * zl[b][u] : tv;
          tv = G.hr ? tv - ar[b][u] * pr[b][u] * zr[b][u] : tv;
          tv = G.hf ? tv - af[b][u] * pf[b][u] * zf_[b][u] : tv;
          if (k > 0) tv = tv - lup * zup;
          zc[k] = tv;
          zup = tv;
          lup = ac[k] * pc[k];
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
        rho = rho + dc[k] * tv;
      }
    }
  }
  if (stop) return;
  ss = call_sum<BS>(ss, lds);
  rho = call_sum<BS>(rho, lds2);
  md = call_max<BS>(md, mlds);
  if (threadIdx.x == 0) {
    part[CP_SSB * C_MAXPART + lb] = ss;
    part[CP_RHOB * C_MAXPART + lb] = rho;
    mpart[CM_DB * C_MAXPART + lb] = md;
  }
}

// the last block reduces the residual's sum of squares and maximum
template <int BS, int NL>
__global__ void __launch_bounds__(BS) k_c_bwd(Layout L, const double *__restrict__ A,
                                              const double *__restrict__ piv,
                                              const double *__restrict__ d,
                                              const double *__restrict__ zf,
                                              double *__restrict__ z, double *part,
                                              const MaxLoc *mpart, const KState *st, CState *cs,
                                              int nc) {
  __shared__ double lds[4], lds2[4];
  __shared__ MaxLoc mlds[4], mlds2[4];
  const int stop = st->stop;
  if ((int)blockIdx.x == nc) {
    double a = cpart<BS, NI_C<BS>>(part + CP_SSR * C_MAXPART, nc);
    double b = cpart<BS, NI_C<BS>>(part + CP_SSB * C_MAXPART, nc);
    MaxLoc r = cmpart<BS, NI_C<BS>>(mpart + CM_DR * C_MAXPART, nc);
    MaxLoc k = cmpart<BS, NI_C<BS>>(mpart + CM_DB * C_MAXPART, nc);
    a = call_sum<BS>(a, lds);
    b = call_sum<BS>(b, lds2);
    r = call_max<BS>(r, mlds);
    k = call_max<BS>(k, mlds2);
    if (threadIdx.x == 0 && !stop) {
      cs->ss = a + b;
      cs->md = maxloc_pick(r, k);
    }
    return;
  }
  const int lb = cblock(blockIdx.x, nc);
  const int NP = L.NP, HP = L.HP;
  const int h2 = lb * BS + threadIdx.x;
  double rho = 0.0;
  if (h2 < L.HP0) {
    const CGeo G(L, 0, h2);
    double zv[2][C_CH], a6[2][C_CH], ab[2][C_CH], zb[2][C_CH], al[2][C_CH], zl[2][C_CH],
        ar[2][C_CH], zr[2][C_CH], af[2][C_CH], zf_[2][C_CH], pv[2][C_CH], dv[2][C_CH];
    // layers k0 + C_CH - 1 down to k0
    auto load = [&](int k0, int b) {
#pragma unroll
      for (int u = 0; u < C_CH; u++) {
        const int k = k0 + u < L.nlay ? k0 + u : L.nlay - 1;
        const int pos = k * HP + h2, bb = L.H + k * HP;
        zv[b][u] = zf[pos];
        a6[b][u] = A[6 * NP + pos];
        ab[b][u] = A[5 * NP + bb + G.ib];
        zb[b][u] = z[bb + G.ib];
        al[b][u] = A[4 * NP + bb + G.il];
        zl[b][u] = z[bb + G.il];
        ar[b][u] = A[4 * NP + pos];
        zr[b][u] = z[bb + G.ir];
        af[b][u] = A[5 * NP + pos];
        zf_[b][u] = z[bb + G.ifr];
        pv[b][u] = piv[pos];
        dv[b][u] = d[pos];
      }
    };
    double zdn = 0.0;
    // the chunks from the last one that holds a layer; NL / C_CH of them at
    // most, so the buffers alternate by the chunk's number
    const int top = (L.nlay - 1) / C_CH * C_CH;
#pragma unroll
    for (int k0 = NL - C_CH; k0 >= 0; k0 -= C_CH) {
      if (k0 > top) continue;
      const int b = (k0 / C_CH) & 1;
      if (k0 == top) load(k0, b);
      if (stop) return;
      if (k0 >= C_CH) load(k0 - C_CH, 1 - b);
#pragma unroll
      for (int u = C_CH - 1; u >= 0; u--) {
        const int k = k0 + u;
        if (k < L.nlay) {
          double tv = zv[b][u];
          if (k < L.nlay - 1) tv = tv - a6[b][u] * zdn;
          tv = G.hb ? tv - ab[b][u] * zb[b][u] : tv;
          tv = G.hl ? tv - al[b][u] * zl[b][u] : tv;
          tv = G.hr ? tv - ar[b][u] * zr[b][u] : tv;
          tv = G.hf ? tv - af[b][u] * zf_[b][u] : tv;
          tv = tv * pv[b][u];
          z[k * HP + h2] = tv;
          zdn = tv;
          rho = rho + dv[b][u] * tv;
        }
      }
    }
  }
  if (stop) return;
  rho = call_sum<BS>(rho, lds);
  if (threadIdx.x == 0) part[CP_RHOR * C_MAXPART + lb] = rho;
}

// The convergence test of iteration S.iter on the residual that the sweeps
// just formed; leaves rho of the next iteration and the stop code.
template <int BS>
__device__ inline void c_test(KState *st, CState *cs, const double *part, int nc, int par,
                              double *hist, int *hloc, FoldHost *hf) {
  __shared__ double l2[4], l3[4];
  const KState S = *st;
  const double rho = cs->rho[1 - par], rho0 = cs->rho[par], ss = cs->ss;
  const MaxLoc md = cs->md, mp = cs->mp;
  double rb = cpart<BS, NI_C<BS>>(part + CP_RHOB * C_MAXPART, nc);
  double rr = cpart<BS, NI_C<BS>>(part + CP_RHOR * C_MAXPART, nc);
  if (S.stop) return;
  rb = call_sum<BS>(rb, l2);
  rr = call_sum<BS>(rr, l3);
  const double rho_new = rb + rr;
  if (threadIdx.x != 0) return;
  const int it = S.iter;
  cs->have = 1;
  if (it > 0) {
    const double l2norm = sqrt(ss);
    const double deltax = S.alpha * mp.v;
    st->deltax = deltax;
    st->xloc = mp.loc;
    st->rmax = md.v;
    st->rloc = md.loc;
    st->l2norm = l2norm;
    if (it <= S.hist_cap) {
      const int cap = S.hist_cap;
      hist[it - 1] = deltax;
      hist[cap + it - 1] = md.v;
      hist[2 * cap + it - 1] = S.alpha;
      hist[3 * cap + it - 1] = 0.0;
      hloc[it - 1] = mp.loc;
      hloc[cap + it - 1] = md.loc;
    }
    const int o = S.icnvgopt;
    const double rcnvg = (o == 2 || o == 3 || o == 4) ? l2norm : md.v;
    int icnvg = S.icnvg;
    c_testcnvg(o, &icnvg, it, deltax, rcnvg, S.l2norm0, S.epfact, S.dvclose, S.rclose);
    if (rcnvg == 0.0) icnvg = 1;
    st->icnvg = icnvg;
    int stop = 0;
    if (icnvg != 0) stop = 1;
    else if (c_close(rho, rho0) || rho == 0.0) stop = 2;
    else if (it >= S.itmax) stop = 3;
    if (stop) {
      cs->stop = stop;
      c_publish(hf, st, stop);
      return;
    }
    st->rho0 = rho;
  }
  st->rho = rho_new;
  cs->rho[par] = rho_new;
}

// One thread per column and chunk of C_CH layers (ny chunks; a product needs no
// walk down the column, and the chunks side by side hide each other's loads);
// adjacent threads take the red and the black column of one index.  The last
// block runs the test.
template <int BS>
__global__ void __launch_bounds__(BS) k_c_spmv(Layout L, const double *__restrict__ A,
                                               const double *__restrict__ z,
                                               const double *__restrict__ pin,
                                               double *__restrict__ pout, double *__restrict__ x,
                                               double *__restrict__ q, double *part,
                                               MaxLoc *mpart, KState *st, CState *cs, int nc,
                                               int nq, int ny, int par, double *hist, int *hloc,
                                               FoldHost *hf) {
  __shared__ double lds[4], lds2[4], lds3[4];
  __shared__ MaxLoc mlds[4];
  if ((int)blockIdx.x == nq) {
    c_test<BS>(st, cs, part, nc, par, hist, hloc, hf);
    return;
  }
  const int lb = cblock(blockIdx.x, nq);
  const int NP = L.NP, HP = L.HP;
  const int stop = st->stop, iter = st->iter;
  const double alpha = st->alpha, rho = cs->rho[1 - par];
  const bool first = iter == 0;
  // rho of the new residual, summed as the test sums it
  double rb = cpart<BS, NI_C<BS>>(part + CP_RHOB * C_MAXPART, nc);
  double rr = cpart<BS, NI_C<BS>>(part + CP_RHOR * C_MAXPART, nc);
  const int t = (lb / ny) * BS + threadIdx.x, k0 = (lb % ny) * C_CH;
  const int c = t & 1, h2 = t >> 1;
  const bool in = h2 < ncols_of(L, c);
  const int h = in ? h2 : 0;
  const CGeo G(L, c, h);
  const int own = c * L.H + h, oth = (1 - c) * L.H;
  // own column: z and the last direction of layers k0 - 1 .. k0 + C_CH
  double zo[C_CH + 2], po[C_CH + 2], xo[C_CH], a6[C_CH + 1];
  double a0[C_CH], a4[C_CH], a5[C_CH], ab[C_CH], al[C_CH];
  double zn[4][C_CH], pn[4][C_CH];
#pragma unroll
  for (int u = 0; u < C_CH + 2; u++) {
    int k = k0 + u - 1;
    k = k < 0 ? 0 : (k < L.nlay ? k : L.nlay - 1);
    zo[u] = z[own + k * HP];
    po[u] = pin[own + k * HP];
    if (u <= C_CH) a6[u] = A[6 * NP + own + k * HP];
  }
#pragma unroll
  for (int u = 0; u < C_CH; u++) {
    const int k = k0 + u < L.nlay ? k0 + u : L.nlay - 1;
    const int pos = own + k * HP, ob = oth + k * HP;
    xo[u] = x[pos];
    a0[u] = A[pos];
    a4[u] = A[4 * NP + pos];
    a5[u] = A[5 * NP + pos];
    ab[u] = A[5 * NP + ob + G.ib];
    al[u] = A[4 * NP + ob + G.il];
    zn[0][u] = z[ob + G.ib];
    zn[1][u] = z[ob + G.il];
    zn[2][u] = z[ob + G.ir];
    zn[3][u] = z[ob + G.ifr];
    pn[0][u] = pin[ob + G.ib];
    pn[1][u] = pin[ob + G.il];
    pn[2][u] = pin[ob + G.ir];
    pn[3][u] = pin[ob + G.ifr];
  }
  if (stop) return;
  rb = call_sum<BS>(rb, lds);
  rr = call_sum<BS>(rr, lds2);
  const double beta = (rb + rr) / rho;
  auto dir = [&](double zv, double pv) { return first ? zv : zv + beta * pv; };
  double s = 0.0;
  MaxLoc mp{0.0, -1};
  if (in) {
    double pprev = dir(zo[0], po[0]), pcur = dir(zo[1], po[1]);
#pragma unroll
    for (int u = 0; u < C_CH; u++) {
      const int k = k0 + u;
      if (k < L.nlay) {
        const int pos = own + k * HP;
        const double pnx = dir(zo[u + 2], po[u + 2]);
        if (!first) x[pos] = xo[u] + alpha * po[u + 1];
        pout[pos] = pcur;
        mp = maxloc_pick(mp, MaxLoc{pcur, k * L.NRC + G.l});
        double tq = 0.0;
        tq = tq + a0[u] * pcur;
        if (k > 0) tq = tq + a6[u] * pprev;
        if (G.hb) tq = tq + ab[u] * dir(zn[0][u], pn[0][u]);
        if (G.hl) tq = tq + al[u] * dir(zn[1][u], pn[1][u]);
        if (G.hr) tq = tq + a4[u] * dir(zn[2][u], pn[2][u]);
        if (G.hf) tq = tq + a5[u] * dir(zn[3][u], pn[3][u]);
        if (k < L.nlay - 1) tq = tq + a6[u + 1] * pnx;
        q[pos] = tq;
        s = s + pcur * tq;
        pprev = pcur;
        pcur = pnx;
      }
    }
  }
  s = call_sum<BS>(s, lds3);
  mp = call_max<BS>(mp, mlds);
  if (threadIdx.x == 0) {
    part[CP_PQ * C_MAXPART + lb] = s;
    mpart[(CM_P + par) * C_MAXPART + lb] = mp;
  }
}

struct FoldGrid {
  int bs, nc, ny, nq;   // threads, blocks of one colour, chunks of layers,
                        // blocks of both colours' chunks
};

// 64 threads a block where 512 blocks hold every column's chunks, else 256:
// small blocks spread a small grid over the CUs and need no reduction through
// LDS, but every block reads all partials.
FoldGrid fold_grid(const Layout &L) {
  FoldGrid g{};
  g.ny = (L.nlay + C_CH - 1) / C_CH;
  g.bs = (2 * L.HP0 + 63) / 64 * g.ny <= 512 ? 64 : 256;
  g.nc = (L.HP0 + g.bs - 1) / g.bs;
  g.nq = (2 * L.HP0 + g.bs - 1) / g.bs * g.ny;
  return g;
}

template <int BS, int NL>
void enqueue_nl(Mf6Handle *h, const FoldGrid &g, int n, hipEvent_t e0, hipEvent_t e1) {
  const Layout &L = h->L;
  hipStream_t s = h->stream;
  KState *st = h->d_state;
  CState *cs = reinterpret_cast<CState *>(h->d_state + 2);
  double *pbuf[2] = {h->p, h->p2};
  for (int r = 0; r < n; r++) {
    const int par = r & 1;
    k_c_red<BS, NL><<<g.nc + 1, BS, 0, s>>>(L, h->A, h->invpiv, h->d, h->q, h->zf, h->d_part,
                                            h->d_mpart, st, cs, g.nc, g.nq, par);
    k_c_black<BS, NL><<<g.nc, BS, 0, s>>>(L, h->A, h->invpiv, h->d, h->q, h->zf, h->z, h->d_part,
                                          h->d_mpart, st);
    k_c_bwd<BS, NL><<<g.nc + 1, BS, 0, s>>>(L, h->A, h->invpiv, h->d, h->zf, h->z, h->d_part,
                                            h->d_mpart, st, cs, g.nc);
    if (e0) (void)hipEventRecord(e0, s);
    k_c_spmv<BS><<<g.nq + 1, BS, 0, s>>>(L, h->A, h->z, pbuf[par], pbuf[1 - par], h->x, h->q,
                                         h->d_part, h->d_mpart, st, cs, g.nc, g.nq, g.ny, par,
                                         h->d_hist, h->d_hloc, h->h_fold);
    if (e0) (void)hipEventRecord(e1, s);
    e0 = e1 = nullptr;
  }
}

// n iterations (n even) from an even round.  The bound 12 is there for the ordinary
// models of nine to twelve layers: with 16 instead a step takes 3 to 5 % longer
// (10x300x300 48.5 -> 50.1 ms, 12x150x150 17.2 -> 18.2).
void enqueue_fold(Mf6Handle *h, const FoldGrid &g, int n, hipEvent_t e0 = nullptr,
                  hipEvent_t e1 = nullptr) {
  const int nl = h->L.nlay;
#define MF6_FOLD(N) \
  (g.bs == 64 ? enqueue_nl<64, N>(h, g, n, e0, e1) : enqueue_nl<256, N>(h, g, n, e0, e1))
  if (nl <= 4) MF6_FOLD(4);
  else if (nl <= 8) MF6_FOLD(8);
  else if (nl <= 12) MF6_FOLD(12);
  else if (nl <= 16) MF6_FOLD(16);
  else MF6_FOLD(32);
#undef MF6_FOLD
}

// iterations of one graph (even); 4 and 16 cost 0.8 to 3 % more a step (3x100x100 5.71 ms
// with 8, 5.88 with 4, 5.82 with 16; 12x150x150 17.25, 17.40, 17.69)
constexpr int FOLD_ITERS = 8;

bool fold_graph(Mf6Handle *h, const FoldGrid &g) {
  if (h->cg_graph) return true;
  if (h->cg_graph_failed) return false;
  hipStream_t s = h->stream;
  hipGraph_t gr = nullptr;
  bool ok = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) == hipSuccess;
  if (ok) {
    enqueue_fold(h, g, FOLD_ITERS);
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

}  // namespace

// Whether the folded CG takes a handle's FP64 CG solves: one-level
// preconditioner, at most FOLD_MAXCOL columns (one wave per SIMD and colour)
// and partials that every block can add.  Up to that many columns the folded
// iteration takes 0.4 to 0.7 of the fused one's time; above it the sweeps need
// a second wave per SIMD, which their registers do not leave room for, and the
// two meet (10 x 420 x 420: 96 against 104 us; 10 x 500 x 500: 120 and 122),
// while the fused kernels' grouped accesses move fewer bytes.
constexpr int FOLD_MAXCOL = 1 << 17;
bool mf6hip_fold_takes(const Mf6Handle *h) {
  return h->s.preconditioner == 0 && 2 * h->L.HP0 <= FOLD_MAXCOL &&
         fold_grid(h->L).nq <= C_MAXPART;
}

// FP64 CG on the device system: d = b - A x in h->d and l2norm0 in the state
// on entry, A symmetric.  Graphs of eight iterations (kernel nodes only) are
// replayed; with the per-launch timing the kernels are enqueued one by one.
int mf6hip_run_cg_fold(Mf6Handle *h) {
  const Layout &L = h->L;
  hipStream_t s = h->stream;
  const FoldGrid g = fold_grid(L);
  static_assert(5 * C_MAXPART <= 7 * MF6_MAXBLK && 4 * C_MAXPART <= 4 * MF6_MAXBLK,
                "partials fit their arrays");
  CState *cs = reinterpret_cast<CState *>(h->d_state + 2);
  HIPCHK(hipMemsetAsync(cs, 0, sizeof(CState), s));
  HIPCHK(hipMemsetAsync(h->q, 0, sizeof(double) * L.NP, s));
  h->h_fold->stop = 0;   // nothing of an earlier solve is still running
  const bool graph = !h->timing && fold_graph(h, g);
  CK(fold_batches(h, FOLD_ITERS, [&]() -> int {
    if (graph) {
      HIPCHK(hipGraphLaunch(h->cg_graph, s));
      return MF6HIP_OK;
    }
    for (int r = 0; r < FOLD_ITERS; r += 2) {
      hipEvent_t e0 = nullptr, e1 = nullptr;
      if (h->timing && (h->spmv_calls % h->spmv_sample) < 2 &&
          2 * (h->last_spmv_n + 1) <= (int)h->spmv_ev.size()) {
        const int slot = h->last_spmv_n++;
        e0 = h->spmv_ev[2 * slot];
        e1 = h->spmv_ev[2 * slot + 1];
      }
      h->spmv_calls += 2;
      enqueue_fold(h, g, 2, e0, e1);
    }
    HIPCHK(hipGetLastError());
    return MF6HIP_OK;
  }));
  h->h_state[0] = h->h_fold->st;
  return MF6HIP_OK;
}
