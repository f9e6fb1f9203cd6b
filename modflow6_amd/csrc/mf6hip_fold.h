// mf6hip_fold.h -- pieces shared by the latency-bound Krylov kernels
// (mf6hip_cgfold.hip, mf6hip_bcgsfold.hip): wave and block reductions, the sum
// of partials that every block adds in the same order, column geometry.
#pragma once
#include "mf6hip_handle.h"

#define DPREC_C 2.220446049250313080847263336181640625e-16
#define DSAME_C (100.0 * DPREC_C)

namespace {

constexpr int C_CH = 4;          // layers whose loads are issued together
constexpr int C_MAXPART = 4096;  // partial slots per quantity

// Wave reductions on DPP moves and the row swaps of gfx950 (a butterfly of
// shuffles through LDS takes about four times as long, and a kernel here has
// two or three of them in a row).  Every lane gets the same bits.
template <int CTRL>
__device__ inline double dpp64(double v) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, CTRL, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// lanes exchanged within rows of 16: xor 1, xor 2, then mirrored halves and rows
constexpr int DPP_X1 = 0xb1, DPP_X2 = 0x4e, DPP_HMIRROR = 0x141, DPP_MIRROR = 0x140;

// {a, b}: the values of a row (ROW16) or half wave and of its partner, in the
// same order in both
template <bool ROW16>
__device__ inline void swap32(unsigned v, unsigned &a, unsigned &b) {
  const auto r = ROW16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                       : __builtin_amdgcn_permlane32_swap(v, v, false, false);
  a = r[0];
  b = r[1];
}
template <bool ROW16>
__device__ inline void swap64(double v, double &a, double &b) {
  const unsigned long long u = __double_as_longlong(v);
  unsigned al, bl, ah, bh;
  swap32<ROW16>((unsigned)u, al, bl);
  swap32<ROW16>((unsigned)(u >> 32), ah, bh);
  a = __longlong_as_double((long long)(((unsigned long long)ah << 32) | al));
  b = __longlong_as_double((long long)(((unsigned long long)bh << 32) | bl));
}

__device__ inline double csum(double v) {
  v = v + dpp64<DPP_X1>(v);
  v = v + dpp64<DPP_X2>(v);
  v = v + dpp64<DPP_HMIRROR>(v);
  v = v + dpp64<DPP_MIRROR>(v);
  double a, b;
  swap64<true>(v, a, b);
  v = a + b;
  swap64<false>(v, a, b);
  return a + b;
}

template <int CTRL>
__device__ inline MaxLoc cmax_dpp(MaxLoc v) {
  return maxloc_pick(v, MaxLoc{dpp64<CTRL>(v.v),
                               __builtin_amdgcn_mov_dpp(v.loc, CTRL, 0xf, 0xf, true)});
}
template <bool ROW16>
__device__ inline MaxLoc cmax_swap(MaxLoc v) {
  MaxLoc a, b;
  unsigned la, lb;
  swap64<ROW16>(v.v, a.v, b.v);
  swap32<ROW16>((unsigned)v.loc, la, lb);
  a.loc = (int)la;
  b.loc = (int)lb;
  return maxloc_pick(a, b);
}

__device__ inline MaxLoc cmax(MaxLoc v) {
  v = cmax_dpp<DPP_X1>(v);
  v = cmax_dpp<DPP_X2>(v);
  v = cmax_dpp<DPP_HMIRROR>(v);
  v = cmax_dpp<DPP_MIRROR>(v);
  v = cmax_swap<true>(v);
  return cmax_swap<false>(v);
}

// sum over the block, in every thread; lds is used by nothing else
template <int BS>
__device__ inline double call_sum(double v, double *lds) {
  v = csum(v);
  if (BS == 64) return v;
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < BS / 64; i++) s = s + lds[i];
  return s;
}

template <int BS>
__device__ inline MaxLoc call_max(MaxLoc v, MaxLoc *lds) {
  v = cmax(v);
  if (BS == 64) return v;
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  MaxLoc s{0.0, -1};
#pragma unroll
  for (int i = 0; i < BS / 64; i++) s = maxloc_pick(s, lds[i]);
  return s;
}

// This thread's share of n partials, at most NI BS of them: every load is
// issued before the first is waited for (a loop of n trips waits for each).
template <int BS, int NI>
__device__ inline double cpart(const double *__restrict__ part, int n) {
  double v[NI], s = 0.0;
#pragma unroll
  for (int u = 0; u < NI; u++) {
    const int i = threadIdx.x + u * BS;
    v[u] = part[i < n ? i : n - 1];
  }
#pragma unroll
  for (int u = 0; u < NI; u++) s = (int)threadIdx.x + u * BS < n ? s + v[u] : s;
  return s;
}

template <int BS, int NI>
__device__ inline MaxLoc cmpart(const MaxLoc *__restrict__ part, int n) {
  MaxLoc v[NI], s{0.0, -1};
#pragma unroll
  for (int u = 0; u < NI; u++) {
    const int i = threadIdx.x + u * BS;
    v[u] = part[i < n ? i : n - 1];
  }
#pragma unroll
  for (int u = 0; u < NI; u++)
    if ((int)threadIdx.x + u * BS < n) s = maxloc_pick(s, v[u]);
  return s;
}

// logical block of a grid of G (XCD-contiguous ranges, as xcd_block)
__device__ inline int cblock(int b, int G) {
  const int x = b & 7, m = b >> 3, q = G >> 3, r = G & 7;
  return x * q + (x < r ? x : r) + m;
}

// neighbours of a column in the other colour's plane (0 and false off grid)
struct CGeo {
  int l, ib, il, ir, ifr;
  bool hb, hl, hr, hf;
  __device__ CGeo(const Layout &L, int c, int h2) {
    l = col_l(L, c, h2);
    const int i = l / L.ncol, j = l - i * L.ncol;
    hb = i > 0;
    hl = j > 0;
    hr = j < L.ncol - 1;
    hf = i < L.nrow - 1;
    ib = hb ? hn(l, -L.ncol) : 0;
    il = hl ? hn(l, -1) : 0;
    ir = hr ? hn(l, 1) : 0;
    ifr = hf ? hn(l, L.ncol) : 0;
  }
};

__device__ inline int c_close(double a, double b) {
  if (a == b) return 1;
  return fabs(a - b) <= fmax(DSAME_C * fmax(fabs(a), fabs(b)), 0.0);
}

// ims_base_testcnvg (ImsLinearBase.f90:1101-1146)
__device__ inline void c_testcnvg(int o, int *icnvg, int it, double dvmax, double rmax,
                                  double rmax0, double epfact, double dvclose, double rclose) {
  if (o == 0) {
    if (fabs(dvmax) <= dvclose && fabs(rmax) <= rclose) *icnvg = 1;
  } else if (o == 1) {
    if (fabs(dvmax) <= dvclose && fabs(rmax) <= rclose) *icnvg = it == 1 ? 1 : -1;
  } else if (o == 2) {
    if (fabs(dvmax) <= dvclose || rmax <= rclose) *icnvg = 1;
    else if (rmax <= rmax0 * epfact) *icnvg = -1;
  } else if (o == 3) {
    if (fabs(dvmax) <= dvclose) *icnvg = 1;
    else if (rmax <= rmax0 * rclose) *icnvg = -1;
  } else if (o == 4) {
    if (fabs(dvmax) <= dvclose && rmax <= rclose) *icnvg = 1;
    else if (rmax <= rmax0 * epfact) *icnvg = -1;
  }
}

// What a solve leaves in pinned host memory when its test stops it: the host
// needs no copy to see it, only the end of the batch that holds the test.
__device__ inline void c_publish(FoldHost *hf, const KState *st, int stop) {
  hf->st = *st;
  hf->st.stop = stop;
  __threadfence_system();
  __hip_atomic_store(&hf->stop, stop, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Batches of a folded solve: `launch` enqueues one graph (or its iterations) of
// `iters` iterations.  The first two batches, up to eight iterations, are waited for
// alone, since many solves end there (an outer loop's last ones take an iteration
// or two: CG at 1x362x362 391 us with a batch queued behind the first, 297 alone,
// BiCGSTAB at 5x500x500 475 and 415, one iteration each); then one batch is queued ahead of the one the host waits for.
// A batch is one graph, from 1024 iterations on four: its end costs the GPU a few us,
// an iteration after the stop 2 us per kernel.  (Growing from 64 iterations on, 2, 4, 8
// graphs, took 5.71 ms a step for 5.52 at 3x100x100 and 17.25 for 16.96 at 12x150x150;
// never growing 157.8 for 157.3 at 10x500x500, with well over a thousand iterations.)
template <typename F>
int fold_batches(Mf6Handle *h, int iters, F launch) {
  FoldHost *hf = h->h_fold;
  int done = 0;
  auto batch = [&](int b) -> int {
    const int n = done < 1024 ? 1 : 4;
    for (int r = 0; r < n; r++) {
      const int rc = launch();
      if (rc != MF6HIP_OK) return rc;
    }
    done += n * iters;
    HIPCHK(hipEventRecord(h->ev_batch[b], h->stream));
    return MF6HIP_OK;
  };
  int rc = MF6HIP_OK;
  for (int k = 0; k < 2 && done < 8; k++) {
    rc = batch(0);
    if (rc != MF6HIP_OK) return rc;
    HIPCHK(hipEventSynchronize(h->ev_batch[0]));
    if (__atomic_load_n(&hf->stop, __ATOMIC_ACQUIRE) != 0) return MF6HIP_OK;
  }
  rc = batch(0);
  for (int b = 0; rc == MF6HIP_OK; b ^= 1) {
    rc = batch(b ^ 1);
    if (rc != MF6HIP_OK) break;
    HIPCHK(hipEventSynchronize(h->ev_batch[b]));
    if (__atomic_load_n(&hf->stop, __ATOMIC_ACQUIRE) != 0) break;
  }
  return rc;
}

}  // namespace
