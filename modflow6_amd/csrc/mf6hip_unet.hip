// mf6hip_unet.hip -- the learned preconditioner network on gfx950: a 4-level
// 3D U-Net (channels c0..c3, 1x2x2 pooling, nearest 1x2x2 upsampling,
// concatenated skips, ReLU, 1x1x1 output convolution) with BF16 weights and
// activations and FP32 accumulation on MFMA (v_mfma_f32_16x16x32_bf16),
// hand-written forward and backward kernels, and an Adam optimiser.
//
// The network has no counterpart in the reference.  Tensors are
// channels-last: voxel v = (d * H + h) * W + w of a (D, H, W) grid, then the
// channel; a tensor slice is (pointer, ld = channel stride, off = first
// channel).  Every channel count the MFMA kernels see is a multiple of 16
// (the 3 input features are padded to 16 zero channels).
//
// 3x3x3 convolution as an implicit GEMM on v_mfma_f32_16x16x32_bf16: a
// workgroup stages the input halo of its voxel tile in LDS, a channel chunk
// at a time, and each wave multiplies MT rows of 16 voxels by the packed
// weights (see k_conv3).
//
// The backward pass reuses the same kernel for the data gradient (weights
// flipped in the tap index and transposed in the channels), an MFMA
// weight- and bias-gradient kernel with split-K partials reduced in a fixed
// order, and elementwise kernels for ReLU masks, pooling, upsampling and the skips.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "mf6hip_handle.h"

namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16;

#define UCK(x)                        \
  do {                                \
    int rc_ = (x);                    \
    if (rc_ != MF6HIP_OK) return rc_; \
  } while (0)

// round to nearest even FP32 -> BF16 (finite inputs)
__host__ __device__ inline bf16 f2bf(float f) {
  unsigned u;
  memcpy(&u, &f, 4);
  unsigned r = u + 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(r >> 16);
}
__host__ __device__ inline float bf2f(bf16 b) {
  unsigned u = ((unsigned)b) << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

struct Grid3 {
  int D, H, W;
  __host__ __device__ int V() const { return D * H * W; }
};

// ---------------------------------------------------------------------------
// 3x3x3 convolution (forward and data gradient)
// ---------------------------------------------------------------------------

// y[v, o] = act(bias[o] + sum_{t, c} x[v + off(t), c] W[t, c, o])
// act: relu when relu != 0; then y *= (mask[v, o] > 0) when mask != 0.
//
// A workgroup of four waves computes WD x (4 / WD) MT x 16 voxels (d, h, w)
// by NC tiles of 16 output channels (blockIdx.y takes the next NC tiles).
// Per chunk of CW input channels the input halo, (WD + 2) x (TH + 2) x 18
// voxels, is staged once in LDS, so a value read from memory serves all 27
// taps; a wave then walks the (kd, kw) pairs of the taps and, per pair, loads
// the MT + 2 input rows its MT output rows need and reuses them for the three
// kh (each row feeds up to three MFMAs per output tile instead of one).
// K of one MFMA is 32: a chunk of 32 channels of one (kd, kw) for CW = 32,
// two (kd, kw) pairs of 16 channels for CW = 16 (cin not a multiple of 32).
// The weights are the A operand (lane l: output channel l % 16, k = 8 (l /
// 16) .. +7), the voxels the B operand, so a lane ends up with four
// consecutive output channels of one voxel and stores them as 8 bytes.
// LDS: the 16-byte pieces of a voxel are permuted by its w so that the 16
// voxels of a row read by one quarter of the wave fall in different banks.
// The first version (one wave per 16 voxels, activations and weights loaded
// per tap from L2, K = 16) was bound by those loads.  On a 16 x 256 x 256
// field the level-0 convolutions of the 16-32-64-64 network went from 228 to
// 56 us each on average, those of level 1 from 160 to 57, and the whole
// forward pass's convolutions from 112 to about 430 TFLOP/s.
template <int CW>
struct ConvGeo {
  static constexpr int PIECES = CW / 8;                 // 16-byte pieces per voxel
  static constexpr int STEPS = CW == 32 ? 9 : 5;        // MFMA steps over the (kd, kw) pairs
  static constexpr int VB = CW * 2;                     // bytes per voxel
  // byte offset in a voxel of piece q of the voxel at halo column pw
  __device__ static int piece(int q, int pw) {
    return CW == 32 ? ((q ^ ((pw >> 2) & 3)) << 4) : ((q ^ ((pw >> 3) & 1)) << 4);
  }
};

// Input of a convolution: the channels of x (stride ldx), preceded for a
// decoder by the cu channels of a coarse tensor on the 1 x 2 x 2 coarser grid
// (rows Hc, columns Wc), upsampled to the nearest fine voxel as they are
// read.  (Writing the upsampled channels out first cost 47 us per decoder
// level at 16 x 256 x 256 and as much again to read them back.)
struct ConvSrc {
  const bf16 *x;
  int ldx;
  const bf16 *up = nullptr;
  int cu = 0, Hc = 0, Wc = 0;
};

// the halo of channels c0 .. c0 + CW - 1 of the tile at (d0, h0, w0) into
// LDS, zero outside the grid; PD x PH x 18 voxels, mph = ceil(2^16 / PH)
template <int CW>
__device__ inline void stage_halo(char *lds, const Grid3 &g, const ConvSrc &src, int c0, int d0,
                                  int h0, int w0, int PD, int PH, int mph) {
  constexpr int P = ConvGeo<CW>::PIECES;
  const int n = PD * PH * 18 * P;
  for (int i = threadIdx.x; i < n; i += 256) {
    const int q = i & (P - 1), vox = i / P;
    const int row = vox / 18, pw = vox - row * 18;
    const int pd = (row * mph) >> 16, ph = row - pd * PH;
    const int d = d0 + pd - 1, h = h0 + ph - 1, w = w0 + pw - 1;
    s8 v = s8{0, 0, 0, 0, 0, 0, 0, 0};
    if (d >= 0 && d < g.D && h >= 0 && h < g.H && w >= 0 && w < g.W) {
      const int c = c0 + 8 * q;
      const bf16 *p = c < src.cu
          ? src.up + (size_t)((d * src.Hc + (h >> 1)) * src.Wc + (w >> 1)) * src.cu + c
          : src.x + (size_t)((d * g.H + h) * g.W + w) * src.ldx + (c - src.cu);
      v = *reinterpret_cast<const s8 *>(p);
    }
    *reinterpret_cast<s8 *>(lds + vox * ConvGeo<CW>::VB + ConvGeo<CW>::piece(q, pw)) = v;
  }
}

// 1x1x1 output convolution computed with the last decoder convolution (16
// channels, from its stored BF16 values): yo[v] = sum_c y[v, c] wo[c] + bo
struct ConvOut1 {
  const float *wo = nullptr, *bo = nullptr;
  float *yo = nullptr;
};

template <int CW, int MT, int NC>
__global__ void __launch_bounds__(256) k_conv3(Grid3 g, ConvSrc src, int cin,
                                               const s8 *__restrict__ wp, int nco,
                                               const float *__restrict__ bias, int relu,
                                               bf16 *__restrict__ y, int ldy,
                                               const bf16 *__restrict__ mask, int ldm,
                                               ConvOut1 o1, int WD, int mph) {
  extern __shared__ char lds[];
  using G = ConvGeo<CW>;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int WH = 4 / WD;
  const int TH = WH * MT, PD = WD + 2, PH = TH + 2;
  const int ntw = (g.W + 15) >> 4, nth = (g.H + TH - 1) / TH;
  const int tile = xcd_block();
  const int w0 = (tile % ntw) << 4, h0 = (tile / ntw) % nth * TH, d0 = tile / (ntw * nth) * WD;
  const int wd = wv % WD, wh = wv / WD;
  const int lw = lane & 15, kq = lane >> 4;
  const int ct0 = blockIdx.y * NC;             // first output-channel tile
  f4 acc[MT][NC];
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[m][c] = f4{0.f, 0.f, 0.f, 0.f};
  const int rowb = 18 * G::VB, planeb = PH * rowb;
  const int base = wd * planeb + wh * MT * rowb;
  // fragments of output tile ct0 + c (a tile past the last reads the last's)
  const s8 *wt[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) {
    const int ct = ct0 + c < nco ? ct0 + c : nco - 1;
    wt[c] = wp + (size_t)ct * (cin / CW) * G::STEPS * 3 * 64;
  }
  for (int c0 = 0; c0 < cin; c0 += CW) {
    if (c0) __syncthreads();
    stage_halo<CW>(lds, g, src, c0, d0, h0, w0, PD, PH, mph);
    __syncthreads();
    // the weights of a step are loaded while the step before it runs
    b8 wn[3][NC];
#pragma unroll
    for (int kh = 0; kh < 3; kh++)
#pragma unroll
      for (int c = 0; c < NC; c++) wn[kh][c] = *reinterpret_cast<const b8 *>(wt[c] + kh * 64 + lane);
#pragma unroll
    for (int s = 0; s < G::STEPS; s++) {
      b8 w[3][NC];
#pragma unroll
      for (int kh = 0; kh < 3; kh++)
#pragma unroll
        for (int c = 0; c < NC; c++) {
          w[kh][c] = wn[kh][c];
          if (s + 1 < G::STEPS)
            wn[kh][c] = *reinterpret_cast<const b8 *>(wt[c] + ((s + 1) * 3 + kh) * 64 + lane);
        }
      // this lane's (kd, kw) pair and 16-byte piece
      int off, pw;
      if (CW == 32) {
        pw = lw + s % 3;
        off = (s / 3) * planeb + pw * G::VB + G::piece(kq, pw);
      } else {
        const int qa = 2 * s, qb = 2 * s + 1 < 9 ? 2 * s + 1 : qa;
        const bool hi = kq >= 2;
        pw = lw + (hi ? qb % 3 : qa % 3);
        off = (hi ? qb / 3 : qa / 3) * planeb + pw * G::VB + G::piece(kq & 1, pw);
      }
      b8 a[MT + 2];
#pragma unroll
      for (int r = 0; r < MT + 2; r++) {
        a[r] = *reinterpret_cast<const b8 *>(lds + base + off + r * rowb);
        if (CW == 16 && s == G::STEPS - 1 && kq >= 2) a[r] = b8{};   // no tenth pair
      }
#pragma unroll
      for (int kh = 0; kh < 3; kh++)
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
          for (int c = 0; c < NC; c++)
            acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[kh][c], a[m + kh], acc[m][c], 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < NC; c++) wt[c] += G::STEPS * 3 * 64;
  }
  const int d = d0 + wd, w = w0 + lw;
  if (d >= g.D || w >= g.W) return;
#pragma unroll
  for (int m = 0; m < MT; m++) {
    const int h = h0 + wh * MT + m;
    if (h >= g.H) break;
    const size_t v = (size_t)(d * g.H + h) * g.W + w;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      if (ct0 + c >= nco) break;
      const int o = (ct0 + c) * 16 + 4 * kq;
      s4 mk = s4{0, 0, 0, 0}, out;
      if (mask) mk = *reinterpret_cast<const s4 *>(mask + v * ldm + o);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float val = acc[m][c][e] + (bias ? bias[o + e] : 0.f);
        if (relu && val < 0.f) val = 0.f;
        if (mask && !(bf2f((bf16)mk[e]) > 0.f)) val = 0.f;
        out[e] = (short)f2bf(val);
      }
      *reinterpret_cast<s4 *>(y + v * ldy + o) = out;
      if (o1.yo) {
        // the four lanes of a voxel hold its 16 channels
        float t = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) t = t + bf2f((bf16)out[e]) * o1.wo[o + e];
        t = t + __shfl_xor(t, 16);
        t = t + __shfl_xor(t, 32);
        if (kq == 0) o1.yo[v] = t + o1.bo[0];
      }
    }
  }
}

// chunk width of a convolution with ci input channels
__host__ __device__ inline int conv_cw(int ci) { return ci % 32 == 0 ? 32 : 16; }

// 16-byte weight fragments of a convolution: [output tile][chunk][step][kh][lane]
__host__ __device__ inline int conv_nfrag(int ci, int co) {
  const int cw = conv_cw(ci);
  return (ci / cw) * (cw == 32 ? 9 : 5) * 3 * (co >> 4) * 64;
}

// pack W (fp32 [27][cin_real][cout]) into the fragments of k_conv3 for a
// cin-channel input (rows cin_real..cin-1 zero); flip != 0 packs the
// data-gradient weights Wt[t][o][c] = W[26 - t][c][o] (input / output
// swapped; cin_real == cin)
//
// All layers and directions of a network in one launch (job q on blocks j[q].b0
// up to the next job's): a launch each, up to 45 of them after every Adam step, took
// 4.2 us and the gap before it.
constexpr int MAXLEV = 8;
constexpr int MAXCONV = 3 * MAXLEV - 1;
struct PackJob {
  const float *w;
  s8 *wp;
  int cin_real, cin, cout, flip, b0;
};
struct PackJobs {
  int n, nblk;
  PackJob j[2 * MAXCONV];
};

__global__ void __launch_bounds__(256) k_pack_w(PackJobs jobs) {
  int q = 0;
  while (q + 1 < jobs.n && (int)blockIdx.x >= jobs.j[q + 1].b0) q++;
  const float *__restrict__ w = jobs.j[q].w;
  s8 *__restrict__ wp = jobs.j[q].wp;
  const int cin_real = jobs.j[q].cin_real, cin = jobs.j[q].cin, cout = jobs.j[q].cout;
  const int flip = jobs.j[q].flip;
  const int ci = flip ? cout : cin;   // fragment input channels
  const int co = flip ? cin : cout;   // fragment output channels
  const int cw = conv_cw(ci), steps = cw == 32 ? 9 : 5;
  const int total = conv_nfrag(ci, co);
  const int i = ((int)blockIdx.x - jobs.j[q].b0) * 256 + threadIdx.x;
  if (i < total) {
    const int lane = i & 63, kq = lane >> 4;
    int r = i >> 6;
    const int kh = r % 3;
    r /= 3;
    const int s = r % steps;
    r /= steps;
    const int cc = r % (ci / cw), c = r / (ci / cw);
    const int pair = cw == 32 ? s : 2 * s + (kq >> 1);           // kd 3 + kw
    const int kin0 = cc * cw + (cw == 32 ? 8 * kq : 8 * (kq & 1));
    const int kout = c * 16 + (lane & 15);
    const int t = (pair / 3) * 9 + kh * 3 + pair % 3;
    s8 v;
    for (int e = 0; e < 8; e++) {
      const int kin = kin0 + e;
      float f = 0.f;
      if (pair < 9) {
        if (flip) f = w[((size_t)(26 - t) * cin_real + kout) * cout + kin];
        else f = kin < cin_real ? w[((size_t)t * cin_real + kin) * cout + kout] : 0.f;
      }
      v[e] = (short)f2bf(f);
    }
    wp[i] = v;
  }
}

// ---------------------------------------------------------------------------
// weight gradient: dW[t][c][o] = sum_v x[v + off(t), c] dy[v, o]
// ---------------------------------------------------------------------------

// and the bias gradient db[o] = sum_v dy[v, o].
//
// A GEMM over the voxels: M = output channels, N = input channels, K = the
// voxels, once per tap.  Workgroup (split, 16 input channels, NC tiles of 16
// output channels) walks its share of the voxel tiles (TD x TH x 16, 256
// voxels), stages the tile's x halo and dy in LDS (channels last, as they lie
// in memory) and keeps all 27 taps' accumulators in registers: wave j takes
// taps j, j + 4, ... (28 with the bias, whose x is all ones), so every staged
// value serves all taps and output tiles.  The MFMA operands need eight
// consecutive voxels of one channel per lane; ds_read_b64_tr_b16 transposes
// four voxels x 16 channels on the way out of LDS (lane i of a quarter wave
// gives the address of voxel i / 4, channels 4 (i % 4) .., and receives
// channel i of the four voxels), so a tap's shift is only an address offset.
// Partials go to part[split] ([27][cin][cout], then [cout]) and are summed
// in split order by k_wgrad_reduce.  The first version (one tap and one 16 x
// 16 tile per workgroup, voxels gathered two bytes at a time) re-read x and
// dy 27 times: over a training step's layers (16 x 256 x 256, 16-32-64-64)
// 630 us each on average, now 51 (the level-0 ones 87, which LDS reads
// bound: seven transposed x reads serve only one output tile), and its own
// bias-gradient kernels are gone.
constexpr int WG_MAXBLK = 512;   // workgroups of one layer's gradient
template <int NC>
__global__ void __launch_bounds__(256, 2) k_wgrad(Grid3 g, ConvSrc src, int cin,
                                                  const bf16 *__restrict__ dy, int cout, int TD,
                                                  int mph, float *__restrict__ part) {
  extern __shared__ char lds[];
  const int TH = 16 / TD, PD = TD + 2, PH = TH + 2;
  char *ldy = lds + PD * PH * 18 * 32;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int kq = lane >> 4, li = lane & 15;
  const int nco = cout >> 4, ncc = cin >> 4;
  const int ct = blockIdx.y % ncc, ot0 = blockIdx.y / ncc * NC;
  const int ntw = (g.W + 15) >> 4, nth = (g.H + TH - 1) / TH, ntd = (g.D + TD - 1) / TD;
  const int ntiles = ntw * nth * ntd;
  const int rowb = 18 * 32, planeb = PH * rowb;
  // LDS offsets of this lane's two transposed reads (voxels +0..3, +4..7 of
  // its eight) for each of the wave's taps, relative to the tile row pair
  int off[7][2];
#pragma unroll
  for (int q = 0; q < 7; q++) {
    const int t = wv + 4 * q < 27 ? wv + 4 * q : 26;
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int pw = t % 3 + 8 * (kq & 1) + 4 * u + (li >> 2);
      off[q][u] = (t / 9) * planeb + ((t / 3) % 3 + (kq >> 1)) * rowb + pw * 32 +
                  ConvGeo<16>::piece((li & 3) >> 1, pw) + (li & 1) * 8;
    }
  }
  const int offd = (16 * (kq >> 1) + 8 * (kq & 1) + (li >> 2)) * NC * 32 + (li & 3) * 8;
  const short one = (short)0x3f80;
  f4 acc[7][NC];
#pragma unroll
  for (int q = 0; q < 7; q++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[q][c] = f4{0.f, 0.f, 0.f, 0.f};
  typedef __attribute__((address_space(3))) s4 *lp4;
  auto tr8 = [](const char *p0, const char *p1) {
    const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp4)p0);
    const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp4)p1);
    const s8 v = s8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(b8, v);
  };
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int w0 = (tile % ntw) << 4, h0 = (tile / ntw) % nth * TH, d0 = tile / (ntw * nth) * TD;
    __syncthreads();
    stage_halo<16>(lds, g, src, ct * 16, d0, h0, w0, PD, PH, mph);
    for (int i = threadIdx.x; i < 256 * NC * 2; i += 256) {
      const int q = i % (NC * 2), vox = i / (NC * 2);
      const int w = w0 + (vox & 15), row = vox >> 4;
      const int h = h0 + row % TH, d = d0 + row / TH;
      s8 v = s8{0, 0, 0, 0, 0, 0, 0, 0};
      if (d < g.D && h < g.H && w < g.W && ot0 + q / 2 < nco)
        v = *reinterpret_cast<const s8 *>(dy + (size_t)((d * g.H + h) * g.W + w) * cout +
                                          ot0 * 16 + 8 * q);
      *reinterpret_cast<s8 *>(ldy + vox * NC * 32 + q * 16) = v;
    }
    __syncthreads();
    // K = 32 voxels a step: rows (dl, hl) and (dl, hl + 1)
    for (int st = 0; st < 8; st++) {
      const int dl = 2 * st / TH, hl = 2 * st % TH;
      const char *xr = lds + dl * planeb + hl * rowb;
      const char *dr = ldy + st * 32 * NC * 32 + offd;
      b8 fd[NC];
#pragma unroll
      for (int c = 0; c < NC; c++) fd[c] = tr8(dr + c * 32, dr + c * 32 + 4 * NC * 32);
#pragma unroll
      for (int q = 0; q < 7; q++) {
        b8 fx = tr8(xr + off[q][0], xr + off[q][1]);
        if (q == 6 && wv == 3)
          fx = __builtin_bit_cast(b8, s8{one, one, one, one, one, one, one, one});
#pragma unroll
        for (int c = 0; c < NC; c++)
          acc[q][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fd[c], fx, acc[q][c], 0, 0, 0);
      }
    }
  }
  // lane: input channel li, output channels 4 kq .. + 3 of each tile
  float *pt = part + (size_t)blockIdx.x * ((size_t)27 * cin + 1) * cout;
#pragma unroll
  for (int q = 0; q < 7; q++) {
    const int t = wv + 4 * q;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      if (ot0 + c >= nco) break;
      const int o = (ot0 + c) * 16 + 4 * kq;
      if (t < 27)
        *reinterpret_cast<f4 *>(pt + ((size_t)t * cin + ct * 16 + li) * cout + o) = acc[q][c];
      else if (ct == 0 && li == 0)
        *reinterpret_cast<f4 *>(pt + (size_t)27 * cin * cout + o) = acc[q][c];
    }
  }
}

// Gradient of a layer's weights and biases (adjacent in the parameter
// vector): grad[i] (+)= sum over the splits' partials in split order, the
// rows cin_real .. cin - 1 of a padded input left out.  Four waves take a
// quarter of the splits each for 64 values, so the loads of a value's many
// partials run in parallel; the quarters are added in order.
__global__ void __launch_bounds__(256) k_wgrad_reduce(const float *__restrict__ part, int nsplit,
                                                      int cin, int cin_real, int cout,
                                                      float *__restrict__ grad, int accumulate) {
  __shared__ float red[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int nw = 27 * cin_real * cout, n = nw + cout;
  const size_t stride = ((size_t)27 * cin + 1) * cout;
  const int i = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (i < n) {
    int e = i;
    if (i >= nw) e = 27 * cin * cout + (i - nw);
    else if (cin_real != cin) {
      const int t = i / (cin_real * cout);
      e = t * cin * cout + (i - t * cin_real * cout);
    }
    const int k0 = (int)((long long)nsplit * wv / 4), k1 = (int)((long long)nsplit * (wv + 1) / 4);
#pragma unroll 8
    for (int k = k0; k < k1; k++) s = s + part[(size_t)k * stride + e];
  }
  red[wv][lane] = s;
  __syncthreads();
  if (wv != 0 || i >= n) return;
  s = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
  grad[i] = accumulate ? grad[i] + s : s;
}

// ---------------------------------------------------------------------------
// elementwise pieces
// ---------------------------------------------------------------------------

// Pooling and upsampling between a fine grid gf and its coarse grid gc with
// gc.H = ceil(gf.H / 2), gc.W = ceil(gf.W / 2): coarse cell (h, w) covers the
// fine cells (2h + a, 2w + b), a, b in {0, 1}, that exist (1, 2 or 4 cells
// on the last row / column of an odd extent).
__device__ __forceinline__ int pool_count(const Grid3 &gf, int hc, int wc) {
  const int nh = (2 * hc + 1 < gf.H) ? 2 : 1, nw = (2 * wc + 1 < gf.W) ? 2 : 1;
  return nh * nw;
}

// The elementwise kernels below take eight channels (16 bytes) per thread;
// C, strides and offsets are multiples of 16.
__device__ __forceinline__ s8 ld8(const bf16 *p) { return *reinterpret_cast<const s8 *>(p); }

// sum over the fine cells of coarse cell (d, h, w) of x[.., c .. c + 7]
__device__ __forceinline__ void fine_sum8(const Grid3 &gf, const bf16 *__restrict__ x, int ldx,
                                          int d, int h, int w, int c, float *s) {
  const bool hr = 2 * h + 1 < gf.H, wr = 2 * w + 1 < gf.W;
  const bf16 *p = x + ((size_t)(d * gf.H + 2 * h) * gf.W + 2 * w) * ldx + c;
  const s8 z = s8{0, 0, 0, 0, 0, 0, 0, 0};
  const s8 a = ld8(p), b = wr ? ld8(p + ldx) : z;
  const s8 e = hr ? ld8(p + (size_t)gf.W * ldx) : z, f = hr && wr ? ld8(p + (size_t)(gf.W + 1) * ldx) : z;
#pragma unroll
  for (int q = 0; q < 8; q++)
    s[q] = (bf2f((bf16)a[q]) + bf2f((bf16)b[q])) + (bf2f((bf16)e[q]) + bf2f((bf16)f[q]));
}

// pooled[v, c] = mean of the fine cells of coarse cell v; c < C
__global__ void k_pool(Grid3 gc, Grid3 gf, const bf16 *__restrict__ x, int C,
                       bf16 *__restrict__ y) {
  const int C8 = C / 8, n = gc.V() * C8;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = i % C8 * 8, v = i / C8;
    const int w = v % gc.W, h = (v / gc.W) % gc.H, d = v / (gc.W * gc.H);
    float s[8];
    fine_sum8(gf, x, C, d, h, w, c, s);
    const float cnt = (float)pool_count(gf, h, w);
    s8 o;
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = (short)f2bf(s[q] / cnt);
    *reinterpret_cast<s8 *>(y + (size_t)v * C + c) = o;
  }
}

// dx (fine grid) = add + dy (coarse) / count, the pooling gradient on top of
// the skip's (channels aoff .. of add), masked by (mask > 0)
__global__ void k_pool_bwd(Grid3 gf, Grid3 gc, const bf16 *__restrict__ dy, int C,
                           const bf16 *__restrict__ add, int lda, int aoff,
                           const bf16 *__restrict__ mask, bf16 *__restrict__ dx) {
  const int C8 = C / 8, n = gf.V() * C8;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = i % C8 * 8, v = i / C8;
    const int w = v % gf.W, h = (v / gf.W) % gf.H, d = v / (gf.W * gf.H);
    const size_t vc = (size_t)(d * gc.H + h / 2) * gc.W + w / 2;
    const float cnt = (float)pool_count(gf, h / 2, w / 2);
    const s8 g = ld8(dy + vc * C + c), a = ld8(add + (size_t)v * lda + aoff + c);
    const s8 m = ld8(mask + (size_t)v * C + c);
    s8 o;
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const float t = bf2f((bf16)a[q]) + bf2f((bf16)g[q]) / cnt;
      o[q] = (short)f2bf(bf2f((bf16)m[q]) > 0.f ? t : 0.f);
    }
    *reinterpret_cast<s8 *>(dx + (size_t)v * C + c) = o;
  }
}

// coarse gradient of the upsampling: sum over the fine cells of the coarse
// cell (the first C of ldd channels), masked
__global__ void k_up_bwd(Grid3 gc, Grid3 gf, const bf16 *__restrict__ dy, int ldd, int C,
                         const bf16 *__restrict__ mask, bf16 *__restrict__ dx) {
  const int C8 = C / 8, n = gc.V() * C8;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int c = i % C8 * 8, v = i / C8;
    const int w = v % gc.W, h = (v / gc.W) % gc.H, d = v / (gc.W * gc.H);
    float s[8];
    fine_sum8(gf, dy, ldd, d, h, w, c, s);
    const s8 m = ld8(mask + (size_t)v * C + c);
    s8 o;
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = (short)f2bf(bf2f((bf16)m[q]) > 0.f ? s[q] : 0.f);
    *reinterpret_cast<s8 *>(dx + (size_t)v * C + c) = o;
  }
}

// loss partials: sum (y - t)^2 and sum t^2 per block
__global__ void k_loss(int V, const float *__restrict__ y, const bf16 *__restrict__ t, int ldt,
                       int toff, float *__restrict__ part) {
  __shared__ float r1[256], r2[256];
  float a = 0.f, b = 0.f;
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < V; v += gridDim.x * blockDim.x) {
    const float tv = bf2f(t[(size_t)v * ldt + toff]);
    const float d = y[v] - tv;
    a = a + d * d;
    b = b + tv * tv;
  }
  r1[threadIdx.x] = a;
  r2[threadIdx.x] = b;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      r1[threadIdx.x] = r1[threadIdx.x] + r1[threadIdx.x + s];
      r2[threadIdx.x] = r2[threadIdx.x] + r2[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r1[0];
    part[2 * blockIdx.x + 1] = r2[0];
  }
}

// one block: the sums of both columns of the nb partials (fixed order)
__global__ void __launch_bounds__(256) k_loss_final(const float *__restrict__ part, int nb,
                                                    float *__restrict__ out) {
  __shared__ float red[2][4];
  float a = 0.f, b = 0.f;
  for (int i = threadIdx.x; i < nb; i += 256) {
    a = a + part[2 * i];
    b = b + part[2 * i + 1];
  }
  for (int o = 32; o > 0; o >>= 1) {
    a = a + __shfl_xor(a, o);
    b = b + __shfl_xor(b, o);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = a;
    red[1][threadIdx.x >> 6] = b;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  a = ((red[0][0] + red[0][1]) + red[0][2]) + red[0][3];
  b = ((red[1][0] + red[1][1]) + red[1][2]) + red[1][3];
  out[0] = a / b;   // loss
  out[1] = b;       // sum t^2
}

// output-layer backward (16 channels): g = 2 (y - t) / sum t^2 ; du[v, c] =
// g wo[c] masked by u > 0 ; partials of d wo[c] = sum_v g u[v, c] and d bo =
// sum_v g, part[block * 17 + c]
__global__ void __launch_bounds__(256) k_out_bwd(int V, const float *__restrict__ y,
                                                 const bf16 *__restrict__ t, int ldt, int toff,
                                                 const float *__restrict__ lossv,
                                                 const bf16 *__restrict__ u,
                                                 const float *__restrict__ wo,
                                                 bf16 *__restrict__ du,
                                                 float *__restrict__ part) {
  __shared__ float red[4][17];
  float acc[17];
#pragma unroll
  for (int c = 0; c < 17; c++) acc[c] = 0.f;
  const float sc = 2.f / lossv[1];
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < V; v += gridDim.x * blockDim.x) {
    const float g = sc * (y[v] - bf2f(t[(size_t)v * ldt + toff]));
#pragma unroll
    for (int p = 0; p < 2; p++) {
      const s8 uv = ld8(u + (size_t)v * 16 + 8 * p);
      s8 o;
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const float x = bf2f((bf16)uv[q]);
        acc[8 * p + q] = acc[8 * p + q] + g * x;
        o[q] = (short)f2bf(x > 0.f ? g * wo[8 * p + q] : 0.f);
      }
      *reinterpret_cast<s8 *>(du + (size_t)v * 16 + 8 * p) = o;
    }
    acc[16] = acc[16] + g;
  }
#pragma unroll
  for (int c = 0; c < 17; c++) {
    for (int o = 32; o > 0; o >>= 1) acc[c] = acc[c] + __shfl_xor(acc[c], o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = acc[c];
  }
  __syncthreads();
  if (threadIdx.x < 17) {
    const int c = threadIdx.x;
    part[blockIdx.x * 17 + c] = ((red[0][c] + red[1][c]) + red[2][c]) + red[3][c];
  }
}

// sum of per-block partial rows, one block per column: out[j] (+)= sum_b
// part[b * n + j] (fixed order)
__global__ void __launch_bounds__(256) k_colsum(const float *__restrict__ part, int nb, int n,
                                                float *__restrict__ out, int accumulate) {
  __shared__ float red[4];
  const int j = blockIdx.x;
  float s = 0.f;
  for (int b = threadIdx.x; b < nb; b += 256) s = s + part[(size_t)b * n + j];
  for (int o = 32; o > 0; o >>= 1) s = s + __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x != 0) return;
  s = ((red[0] + red[1]) + red[2]) + red[3];
  out[j] = accumulate ? out[j] + s : s;
}

// Adam (bias-corrected) on fp32 master parameters; grads scaled by gscale
__global__ void k_adam(int n, float *__restrict__ p, const float *__restrict__ g,
                       float *__restrict__ m, float *__restrict__ v, float lr, float b1,
                       float b2, float eps, float c1, float c2, float gscale) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float gi = g[i] * gscale;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// network input (16 channels, one voxel per thread): channels 0..nin-1 from
// fp32 natural-order planes, rest 0
__global__ void k_make_input(int V, int nin, const float *__restrict__ src,
                             bf16 *__restrict__ x) {
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < V; v += gridDim.x * blockDim.x) {
#pragma unroll
    for (int p = 0; p < 2; p++) {
      s8 o;
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const int c = 8 * p + q;
        o[q] = c < nin ? (short)f2bf(src[(size_t)c * V + v]) : (short)0;
      }
      *reinterpret_cast<s8 *>(x + (size_t)v * 16 + 8 * p) = o;
    }
  }
}

// a training sample (bf16, [V][4]: 3 inputs + target) into the padded input
__global__ void k_expand_sample(int V, const bf16 *__restrict__ s, bf16 *__restrict__ x) {
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < V; v += gridDim.x * blockDim.x) {
    const s4 a = *reinterpret_cast<const s4 *>(s + (size_t)v * 4);
    *reinterpret_cast<s8 *>(x + (size_t)v * 16) = s8{a[0], a[1], a[2], 0, 0, 0, 0, 0};
    *reinterpret_cast<s8 *>(x + (size_t)v * 16 + 8) = s8{0, 0, 0, 0, 0, 0, 0, 0};
  }
}

__global__ void k_f32_to_bf16(int n, const float *__restrict__ a, bf16 *__restrict__ b) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    b[i] = f2bf(a[i]);
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct UConv {
  int cin, cout;        // cin as the kernels see it (padded to 16)
  int cin_real;         // parameter rows (the first layer: the real inputs)
  size_t w_off, b_off;  // offsets into the flat parameter vector
  s8 *wp = nullptr;     // forward fragments
  s8 *wt = nullptr;     // data-gradient fragments
};

// levels 0..nlev-1; conv layers in the order e0a e0b e1a e1b ... (two per
// level, encoder), then the decoder d_{nlev-2} ... d0, one per level

struct UNetHandle {
  int nin = 3;
  int nlev = 4;
  int ch[MAXLEV];
  Grid3 g[MAXLEV];
  UConv conv[MAXCONV];
  size_t wo_off, bo_off, nparam;
  float *p = nullptr, *grad = nullptr, *m = nullptr, *v = nullptr;
  // forward's and grad's inputs, grad's target as FP32 and BF16: allocated by the
  // first call that needs them and, like the activations, kept
  float *dx = nullptr, *dt32 = nullptr;
  bf16 *dt = nullptr;
  float *part = nullptr;   // split-K and block partials
  size_t part_n = 0;
  // activations (bf16) per level
  bf16 *in0 = nullptr;                 // level-0 input, 16 channels
  bf16 *pin[MAXLEV] = {};              // pooled inputs (levels 1..nlev-1)
  bf16 *ha[MAXLEV] = {};               // first conv output
  bf16 *hb[MAXLEV] = {};               // second conv output (the skips; the bottom output)
  bf16 *u[MAXLEV] = {};                // decoder outputs (levels < nlev-1)
  float *y = nullptr;                  // fp32 output
  float *lossv = nullptr;              // [2]
  // gradients
  bf16 *gu[MAXLEV] = {}, *gcat[MAXLEV] = {}, *ghb[MAXLEV] = {}, *gha[MAXLEV] = {},
       *gpin[MAXLEV] = {};
  bf16 *data = nullptr;                // training samples [nsamples][V][4]
  int nsamples = 0;
  int adam_t = 0;
  hipStream_t stream = nullptr;
  int nconv() const { return 3 * nlev - 1; }
  // decoder conv of level l (< nlev - 1)
  int dconv(int l) const { return 2 * nlev + (nlev - 2 - l); }
  // channels of the upsampled part of a decoder's input
  int cup(int l) const { return ch[l + 1]; }
  // input of level l's decoder: the coarser output upsampled, then the skip
  ConvSrc dec_src(int l) const {
    return ConvSrc{hb[l], ch[l], l == nlev - 2 ? hb[l + 1] : this->u[l + 1], ch[l + 1],
                   g[l + 1].H, g[l + 1].W};
  }
  // input of level l's first convolution
  ConvSrc enc_src(int l) const {
    return l == 0 ? ConvSrc{in0, 16} : ConvSrc{pin[l], ch[l - 1]};
  }
};

namespace {

template <typename T>
int ualloc(T **p, size_t n) {
  if (hipMalloc((void **)p, sizeof(T) * (n ? n : 1)) != hipSuccess) {
    mf6hip_set_error("hipMalloc failed (learned preconditioner)");
    return MF6HIP_EHIP;
  }
  return MF6HIP_OK;
}

inline int nblk(size_t n) {
  size_t b = (n + 255) / 256;
  if (b > 8192) b = 8192;
  return (int)(b < 1 ? 1 : b);
}

// Tile of k_conv3 for a grid: MT output rows per wave, WD waves along d and 4 /
// WD along h, NC output tiles per workgroup.  Four rows per wave where that
// leaves at least two workgroups per CU (512), else two or one, and on the
// coarsest grids one output tile per workgroup: below that, idle CUs cost
// more than the rows' and weights' reuse gains.  WD: the split that pads the
// grid least (the widest on a tie, which has the smallest halo).
struct ConvTile {
  int MT, WD, NC, tiles, gy;
};

ConvTile conv_tile(const Grid3 &g, int nco) {
  ConvTile best{};
  for (int step = 0; step < 4; step++) {
    ConvTile t{};
    t.MT = step == 0 ? 4 : step == 1 ? 2 : 1;
    t.gy = step == 3 ? nco : (nco + 3) / 4;
    t.NC = (nco + t.gy - 1) / t.gy;
    long long pad = -1;
    for (int wd = 4; wd >= 1; wd >>= 1) {
      const int th = 4 / wd * t.MT;
      const int nd = (g.D + wd - 1) / wd, nh = (g.H + th - 1) / th;
      const long long v = (long long)nd * wd * nh * th;
      if (pad < 0 || v < pad) {
        pad = v;
        t.WD = wd;
        t.tiles = nd * nh * ((g.W + 15) / 16);
      }
    }
    if (step == 0 || (long long)t.tiles * t.gy > (long long)best.tiles * best.gy) best = t;
    if ((long long)best.tiles * best.gy >= 512) break;
  }
  return best;
}

template <int CW, int MT>
void launch_conv_nc(int nc, dim3 grid, int shm, hipStream_t s, const Grid3 &g, const ConvSrc &src,
                    int cin, const s8 *wp, int nco, const float *bias, int relu, bf16 *y, int ldy,
                    const bf16 *mask, int ldm, const ConvOut1 &o1, int WD, int mph) {
#define MF6_CONV(N)                                                                             \
  k_conv3<CW, MT, N><<<grid, 256, shm, s>>>(g, src, cin, wp, nco, bias, relu, y, ldy, mask, ldm, \
                                            o1, WD, mph)
  if (nc == 1) MF6_CONV(1);
  else if (nc == 2) MF6_CONV(2);
  else if (nc == 3) MF6_CONV(3);
  else MF6_CONV(4);
#undef MF6_CONV
}

int launch_conv(UNetHandle *u, const Grid3 &g, const ConvSrc &src, int cin, const s8 *wp, int cout,
                const float *bias, int relu, bf16 *y, const bf16 *mask,
                const ConvOut1 &o1 = ConvOut1{}) {
  if (cin % 16 || cout % 16 || cout > 256) {
    mf6hip_set_error("unsupported channel count " + std::to_string(cout));
    return MF6HIP_EUNSUPPORTED;
  }
  const int nco = cout / 16, cw = conv_cw(cin);
  const ConvTile t = conv_tile(g, nco);
  const int PH = 4 / t.WD * t.MT + 2, PD = t.WD + 2;
  const int shm = PD * PH * 18 * cw * 2;            // at most 62 KB
  const int mph = (65536 + PH - 1) / PH;
  const dim3 grid(t.tiles, t.gy);
  hipStream_t s = u->stream;
#define MF6_CONV(C, M)                                                                           \
  launch_conv_nc<C, M>(t.NC, grid, shm, s, g, src, cin, wp, nco, bias, relu, y, cout, mask, cout, \
                       o1, t.WD, mph)
  if (cw == 32) {
    if (t.MT == 4) MF6_CONV(32, 4);
    else if (t.MT == 2) MF6_CONV(32, 2);
    else MF6_CONV(32, 1);
  } else {
    if (t.MT == 4) MF6_CONV(16, 4);
    else if (t.MT == 2) MF6_CONV(16, 2);
    else MF6_CONV(16, 1);
  }
#undef MF6_CONV
  if (hipGetLastError() != hipSuccess) { mf6hip_set_error("conv launch failed"); return MF6HIP_EHIP; }
  return MF6HIP_OK;
}

// Splits of one layer's weight gradient: WG_MAXBLK workgroups over its
// channel tiles, at most one per voxel tile.  TD: the tile shape (4 x 4, 2 x
// 8 or 1 x 16 rows of 16 voxels) that pads the grid least.
struct WgradTile {
  int NC, gy, TD, nsplit;
};

WgradTile wgrad_tile(const Grid3 &g, int cin, int cout) {
  WgradTile t{};
  const int nco = cout / 16, ng = (nco + 3) / 4;
  t.NC = (nco + ng - 1) / ng;
  t.gy = cin / 16 * ng;
  long long pad = -1;
  int ntiles = 1;
  for (int td = 4; td >= 1; td >>= 1) {
    const int th = 16 / td, nd = (g.D + td - 1) / td, nh = (g.H + th - 1) / th;
    const long long v = (long long)nd * td * nh * th;
    if (pad < 0 || v < pad) {
      pad = v;
      t.TD = td;
      ntiles = nd * nh * ((g.W + 15) / 16);
    }
  }
  t.nsplit = (WG_MAXBLK + t.gy - 1) / t.gy;
  if (t.nsplit > ntiles) t.nsplit = ntiles;
  return t;
}

// floats of partials that a layer's weight gradient needs
size_t wgrad_part(const Grid3 &g, int cin, int cout) {
  return (size_t)wgrad_tile(g, cin, cout).nsplit * ((size_t)27 * cin + 1) * cout;
}

// weight + bias gradients of one conv layer into u->grad (accumulate)
int conv_wgrad(UNetHandle *u, const Grid3 &g, const UConv &L, const ConvSrc &src, const bf16 *dy,
               int accumulate) {
  hipStream_t s = u->stream;
  const WgradTile t = wgrad_tile(g, L.cin, L.cout);
  if (wgrad_part(g, L.cin, L.cout) > u->part_n) { mf6hip_set_error("partial buffer too small"); return MF6HIP_EINVAL; }
  const int PD = t.TD + 2, PH = 16 / t.TD + 2;
  const int shm = PD * PH * 18 * 32 + 256 * t.NC * 32;   // at most 64 KB
  const int mph = (65536 + PH - 1) / PH;
  const dim3 grid(t.nsplit, t.gy);
#define MF6_WGRAD(N)                                                                          \
  k_wgrad<N><<<grid, 256, shm, s>>>(g, src, L.cin, dy, L.cout, t.TD, mph, u->part)
  if (t.NC == 1) MF6_WGRAD(1);
  else if (t.NC == 2) MF6_WGRAD(2);
  else if (t.NC == 3) MF6_WGRAD(3);
  else MF6_WGRAD(4);
#undef MF6_WGRAD
  const int n = 27 * L.cin_real * L.cout + L.cout;
  k_wgrad_reduce<<<(n + 63) / 64, 256, 0, s>>>(u->part, t.nsplit, L.cin, L.cin_real, L.cout,
                                               u->grad + L.w_off, accumulate);
  if (hipGetLastError() != hipSuccess) { mf6hip_set_error("wgrad launch failed"); return MF6HIP_EHIP; }
  return MF6HIP_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// network set-up, forward, backward, training
// ---------------------------------------------------------------------------

static int u_pack(UNetHandle *u) {
  PackJobs jobs{};
  auto add = [&](const UConv &L, int flip, s8 *wp) {
    const int total = flip ? conv_nfrag(L.cout, L.cin) : conv_nfrag(L.cin, L.cout);
    jobs.j[jobs.n++] = PackJob{u->p + L.w_off, wp, L.cin_real, L.cin, L.cout, flip, jobs.nblk};
    jobs.nblk += (total + 255) / 256;
  };
  for (int i = 0; i < u->nconv(); i++) {
    const UConv &L = u->conv[i];
    add(L, 0, L.wp);
    if (L.wt) add(L, 1, L.wt);
  }
  k_pack_w<<<jobs.nblk, 256, 0, u->stream>>>(jobs);
  if (hipGetLastError() != hipSuccess) { mf6hip_set_error("pack launch failed"); return MF6HIP_EHIP; }
  return MF6HIP_OK;
}

// the input buffers of forward, and of grad (a call that fails leaves none behind)
static int u_inputs(UNetHandle *u, bool grad) {
  const size_t V0 = u->g[0].V();
  auto need = [](auto **p, size_t n) {
    if (*p) return (int)MF6HIP_OK;
    const int rc = ualloc(p, n);
    if (rc) *p = nullptr;
    return rc;
  };
  UCK(need(&u->dx, V0 * u->nin));
  if (grad) UCK(need(&u->dt32, V0));
  if (grad) UCK(need(&u->dt, V0));
  return MF6HIP_OK;
}

// forward from the padded level-0 input u->in0 to u->y
static int u_forward(UNetHandle *u) {
  hipStream_t s = u->stream;
  const int *c = u->ch;
  const int nl = u->nlev, bot = nl - 1;
  for (int l = 0; l < nl; l++) {
    const Grid3 &g = u->g[l];
    if (l > 0)
      k_pool<<<nblk((size_t)g.V() * c[l - 1] / 8), 256, 0, s>>>(g, u->g[l - 1], u->hb[l - 1],
                                                                c[l - 1], u->pin[l]);
    const UConv &A = u->conv[2 * l], &B = u->conv[2 * l + 1];
    UCK(launch_conv(u, g, u->enc_src(l), A.cin, A.wp, A.cout, u->p + A.b_off, 1, u->ha[l], nullptr));
    UCK(launch_conv(u, g, ConvSrc{u->ha[l], c[l]}, B.cin, B.wp, B.cout, u->p + B.b_off, 1, u->hb[l],
                    nullptr));
  }
  for (int l = bot - 1; l >= 0; l--) {
    const UConv &D = u->conv[u->dconv(l)];
    ConvOut1 o1;
    if (l == 0) o1 = ConvOut1{u->p + u->wo_off, u->p + u->bo_off, u->y};
    UCK(launch_conv(u, u->g[l], u->dec_src(l), D.cin, D.wp, D.cout, u->p + D.b_off, 1, u->u[l],
                    nullptr, o1));
  }
  if (hipGetLastError() != hipSuccess) { mf6hip_set_error("forward launch failed"); return MF6HIP_EHIP; }
  return MF6HIP_OK;
}

// loss of u->y against the target (bf16 slice) and the parameter gradients
// (accumulated into u->grad when accumulate != 0); u_forward must have run
static int u_backward(UNetHandle *u, const bf16 *tgt, int ldt, int toff, int accumulate) {
  hipStream_t s = u->stream;
  const int *c = u->ch;
  const int nl = u->nlev, bot = nl - 1;
  const int V0 = u->g[0].V();
  const int nb = nblk(V0) > 1024 ? 1024 : nblk(V0);
  k_loss<<<nb, 256, 0, s>>>(V0, u->y, tgt, ldt, toff, u->part);
  k_loss_final<<<1, 256, 0, s>>>(u->part, nb, u->lossv);
  k_out_bwd<<<nb, 256, 0, s>>>(V0, u->y, tgt, ldt, toff, u->lossv, u->u[0], u->p + u->wo_off,
                               u->gu[0], u->part);
  k_colsum<<<c[0] + 1, 256, 0, s>>>(u->part, nb, c[0] + 1, u->grad + u->wo_off, accumulate);
  // decoder, top to bottom
  for (int l = 0; l < bot; l++) {
    const Grid3 &g = u->g[l];
    const int cu = u->cup(l), ldc = cu + c[l];
    const UConv &D = u->conv[u->dconv(l)];
    UCK(conv_wgrad(u, g, D, u->dec_src(l), u->gu[l], accumulate));
    UCK(launch_conv(u, g, ConvSrc{u->gu[l], c[l]}, c[l], D.wt, ldc, nullptr, 0, u->gcat[l], nullptr));
    const Grid3 &gc = u->g[l + 1];
    // gradient of the coarser decoder output (or of the bottom output)
    // through the upsampling, masked by that output > 0
    const bf16 *msk = l < bot - 1 ? u->u[l + 1] : u->hb[bot];
    bf16 *dst = l < bot - 1 ? u->gu[l + 1] : u->ghb[bot];
    k_up_bwd<<<nblk((size_t)gc.V() * cu / 8), 256, 0, s>>>(gc, g, u->gcat[l], ldc, cu, msk, dst);
  }
  // encoder, bottom to top
  for (int l = bot; l >= 0; l--) {
    const Grid3 &g = u->g[l];
    if (l < bot) {
      // hb_l gradient: skip part of gcat[l] + pooled gradient from level l+1,
      // masked by hb_l > 0
      const int cu = u->cup(l), ldc = cu + c[l];
      k_pool_bwd<<<nblk((size_t)g.V() * c[l] / 8), 256, 0, s>>>(g, u->g[l + 1], u->gpin[l + 1],
                                                                c[l], u->gcat[l], ldc, cu,
                                                                u->hb[l], u->ghb[l]);
    }
    const UConv &A = u->conv[2 * l], &B = u->conv[2 * l + 1];
    const ConvSrc ha{u->ha[l], c[l]}, ghb{u->ghb[l], c[l]}, gha{u->gha[l], c[l]};
    UCK(conv_wgrad(u, g, B, ha, u->ghb[l], accumulate));
    UCK(launch_conv(u, g, ghb, c[l], B.wt, c[l], nullptr, 0, u->gha[l], u->ha[l]));
    UCK(conv_wgrad(u, g, A, u->enc_src(l), u->gha[l], accumulate));
    if (l > 0) UCK(launch_conv(u, g, gha, c[l], A.wt, c[l - 1], nullptr, 0, u->gpin[l], nullptr));
  }
  if (hipGetLastError() != hipSuccess) { mf6hip_set_error("backward launch failed"); return MF6HIP_EHIP; }
  return MF6HIP_OK;
}

static int u_adam(UNetHandle *u, float lr, float gscale) {
  u->adam_t++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - powf(b1, (float)u->adam_t), c2 = 1.f - powf(b2, (float)u->adam_t);
  k_adam<<<nblk(u->nparam), 256, 0, u->stream>>>((int)u->nparam, u->p, u->grad, u->m, u->v, lr,
                                                 b1, b2, 1e-8f, c1, c2, gscale);
  if (hipGetLastError() != hipSuccess) { mf6hip_set_error("adam launch failed"); return MF6HIP_EHIP; }
  return u_pack(u);
}

static void u_free(UNetHandle *u) {
  if (!u) return;
  if (u->stream) hipStreamSynchronize(u->stream);
  void *bufs[] = {u->p, u->grad, u->m, u->v, u->part, u->in0, u->y, u->lossv, u->data,
                  u->dx, u->dt32, u->dt};
  for (void *b : bufs)
    if (b) hipFree(b);
  for (int l = 0; l < MAXLEV; l++) {
    void *b2[] = {u->pin[l], u->ha[l], u->ghb[l], u->gha[l], u->gpin[l],
                  u->hb[l], u->u[l], u->gu[l], u->gcat[l]};
    for (void *b : b2)
      if (b) hipFree(b);
  }
  for (int i = 0; i < MAXCONV; i++) {
    if (u->conv[i].wp) hipFree(u->conv[i].wp);
    if (u->conv[i].wt) hipFree(u->conv[i].wt);
  }
  if (u->stream) hipStreamDestroy(u->stream);
  delete u;
}

extern "C" int mf6hip_unet_create(int nlay, int nrow, int ncol, int nin, int nlev,
                                  const int *channels, void **handle) {
  if (!handle || !channels) { mf6hip_set_error("null argument"); return MF6HIP_EINVAL; }
  *handle = nullptr;
  if (nlev < 2 || nlev > MAXLEV) {
    mf6hip_set_error("the network has 2.." + std::to_string(MAXLEV) + " levels");
    return MF6HIP_EUNSUPPORTED;
  }
  if (nlay < 1 || nrow < 2 || ncol < 2) {
    mf6hip_set_error("the learned preconditioner needs nrow and ncol >= 2");
    return MF6HIP_EUNSUPPORTED;
  }
  if (nin < 1 || nin > 16) { mf6hip_set_error("1..16 input channels"); return MF6HIP_EINVAL; }
  for (int l = 0; l < nlev; l++)
    if (channels[l] < 16 || channels[l] > 64 || channels[l] % 16) {
      mf6hip_set_error("channels must be 16, 32, 48 or 64");
      return MF6HIP_EUNSUPPORTED;
    }
  if (channels[0] != 16) { mf6hip_set_error("level-0 channels must be 16"); return MF6HIP_EUNSUPPORTED; }
  if ((long long)nlay * nrow * ncol > (1LL << 28)) { mf6hip_set_error("grid too large"); return MF6HIP_EUNSUPPORTED; }
  UNetHandle *u = new UNetHandle();
  u->nin = nin;
  u->nlev = nlev;
  for (int l = 0; l < nlev; l++) {
    u->ch[l] = channels[l];
    u->g[l] = l == 0 ? Grid3{nlay, nrow, ncol}
                     : Grid3{nlay, (u->g[l - 1].H + 1) / 2, (u->g[l - 1].W + 1) / 2};
  }
  const int *c = u->ch;
  const int bot = nlev - 1;
  size_t off = 0;
  int rc = MF6HIP_OK;
  for (int i = 0; i < u->nconv(); i++) {
    UConv &L = u->conv[i];
    if (i < 2 * nlev) {
      const int l = i / 2;
      L.cin = i == 0 ? 16 : (i % 2 ? c[l] : c[l - 1]);
      L.cin_real = i == 0 ? nin : L.cin;
      L.cout = c[l];
    } else {
      const int l = bot - 1 - (i - 2 * nlev);   // decoder level
      L.cin = u->cup(l) + c[l];
      L.cin_real = L.cin;
      L.cout = c[l];
    }
    L.w_off = off;
    off += (size_t)27 * L.cin_real * L.cout;
    L.b_off = off;
    off += L.cout;
    if (!rc) rc = ualloc(&L.wp, conv_nfrag(L.cin, L.cout));
    if (!rc && i != 0) rc = ualloc(&L.wt, conv_nfrag(L.cout, L.cin));
  }
  u->wo_off = off;
  off += c[0];
  u->bo_off = off;
  off += 1;
  u->nparam = off;
  if (!rc) rc = ualloc(&u->p, off);
  if (!rc) rc = ualloc(&u->grad, off);
  if (!rc) rc = ualloc(&u->m, off);
  if (!rc) rc = ualloc(&u->v, off);
  // partials: the largest layer's weight-gradient splits
  size_t pn = 1 << 20;
  for (int i = 0; i < u->nconv(); i++) {
    const UConv &L = u->conv[i];
    const int l = i < 2 * nlev ? i / 2 : bot - 1 - (i - 2 * nlev);
    pn = std::max(pn, wgrad_part(u->g[l], L.cin, L.cout));
  }
  u->part_n = pn;
  if (!rc) rc = ualloc(&u->part, pn);
  const size_t V0 = u->g[0].V();
  if (!rc) rc = ualloc(&u->in0, V0 * 16);
  if (!rc) rc = ualloc(&u->y, V0);
  if (!rc) rc = ualloc(&u->lossv, 4);
  for (int l = 0; l < nlev && !rc; l++) {
    const size_t V = u->g[l].V();
    if (l > 0) rc = ualloc(&u->pin[l], V * c[l - 1]);
    if (!rc) rc = ualloc(&u->ha[l], V * c[l]);
    if (!rc) rc = ualloc(&u->ghb[l], V * c[l]);
    if (!rc) rc = ualloc(&u->gha[l], V * c[l]);
    if (!rc && l > 0) rc = ualloc(&u->gpin[l], V * c[l - 1]);
    if (!rc) rc = ualloc(&u->hb[l], V * c[l]);
    if (!rc && l < bot) {
      rc = ualloc(&u->u[l], V * c[l]);
      if (!rc) rc = ualloc(&u->gu[l], V * c[l]);
      if (!rc) rc = ualloc(&u->gcat[l], V * (u->cup(l) + c[l]));
    }
  }
  if (!rc && hipStreamCreateWithFlags(&u->stream, hipStreamNonBlocking) != hipSuccess) {
    mf6hip_set_error("hipStreamCreate failed");
    rc = MF6HIP_EHIP;
  }
  if (!rc) {
    hipMemsetAsync(u->p, 0, sizeof(float) * off, u->stream);
    hipMemsetAsync(u->m, 0, sizeof(float) * off, u->stream);
    hipMemsetAsync(u->v, 0, sizeof(float) * off, u->stream);
    hipMemsetAsync(u->grad, 0, sizeof(float) * off, u->stream);
    rc = u_pack(u);
  }
  if (rc) { u_free(u); return rc; }
  *handle = u;
  return MF6HIP_OK;
}

extern "C" int mf6hip_unet_destroy(void *handle) {
  u_free((UNetHandle *)handle);
  return MF6HIP_OK;
}

extern "C" int mf6hip_unet_num_params(void *handle, long long *n) {
  UNetHandle *u = (UNetHandle *)handle;
  if (!u || !n) { mf6hip_set_error("null argument"); return MF6HIP_EINVAL; }
  *n = (long long)u->nparam;
  return MF6HIP_OK;
}

extern "C" int mf6hip_unet_set_params(void *handle, const float *params) {
  UNetHandle *u = (UNetHandle *)handle;
  if (!u || !params) { mf6hip_set_error("null argument"); return MF6HIP_EINVAL; }
  if (hipMemcpyAsync(u->p, params, sizeof(float) * u->nparam, hipMemcpyHostToDevice, u->stream) != hipSuccess) {
    mf6hip_set_error("hipMemcpy failed");
    return MF6HIP_EHIP;
  }
  hipMemsetAsync(u->m, 0, sizeof(float) * u->nparam, u->stream);
  hipMemsetAsync(u->v, 0, sizeof(float) * u->nparam, u->stream);
  u->adam_t = 0;
  UCK(u_pack(u));
  if (hipStreamSynchronize(u->stream) != hipSuccess) { mf6hip_set_error("sync failed"); return MF6HIP_EHIP; }
  return MF6HIP_OK;
}

extern "C" int mf6hip_unet_get_params(void *handle, float *params) {
  UNetHandle *u = (UNetHandle *)handle;
  if (!u || !params) { mf6hip_set_error("null argument"); return MF6HIP_EINVAL; }
  if (hipMemcpyAsync(params, u->p, sizeof(float) * u->nparam, hipMemcpyDeviceToHost, u->stream) != hipSuccess ||
      hipStreamSynchronize(u->stream) != hipSuccess) {
    mf6hip_set_error("hipMemcpy failed");
    return MF6HIP_EHIP;
  }
  return MF6HIP_OK;
}

// x: nin planes of V0 fp32 values (natural order), y: V0 fp32
extern "C" int mf6hip_unet_forward(void *handle, const float *x, float *y) {
  UNetHandle *u = (UNetHandle *)handle;
  if (!u || !x || !y) { mf6hip_set_error("null argument"); return MF6HIP_EINVAL; }
  const int V0 = u->g[0].V();
  UCK(u_inputs(u, false));
  float *dx = u->dx;
  int rc = MF6HIP_OK;
  if (hipMemcpyAsync(dx, x, sizeof(float) * V0 * u->nin, hipMemcpyHostToDevice, u->stream) != hipSuccess) rc = MF6HIP_EHIP;
  if (!rc) k_make_input<<<nblk(V0), 256, 0, u->stream>>>(V0, u->nin, dx, u->in0);
  if (!rc) rc = u_forward(u);
  if (!rc && hipMemcpyAsync(y, u->y, sizeof(float) * V0, hipMemcpyDeviceToHost, u->stream) != hipSuccess) rc = MF6HIP_EHIP;
  if (hipStreamSynchronize(u->stream) != hipSuccess && !rc) rc = MF6HIP_EHIP;
  if (rc == MF6HIP_EHIP) mf6hip_set_error("unet forward failed");
  return rc;
}

// loss and parameter gradients of one sample: x as in forward, t: V0 fp32
extern "C" int mf6hip_unet_grad(void *handle, const float *x, const float *t, float *loss,
                                float *grad) {
  UNetHandle *u = (UNetHandle *)handle;
  if (!u || !x || !t || !loss || !grad) { mf6hip_set_error("null argument"); return MF6HIP_EINVAL; }
  const int V0 = u->g[0].V();
  UCK(u_inputs(u, true));
  float *dx = u->dx;
  bf16 *dt = u->dt;
  int rc = MF6HIP_OK;
  if (!rc && hipMemcpyAsync(dx, x, sizeof(float) * V0 * u->nin, hipMemcpyHostToDevice, u->stream) != hipSuccess) rc = MF6HIP_EHIP;
  if (!rc && hipMemcpyAsync(u->dt32, t, sizeof(float) * V0, hipMemcpyHostToDevice, u->stream) != hipSuccess) rc = MF6HIP_EHIP;
  if (!rc) {
    k_make_input<<<nblk(V0), 256, 0, u->stream>>>(V0, u->nin, dx, u->in0);
    k_f32_to_bf16<<<nblk(V0), 256, 0, u->stream>>>(V0, u->dt32, dt);
    rc = u_forward(u);
  }
  if (!rc) rc = u_backward(u, dt, 1, 0, 0);
  float lv[2] = {0.f, 0.f};
  if (!rc && hipMemcpyAsync(lv, u->lossv, sizeof(lv), hipMemcpyDeviceToHost, u->stream) != hipSuccess) rc = MF6HIP_EHIP;
  if (!rc && hipMemcpyAsync(grad, u->grad, sizeof(float) * u->nparam, hipMemcpyDeviceToHost, u->stream) != hipSuccess) rc = MF6HIP_EHIP;
  if (hipStreamSynchronize(u->stream) != hipSuccess && !rc) rc = MF6HIP_EHIP;
  *loss = lv[0];
  if (rc == MF6HIP_EHIP) mf6hip_set_error("unet grad failed");
  return rc;
}

// training samples: n samples of V0 voxels x (nin inputs + 1 target), fp32
// planes [n][nin + 1][V0]; stored on the device in BF16 ([n][V0][4])
extern "C" int mf6hip_unet_set_data(void *handle, int n, const float *samples) {
  UNetHandle *u = (UNetHandle *)handle;
  if (!u || !samples || n < 1) { mf6hip_set_error("bad argument"); return MF6HIP_EINVAL; }
  if (u->nin != 3) { mf6hip_set_error("training data needs 3 input channels"); return MF6HIP_EUNSUPPORTED; }
  const size_t V0 = u->g[0].V();
  if (u->data) { hipFree(u->data); u->data = nullptr; }
  UCK(ualloc(&u->data, (size_t)n * V0 * 4));
  std::vector<bf16> tmp(V0 * 4);
  for (int i = 0; i < n; i++) {
    const float *sp = samples + (size_t)i * 4 * V0;
    for (size_t v = 0; v < V0; v++)
      for (int c = 0; c < 4; c++) tmp[v * 4 + c] = f2bf(sp[(size_t)c * V0 + v]);
    if (hipMemcpy(u->data + (size_t)i * V0 * 4, tmp.data(), sizeof(bf16) * V0 * 4, hipMemcpyHostToDevice) != hipSuccess) {
      mf6hip_set_error("hipMemcpy failed");
      return MF6HIP_EHIP;
    }
  }
  u->nsamples = n;
  return MF6HIP_OK;
}

// Adam training over the stored samples: nsteps steps of `batch` samples
// taken in the order given by order[nsteps * batch]; loss_out[nsteps]
// receives each step's mean sample loss.
extern "C" int mf6hip_unet_train(void *handle, int nsteps, int batch, const int *order, float lr,
                                 float *loss_out) {
  UNetHandle *u = (UNetHandle *)handle;
  if (!u || !order || !loss_out || nsteps < 1 || batch < 1) { mf6hip_set_error("bad argument"); return MF6HIP_EINVAL; }
  if (!u->data) { mf6hip_set_error("no training data"); return MF6HIP_EINVAL; }
  const size_t V0 = u->g[0].V();
  float *dl = nullptr;
  UCK(ualloc(&dl, (size_t)nsteps * batch));
  int rc = MF6HIP_OK;
  for (int st = 0; st < nsteps && !rc; st++) {
    for (int b = 0; b < batch && !rc; b++) {
      const int idx = order[st * batch + b];
      if (idx < 0 || idx >= u->nsamples) { mf6hip_set_error("sample index out of range"); rc = MF6HIP_EINVAL; break; }
      const bf16 *smp = u->data + (size_t)idx * V0 * 4;
      k_expand_sample<<<nblk(V0), 256, 0, u->stream>>>((int)V0, smp, u->in0);
      rc = u_forward(u);
      if (!rc) rc = u_backward(u, smp, 4, 3, b > 0);
      if (!rc && hipMemcpyAsync(dl + (size_t)st * batch + b, u->lossv, sizeof(float), hipMemcpyDeviceToDevice, u->stream) != hipSuccess) rc = MF6HIP_EHIP;
    }
    if (!rc) rc = u_adam(u, lr, 1.f / batch);
  }
  std::vector<float> hl((size_t)nsteps * batch);
  if (!rc && hipMemcpyAsync(hl.data(), dl, sizeof(float) * hl.size(), hipMemcpyDeviceToHost, u->stream) != hipSuccess) rc = MF6HIP_EHIP;
  if (hipStreamSynchronize(u->stream) != hipSuccess && !rc) rc = MF6HIP_EHIP;
  hipFree(dl);
  if (!rc)
    for (int st = 0; st < nsteps; st++) {
      float s = 0.f;
      for (int b = 0; b < batch; b++) s += hl[(size_t)st * batch + b];
      loss_out[st] = s / batch;
    }
  if (rc == MF6HIP_EHIP) mf6hip_set_error("unet training failed");
  return rc;
}

// device-side application used by the solver: in0 already filled by the
// caller on the network's stream; result in u->y (fp32, natural order)
int mf6hip_unet_apply_device(void *handle, hipStream_t s) {
  UNetHandle *u = (UNetHandle *)handle;
  hipStream_t keep = u->stream;
  u->stream = s;
  int rc = u_forward(u);
  u->stream = keep;
  return rc;
}

unsigned short *mf6hip_unet_input(void *net) { return ((UNetHandle *)net)->in0; }
float *mf6hip_unet_output(void *net) { return ((UNetHandle *)net)->y; }
int mf6hip_unet_dims(void *net, int *nlay, int *nrow, int *ncol, int *nin) {
  UNetHandle *u = (UNetHandle *)net;
  if (!u) { mf6hip_set_error("null network"); return MF6HIP_EINVAL; }
  *nlay = u->g[0].D;
  *nrow = u->g[0].H;
  *ncol = u->g[0].W;
  *nin = u->nin;
  return MF6HIP_OK;
}
