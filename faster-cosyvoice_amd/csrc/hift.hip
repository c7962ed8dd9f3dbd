// HiFT vocoder kernels on gfx950 (see hift.hpp for the layout and the launch contracts).
//
// Every convolution of the vocoder is one implicit GEMM on the matrix cores.  The causal
// unit-stride ones (upsampling, resblocks, conv_post) run in hift_split.hip where the handle has
// split weights; the rest -- conv_pre, the strided source convs, and the fp64 F0 predictor with a
// kernel of its own -- run here on v_mfma_{f32,f64}_16x16x4: weights are the A operand (rows = output
// channels), the gathered input rows the B operand, so a lane's four accumulators are four channels
// of one time step (consecutive in fp32; four apart in fp64, whose 16x16 result is laid out by rows
// 4 e + lane / 16).  Operands of the fp32 convolutions go through LDS K-contiguous, 32 (or 16)
// input channels of one tap per chunk, with a register-prefetched double buffer.  A workgroup owns
// 64 time rows x 64 output channels (32 x 32 in launches too small to give every CU a 64 x 64
// tile).  Activations that sit between two convolutions are fused: LeakyReLU into the input
// prologue, bias, ELU, residual add, Snake and the resblock mean into the epilogue, and the
// epilogue can also write Snake(y) as a second output for the next conv.
#include <math.h>

#include <cstdlib>

#include "hift.hpp"
#include "hift_device.hpp"

namespace fcv {
namespace {

constexpr int kTileR = 64;  // time rows per workgroup
constexpr int kTileC = 64;  // output channels per workgroup
constexpr long kSmallTileBelow = 256;  // 64x64 tiles per launch under which 32x32 tiles run

typedef double f64x4 __attribute__((ext_vector_type(4)));


__device__ __forceinline__ f32x4 mfma_16x16x4(float a, float b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f64x4 mfma_16x16x4(double a, double b, const f64x4& c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ double elu(double x) { return x > 0.0 ? x : expm1(x); }

// epilogue of one output element (row, channel c) from its accumulator value
__device__ __forceinline__ void conv_store1(const HiftConv& p, long row, int c, float acc) {
  float v = acc + static_cast<const float*>(p.bias)[c];
  const long i = row * p.ldo + c;
  if (p.add) v = v + static_cast<const float*>(p.add)[row * p.ld_add + c];
  if (p.mode == HIFT_ACC_ADD) v = static_cast<const float*>(p.accin)[i] + v;
  if (p.mode == HIFT_ACC_ADD_DIV) v = (static_cast<const float*>(p.accin)[i] + v) / p.div;
  if (p.snake_out) v = snake(v, p.alpha[c], p.inv_alpha[c]);
  if (p.n_snakes) p.snakes[0].out[i] = snake(v, p.snakes[0].alpha[c], p.snakes[0].inv_alpha[c]);
  static_cast<float*>(p.out)[i] = v;
}

__device__ __forceinline__ float4 ld4f(const float* q) { return *reinterpret_cast<const float4*>(q); }

// conv_store1 for the four consecutive fp32 channels c .. c + 3 of one row, with 16-byte loads
// and stores (same operations in the same order, so the results are bit-identical)
__device__ __forceinline__ void conv_store4(const HiftConv& p, long row, int c, const f32x4& acc) {
  const float4 b = ld4f(static_cast<const float*>(p.bias) + c);
  float v[4] = {acc[0] + b.x, acc[1] + b.y, acc[2] + b.z, acc[3] + b.w};
  const long i = row * p.ldo + c;
  if (p.add) {
    const float4 a = ld4f(static_cast<const float*>(p.add) + row * p.ld_add + c);
    v[0] = v[0] + a.x; v[1] = v[1] + a.y; v[2] = v[2] + a.z; v[3] = v[3] + a.w;
  }
  if (p.mode != HIFT_ACC_WRITE) {
    const float4 a = ld4f(static_cast<const float*>(p.accin) + i);
    v[0] = a.x + v[0]; v[1] = a.y + v[1]; v[2] = a.z + v[2]; v[3] = a.w + v[3];
    if (p.mode == HIFT_ACC_ADD_DIV)
      for (int e = 0; e < 4; ++e) v[e] = v[e] / p.div;
  }
  // the Snakes one channel at a time: four inlined sinf at once spill
  if (p.snake_out) {
#pragma unroll 1
    for (int e = 0; e < 4; ++e) v[e] = snake(v[e], p.alpha[c + e], p.inv_alpha[c + e]);
  }
  if (p.n_snakes) {
    const HiftConv::Snake& q = p.snakes[0];
    float w[4];
#pragma unroll 1
    for (int e = 0; e < 4; ++e) w[e] = snake(v[e], q.alpha[c + e], q.inv_alpha[c + e]);
    *reinterpret_cast<float4*>(q.out + i) = float4{w[0], w[1], w[2], w[3]};
  }
  *reinterpret_cast<float4*>(static_cast<float*>(p.out) + i) = float4{v[0], v[1], v[2], v[3]};
}

// The 16x16x4 accumulators of lane (li, lg) hold channels cb + 4 lg + e (e = 0..3) of the tile's
// channel base cb
__device__ void conv_store(const HiftConv& p, long row, int cb, int lg,
                           const f32x4& acc) {
  const int c = cb + 4 * lg;
  if (p.vec4 && c + 3 < p.cout) {
    conv_store4(p, row, c, acc);
    return;
  }
  for (int e = 0; e < 4; ++e)
    if (c + e < p.cout) conv_store1(p, row, c + e, acc[e]);
}

// BK input channels of one tap per chunk (cin_pad % BK == 0), each lane feeding
// k = 16 m + 4 lg + s at MFMA step (m, s).  A workgroup owns TS time rows x TS output channels
// (TS = 64, or 32 for launches too small to give every CU a 64x64 tile); its four waves each
// own a TS/2 x TS/2 quarter.  Loaders: at TS = 64 every thread moves BK / 16 groups of 4
// elements of one weight row and one input row; at TS = 32 waves 0-1 move the weight rows and
// waves 2-3 the input rows, the same groups each.  Every output element accumulates the chunks
// in the same order with the same lane/slot -> k rule at both sizes, so the tile size does not
// change a result.
template <int BK, int TS>
__global__ __launch_bounds__(256) void hift_conv_kernel(const HiftConv p) {
  const HiftDocs* __restrict__ docs = p.docs;
  using VT = f32x4;
  constexpr int PITCH = BK + 4;  // LDS row pitch in elements (conflict-free 16-byte reads)
  constexpr int G = BK / 16;
  constexpr int NQ = TS / 32;    // 16x16 accumulator tiles per wave along each side
  static_assert(TS == 64 || TS == 32, "tile size");
  __shared__ __attribute__((aligned(16))) float sA[2][TS][PITCH];
  __shared__ __attribute__((aligned(16))) float sB[2][TS][PITCH];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wc = wave & 1, wt = wave >> 1;
  const int li = lane & 15, lg = lane >> 4;
  const int n_docs = docs->n;
  const int rows_out = docs->b[n_docs];  // live rows (the grid covers the capacity)
  const int r0 = blockIdx.x * TS;
  if (r0 >= rows_out) return;
  const int co0 = blockIdx.y * TS;
  const int cpt = p.cin_pad / BK;
  const int KC = p.k * cpt;
  const long kcin = (long)p.k * p.cin_pad;

  // loader roles: weight row / input row lr, 4-element quarter lq of each 16-channel group;
  // at TS = 32 a thread loads the weights (ld_w) or the inputs (ld_x), not both
  const int lr = TS == 64 ? tid >> 2 : (tid & 127) >> 2, lq = tid & 3;
  const bool ld_w = TS == 64 || tid < 128, ld_x = TS == 64 || tid >= 128;
  const int r = r0 + lr;
  const bool valid = ld_x && r < rows_out;
  int in_base = 0, in_len = 0, pos = 0;
  if (valid) {
    const int d = doc_of(docs->b, n_docs, r);
    pos = r - docs->b[d];
    in_base = docs->a[d];
    in_len = docs->a[d + 1] - in_base;
  }
  const float* X = static_cast<const float*>(p.x);
  const float* W = static_cast<const float*>(p.w) + (long)(co0 + lr) * kcin + 4 * lq;

  // Two register sets: the loads of chunk kc + 2 are issued while chunk kc is computed and
  // chunk kc + 1 (loaded one iteration earlier) is written to LDS, so every load has about two
  // chunk computations to arrive.  The sets are picked by compile-time index (loop unrolled by 2).
  VT ra[2][G], rb[2][G];
  auto fetch = [&](int kc, VT (&a)[G], VT (&b)[G]) {
    const int tap = kc / cpt;
    const int c0 = (kc - tap * cpt) * BK + 4 * lq;
    const int u = pos * p.stride + tap * p.dil - p.pad;
    const int q = p.up > 1 ? (u >= 0 ? u / p.up : -1) : u;
    const bool live = valid && q >= 0 && q < in_len;
    const float* xr = X + (long)(in_base + q) * p.ldx + c0;
#pragma unroll
    for (int m = 0; m < G; ++m) {
      if (ld_w) a[m] = *reinterpret_cast<const VT*>(W + (long)kc * BK + 16 * m);
      b[m] = VT{0.0f, 0.0f, 0.0f, 0.0f};
      if (live) b[m] = *reinterpret_cast<const VT*>(xr + 16 * m);
    }
  };
  // the input prologue runs here, when the data is needed, so fetch never waits for its loads
  auto stash = [&](int buf, const VT (&a)[G], const VT (&b)[G]) {
#pragma unroll
    for (int m = 0; m < G; ++m) {
      VT bm = b[m];
      if (p.pro == HIFT_PRO_LEAKY) {
#pragma unroll
        for (int e = 0; e < 4; ++e) bm[e] = bm[e] > 0.0f ? bm[e] : bm[e] * p.slope;
      }
      if (ld_w) *reinterpret_cast<VT*>(&sA[buf][lr][16 * m + 4 * lq]) = a[m];
      if (ld_x) *reinterpret_cast<VT*>(&sB[buf][lr][16 * m + 4 * lq]) = bm;
    }
  };

  VT acc[NQ][NQ];
#pragma unroll
  for (int a = 0; a < NQ; ++a)
#pragma unroll
    for (int b = 0; b < NQ; ++b) acc[a][b] = VT{0.0f, 0.0f, 0.0f, 0.0f};

  auto compute = [&](int cur) {
#pragma unroll
    for (int m = 0; m < G; ++m) {
      VT av[NQ], bv[NQ];
#pragma unroll
      for (int a = 0; a < NQ; ++a)
        av[a] = *reinterpret_cast<const VT*>(&sA[cur][wc * (TS / 2) + a * 16 + li][16 * m + 4 * lg]);
#pragma unroll
      for (int b = 0; b < NQ; ++b)
        bv[b] = *reinterpret_cast<const VT*>(&sB[cur][wt * (TS / 2) + b * 16 + li][16 * m + 4 * lg]);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int a = 0; a < NQ; ++a)
#pragma unroll
          for (int b = 0; b < NQ; ++b) acc[a][b] = mfma_16x16x4(av[a][s], bv[b][s], acc[a][b]);
    }
  };

  fetch(0, ra[0], rb[0]);
  fetch(min(1, KC - 1), ra[1], rb[1]);
  stash(0, ra[0], rb[0]);
  __syncthreads();
  // Fetches and stashes run unconditionally (chunk indices clamped to the last chunk; a surplus
  // chunk lands in the LDS buffer no later computation reads), so no path leaves a load
  // pending and the compiler does not wait for the loads before the computation they overlap.
  // The fences keep each fetch ahead of its computation.
  for (int kc = 0; kc < KC; kc += 2) {
    // chunk kc is in LDS buffer 0; register set 1 holds chunk kc + 1
    fetch(min(kc + 2, KC - 1), ra[0], rb[0]);
    __builtin_amdgcn_sched_barrier(0);
    compute(0);
    stash(1, ra[1], rb[1]);
    __syncthreads();
    if (kc + 1 >= KC) break;
    // chunk kc + 1 is in buffer 1; register set 0 holds chunk kc + 2
    fetch(min(kc + 3, KC - 1), ra[1], rb[1]);
    __builtin_amdgcn_sched_barrier(0);
    compute(1);
    stash(0, ra[0], rb[0]);
    __syncthreads();
  }

  // D[i = channel][j = row]: lane holds row li and four channels of each 16x16 tile
#pragma unroll
  for (int b = 0; b < NQ; ++b) {
    const int rr = r0 + wt * (TS / 2) + b * 16 + li;
    if (rr >= rows_out) continue;
    const int d = doc_of(docs->b, n_docs, rr);
    const int pp = rr - docs->b[d];
    const long row_w = p.reflect ? (long)docs->b[d] + d + 1 + pp : rr;
#pragma unroll
    for (int a = 0; a < NQ; ++a) {
      const int cb = co0 + wc * (TS / 2) + a * 16;
      conv_store(p, row_w, cb, lg, acc[a][b]);
      // reflection padding (1, 0): row 0 of the document repeats the result's row 1
      if (p.reflect && pp == 1) conv_store(p, (long)docs->b[d] + d, cb, lg, acc[a][b]);
    }
  }
}

// out[r][c] = snake(x[r][c]), four channels a thread
__global__ __launch_bounds__(256) void snake_kernel(const float* __restrict__ x, int ldx,
                                                    float* __restrict__ out, int ldo, int C,
                                                    const float* __restrict__ alpha,
                                                    const float* __restrict__ inv_alpha,
                                                    const HiftDocs* __restrict__ docs) {
  const int q = C / 4;
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long r = i / q;
  if (r >= docs->b[docs->n]) return;
  const int c = (int)(i - r * q) * 4;
  const f32x4 v = *reinterpret_cast<const f32x4*>(x + r * ldx + c);
  f32x4 y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = snake(v[e], alpha[c + e], inv_alpha[c + e]);
  *reinterpret_cast<f32x4*>(out + r * ldo + c) = y;
}

// out = the mean of in.n tensors, four values a thread, summed in order
__global__ __launch_bounds__(256) void mean_kernel(const HiftMean in, float* __restrict__ out, int C,
                                                   const HiftDocs* __restrict__ docs) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)docs->b[docs->n] * (C / 4)) return;
  f32x4 v = reinterpret_cast<const f32x4*>(in.x[0])[i];
  for (int k = 1; k < in.n; ++k) v += reinterpret_cast<const f32x4*>(in.x[k])[i];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = v[e] / (float)in.n;
  reinterpret_cast<f32x4*>(out)[i] = v;
}

// One layer of the fp64 F0 predictor on v_mfma_f64_16x16x4: out[r][co] = elu(b[co] + sum_k W[co][k]
// x[r + tap][c]), k = tap * cin + c.  A workgroup owns a 16 T x 16 T tile and its four waves a
// quarter of K each (added in order in LDS), straight from global memory: these products have 72 to
// a few thousand rows, so what counts is the chain of MFMAs a wave runs (64 cycles each), and a
// quarter of K on four times the waves cuts it to a quarter.  One layer at 72 rows 44 -> 15 us
// against 32x32 tiles with K in one chain through LDS (1664 rows: the same); T = 2 halves the operand
// reads where 16x16 tiles would be many (the sums are the same).
template <typename X, int T>
__global__ __launch_bounds__(256) void f0_conv_kernel(const HiftConv p) {
  constexpr int TS = 16 * T;
  const HiftDocs* __restrict__ docs = p.docs;
  __shared__ double part[4][TS][TS + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int n_docs = docs->n, rows_out = docs->b[n_docs];
  const int r0 = blockIdx.x * TS, co0 = blockIdx.y * TS;
  if (r0 >= rows_out) return;
  const int K = p.k * p.cin_pad, quarter = K / 4;
  const int k_begin = wave * quarter, k_end = k_begin + quarter;

  // lane (li, lg) holds k = k0 + 4 lg + 0..3 of weight row li and of input row li
  const double* W[T];
  int pos[T], in_base[T], in_len[T];
#pragma unroll
  for (int i = 0; i < T; ++i) {
    W[i] = static_cast<const double*>(p.w) + (long)(co0 + 16 * i + li) * K + 4 * lg;
    const int r = r0 + 16 * i + li;
    pos[i] = -(1 << 29);
    in_base[i] = in_len[i] = 0;
    if (r < rows_out) {
      const int d = doc_of(docs->b, n_docs, r);
      pos[i] = r - docs->b[d] - p.pad;
      in_base[i] = docs->a[d];
      in_len[i] = docs->a[d + 1] - in_base[i];
    }
  }
  const X* x = static_cast<const X*>(p.x) + 4 * lg;
  constexpr int PD = T == 1 ? 4 : 2;
  f64x4 wa[PD][T], xb[PD][T];
  auto fetch = [&](int slot, int k0) {
    const int tap = k0 / p.cin_pad, c = k0 - tap * p.cin_pad;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      wa[slot][i] = *reinterpret_cast<const f64x4*>(W[i] + k0);
      const int q = pos[i] + tap;
      xb[slot][i] = f64x4{0.0, 0.0, 0.0, 0.0};
      if (q >= 0 && q < in_len[i]) {
        typedef X x4 __attribute__((ext_vector_type(4)));
        const x4 v = *reinterpret_cast<const x4*>(x + (long)(in_base[i] + q) * p.ldx + c);
        xb[slot][i] = f64x4{(double)v[0], (double)v[1], (double)v[2], (double)v[3]};
      }
    }
  };
  f64x4 acc[T][T];
#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int b = 0; b < T; ++b) acc[a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int u = 0; u < PD - 1; ++u) fetch(u, min(k_begin + 16 * u, k_end - 16));
  for (int k0 = k_begin; k0 < k_end; k0 += 16 * PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      const int kk = k0 + 16 * u;
      if (kk >= k_end) break;
      fetch((u + PD - 1) % PD, min(kk + 16 * (PD - 1), k_end - 16));
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int a = 0; a < T; ++a)
#pragma unroll
          for (int b = 0; b < T; ++b)
            acc[a][b] = mfma_16x16x4(wa[u][a][e], xb[u][b][e], acc[a][b]);
    }
  }
  // D: lane holds row li, channels 4 e + lg
#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int b = 0; b < T; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[wave][16 * b + li][16 * a + 4 * e + lg] = acc[a][b][e];
  __syncthreads();
  for (int i = tid; i < TS * TS; i += 256) {
    const int t = i / TS, c = i - t * TS;
    if (r0 + t >= rows_out || co0 + c >= p.cout) continue;
    const double v = ((part[0][t][c] + part[1][t][c]) + part[2][t][c]) + part[3][t][c];
    static_cast<double*>(p.out)[(long)(r0 + t) * p.ldo + co0 + c] =
        elu(v + static_cast<const double*>(p.bias)[co0 + c]);
  }
}

__global__ __launch_bounds__(64) void f0_head_kernel(const double* __restrict__ h, int C,
                                                     const double* __restrict__ w,
                                                     const double* __restrict__ b,
                                                     float* __restrict__ f0,
                                                     const HiftDocs* __restrict__ docs) {
  const long r = blockIdx.x;
  if (r >= docs->b[docs->n]) return;
  double s = 0.0;
  for (int c = threadIdx.x; c < C; c += 64) s = fma(h[r * C + c], w[c], s);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
  if (threadIdx.x == 0) f0[r] = (float)fabs(s + b[0]);
}

// One workgroup per (document, harmonic): the per-frame phase increment of harmonic h is
// rad = frac(f0 (h+1) / sr); the frame-rate value is the linear interpolation the reference
// takes from the sample-rate sequence (whose first sample also carries rand_ini[h]); the
// phase is the running sum in frame order, times 2 pi, times the upsampling scale.  The running
// sum is held in fp64 and rounded to fp32 at every frame, which is what the reference's
// torch.cumsum over the fp32 rad values (cosyvoice/hifigan/generator.py:255) computes on the
// CPU, whose kernel accumulates fp32 in double: an fp32 running sum drifts by ~1e-6 relative
// per few hundred frames, and the phase multiplies that by 2 pi x 480.  The sum is a scan over
// blocks of 256 frames (lanes, waves, blocks): fp64 holds these sums of fp32 values below 2
// exactly unless a value is under 2^-20 of them, so its order does not show.  One thread a harmonic
// that walks the frames took 690 us for 900 frames.
__global__ __launch_bounds__(256) void source_phase_kernel(const HiftSource p,
                                                           const HiftDocs* __restrict__ docs) {
#pragma clang fp contract(off)
  const int d = blockIdx.x, h = blockIdx.y;
  if (d >= docs->n) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  __shared__ double wsum[2][4];
  const int f_base = docs->a[d];
  const int T = docs->a[d + 1] - f_base;
  const long L = (long)T * p.scale;
  const float mult = (float)(h + 1);
  const float sr = (float)p.sampling_rate;
  const float scale = (float)p.scale;
  auto rad_at = [&](long i) {
    const float x = (p.f0[f_base + i / p.scale] * mult) / sr;
    float v = x - floorf(x);
    if (i == 0) v = v + p.rand_ini[h];
    return v;
  };
  double before = 0.0;  // the sum of the earlier blocks
  for (int t0 = 0, par = 0; t0 < T; t0 += 256, par ^= 1) {
    const int t = t0 + tid;
    double c = 0.0;
    if (t < T) {
      float src = scale * ((float)t + 0.5f) - 0.5f;
      if (src < 0.0f) src = 0.0f;
      const long i0 = (long)src;
      const float l1 = fminf(fmaxf(src - (float)i0, 0.0f), 1.0f);
      const float l0 = 1.0f - l1;
      const long i1 = i0 + (i0 < L - 1 ? 1 : 0);
      const float a = l0 * rad_at(i0);
      const float b = l1 * rad_at(i1);
      c = (double)(a + b);
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double o = __shfl_up(c, off, 64);
      if (lane >= off) c = o + c;
    }
    if (lane == 63) wsum[par][wave] = c;
    __syncthreads();  // (the next block writes the other half)
    double base = before;
    for (int w = 0; w < 4; ++w) {
      if (w == wave) c = base + c;
      base = base + wsum[par][w];
    }
    before = base;
    if (t < T) {
      float ph = ((float)c * 2.0f) * 3.14159265358979323846f;
      ph = ph * scale;
      p.sines[(long)(f_base + t) * p.H + h] = sinf(ph) * p.sine_amp;
    }
  }
}

__global__ __launch_bounds__(256) void source_sample_kernel(const HiftSource p,
                                                            const HiftDocs* __restrict__ docs) {
#pragma clang fp contract(off)
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= docs->b[docs->n]) return;
  const int d = doc_of(docs->b, docs->n, n);
  const int pos = n - docs->b[d];
  const int fr = docs->a[d] + pos / p.scale;
  const float f0 = p.f0[fr];
  const float uv = f0 > p.voiced_threshold ? 1.0f : 0.0f;
  const float amp = uv * p.noise_std + ((1.0f - uv) * p.sine_amp) / 3.0f;
  const float* noise = p.table + (long)pos * p.H;
  float acc = 0.0f;
  for (int h = 0; h < p.H; ++h) {
    const float wave = p.sines[(long)fr * p.H + h] * uv + amp * noise[h];
    acc = acc + p.lin_w[h] * wave;
  }
  p.s[n] = tanhf(acc + p.lin_b[0]);
}

// cos / sin of 2 pi m / 16 for m = 0..15
__device__ __forceinline__ float cos16(int m) { return cospif((float)(m & 15) / 8.0f); }
__device__ __forceinline__ float sin16(int m) { return sinpif((float)(m & 15) / 8.0f); }

__global__ __launch_bounds__(256) void stft_kernel(const float* __restrict__ s,
                                                   const float* __restrict__ win,
                                                   float* __restrict__ out, int ld,
                                                   const HiftDocs* __restrict__ docs) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= docs->b[docs->n]) return;
  const int d = doc_of(docs->b, docs->n, f);
  const int fl = f - docs->b[d];
  const float* x = s + docs->a[d];
  const int L = docs->a[d + 1] - docs->a[d];
  float v[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    int i = 4 * fl + j - 8;
    if (i < 0) i = -i;
    if (i >= L) i = 2 * (L - 1) - i;
    v[j] = x[i] * win[j];
  }
  float* o = out + (long)f * ld;
#pragma unroll
  for (int k = 0; k <= 8; ++k) {
    float re = 0.0f, im = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      re = fmaf(v[j], cos16(j * k), re);
      im = fmaf(-v[j], sin16(j * k), im);
    }
    o[k] = re;
    o[9 + k] = im;
  }
  for (int c = 18; c < ld; ++c) o[c] = 0.0f;
}

// windowed inverse real DFT of one frame: mag = min(exp(y[k]), 100), ph = sin(y[9 + k])
__global__ __launch_bounds__(256) void istft_frame_kernel(const float* __restrict__ y, int ldy,
                                                          const float* __restrict__ win,
                                                          float* __restrict__ fr,
                                                          const HiftDocs* __restrict__ docs) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= docs->a[docs->n]) return;
  const float* row = y + (long)f * ldy;
  float re[9], im[9];
#pragma unroll
  for (int k = 0; k <= 8; ++k) {
    const float mag = fminf(expf(row[k]), 100.0f);
    const float ph = sinf(row[9 + k]);
    re[k] = mag * cosf(ph);
    im[k] = mag * sinf(ph);
  }
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    float acc = re[0] + ((j & 1) ? -re[8] : re[8]);
    float h = 0.0f;
#pragma unroll
    for (int k = 1; k <= 7; ++k) h = h + (re[k] * cos16(j * k) - im[k] * sin16(j * k));
    acc = (acc + 2.0f * h) * (1.0f / 16.0f);
    fr[(long)f * 16 + j] = acc * win[j];
  }
}

// overlap-add: output sample pos of document d sits at padded position pos + 8 of the frame
// sequence; divided by the overlap-added squared window, clamped
__global__ __launch_bounds__(256) void istft_ola_kernel(const float* __restrict__ fr,
                                                        const float* __restrict__ win,
                                                        float* __restrict__ out, float limit,
                                                        const HiftDocs* __restrict__ docs) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= docs->b[docs->n]) return;
  const int d = doc_of(docs->b, docs->n, n);
  const int P = n - docs->b[d] + 8;
  const int f_base = docs->a[d];
  const int F = docs->a[d + 1] - f_base;
  float y = 0.0f, env = 0.0f;
  const int f_hi = min(P / 4, F - 1);
  for (int f = max(0, (P - 12) / 4); f <= f_hi; ++f) {
    const int j = P - 4 * f;
    if (j < 0 || j >= 16) continue;
    y = y + fr[(long)(f_base + f) * 16 + j];
    env = env + win[j] * win[j];
  }
  const float v = y / env;
  out[n] = fminf(fmaxf(v, -limit), limit);
}

__global__ __launch_bounds__(256) void copy_live_kernel(const float* __restrict__ src,
                                                        float* __restrict__ dst,
                                                        const HiftDocs* __restrict__ docs) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < docs->b[docs->n]) dst[i] = src[i];
}

unsigned blocks_for(long n, int threads) { return (unsigned)((n + threads - 1) / threads); }

bool aligned16(const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; }

hipError_t launch_conv(const HiftConv& p_in, hipStream_t stream) {
  if (p_in.rows_out <= 0) return hipSuccess;
  if (p_in.cin_pad % 16 != 0) return hipErrorInvalidValue;
  HiftConv p = p_in;
  // 16-byte epilogue accesses when every row pitch and base the epilogue touches allows them
  p.vec4 = p.ldo % 4 == 0 && aligned16(p.out) && aligned16(p.bias) &&
           (!p.add || (p.ld_add % 4 == 0 && aligned16(p.add))) &&
           (p.mode == HIFT_ACC_WRITE || aligned16(p.accin)) &&
           (!p.snake_out || (aligned16(p.alpha) && aligned16(p.inv_alpha))) &&
           (!p.n_snakes || (aligned16(p.snakes[0].out) && aligned16(p.snakes[0].alpha) &&
                            aligned16(p.snakes[0].inv_alpha)));
  if (p.n_snakes > 1 || !p.docs) return hipErrorInvalidValue;
  // 64x64 tiles, or 32x32 where 64x64 tiles would not give every CU one (results do not depend on
  // it).
  // FCV_HIFT_TILE=32 or 64 forces one size: a test hook, since both must give the same bits.
  const long tiles64 =
      (long)((p.rows_live + kTileR - 1) / kTileR) * ((p.cout + kTileC - 1) / kTileC);
  const char* forced = std::getenv("FCV_HIFT_TILE");
  const int force = forced ? std::atoi(forced) : 0;
  if (force == 32 || (force != 64 && tiles64 < kSmallTileBelow)) {
    const dim3 grid((p.rows_out + 31) / 32, (p.cout + 31) / 32);
    if (p.cin_pad % 32 == 0)
      hipLaunchKernelGGL((hift_conv_kernel<32, 32>), grid, dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL((hift_conv_kernel<16, 32>), grid, dim3(256), 0, stream, p);
    return hipGetLastError();
  }
  const dim3 grid((p.rows_out + kTileR - 1) / kTileR, (p.cout + kTileC - 1) / kTileC);
  if (p.cin_pad % 32 == 0)
    hipLaunchKernelGGL((hift_conv_kernel<32, 64>), grid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((hift_conv_kernel<16, 64>), grid, dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace

hipError_t hift_conv_f32(const HiftConv& p, hipStream_t stream) {
  return launch_conv(p, stream);
}

hipError_t hift_snake(const float* x, int ldx, float* out, int ldo, int rows, int C,
                      const float* alpha, const float* inv_alpha, const HiftDocs* docs,
                      hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const long n = (long)rows * (C / 4);
  hipLaunchKernelGGL(snake_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, stream, x, ldx, out,
                     ldo, C, alpha, inv_alpha, docs);
  return hipGetLastError();
}

hipError_t hift_mean(const HiftMean& in, float* out, int rows, int C, const HiftDocs* docs,
                     hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  if (in.n < 1 || in.n > 4 || C % 4 != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(mean_kernel, dim3(blocks_for((long)rows * (C / 4), 256)), dim3(256), 0, stream,
                     in, out, C, docs);
  return hipGetLastError();
}

namespace {
template <typename X>
hipError_t launch_f0(const HiftConv& p, hipStream_t stream) {
  // 16x16 tiles up to two 32x32 tiles a CU
  const long tiles32 = (long)((p.rows_out + 31) / 32) * ((p.cout + 31) / 32);
  const int ts = tiles32 > 512 ? 32 : 16;
  const dim3 grid((p.rows_out + ts - 1) / ts, (p.cout + ts - 1) / ts);
  if (ts == 32)
    hipLaunchKernelGGL((f0_conv_kernel<X, 2>), grid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((f0_conv_kernel<X, 1>), grid, dim3(256), 0, stream, p);
  return hipGetLastError();
}
}  // namespace

hipError_t hift_f0_conv(const HiftConv& p, int x_f32, hipStream_t stream) {
  if (p.rows_out <= 0) return hipSuccess;
  // K in four equal runs of 16-value groups, each inside one tap
  if (!p.docs || p.cin_pad % 16 != 0 || (p.k * p.cin_pad) % 64 != 0 || p.ldx % 4 != 0 ||
      p.stride != 1 || p.dil != 1 || p.up != 1 || !aligned16(p.w))
    return hipErrorInvalidValue;
  return x_f32 ? launch_f0<float>(p, stream) : launch_f0<double>(p, stream);
}

hipError_t hift_f0_head(const double* h, int C, const double* cls_w, const double* cls_b,
                        int rows, float* f0, const HiftDocs* docs, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(f0_head_kernel, dim3(rows), dim3(64), 0, stream, h, C, cls_w, cls_b, f0,
                     docs);
  return hipGetLastError();
}

hipError_t hift_source(const HiftSource& p, const HiftDocs* docs, hipStream_t stream) {
  if (p.docs_cap <= 0) return hipSuccess;
  hipLaunchKernelGGL(source_phase_kernel, dim3(p.docs_cap, p.H), dim3(256), 0, stream, p, docs);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (p.samples_cap <= 0) return hipSuccess;
  hipLaunchKernelGGL(source_sample_kernel, dim3(blocks_for(p.samples_cap, 256)), dim3(256), 0,
                     stream, p, docs);
  return hipGetLastError();
}

hipError_t hift_copy_live(const float* src, float* dst, int rows, const HiftDocs* docs,
                          hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(copy_live_kernel, dim3(blocks_for(rows, 256)), dim3(256), 0, stream, src,
                     dst, docs);
  return hipGetLastError();
}

hipError_t hift_stft(const float* s, const float* window, float* out, int ld, int frames,
                     const HiftDocs* docs, hipStream_t stream) {
  if (frames <= 0) return hipSuccess;
  hipLaunchKernelGGL(stft_kernel, dim3(blocks_for(frames, 256)), dim3(256), 0, stream, s, window,
                     out, ld, docs);
  return hipGetLastError();
}

hipError_t hift_istft(const float* y, int ldy, const float* window, float* fr, float* out,
                      float limit, int frames, int samples, const HiftDocs* docs,
                      hipStream_t stream) {
  if (frames > 0) {
    hipLaunchKernelGGL(istft_frame_kernel, dim3(blocks_for(frames, 256)), dim3(256), 0, stream, y,
                       ldy, window, fr, docs);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (samples <= 0) return hipSuccess;
  hipLaunchKernelGGL(istft_ola_kernel, dim3(blocks_for(samples, 256)), dim3(256), 0, stream, fr,
                     window, out, limit, docs);
  return hipGetLastError();
}

}  // namespace fcv
