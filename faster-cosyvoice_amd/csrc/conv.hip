// Causal grouped conv1d + Mish (CausalConvPositionEmbedding) as an implicit GEMM on MFMA.
//
// Per (row tile, group g of 64 channels):
//   y[r, co] = mish(bias[co] + sum_{j<taps} sum_{ci<64} W[g][j][co][ci] * x[r - (taps-1) + j, ci])
// The tile's input rows and the taps - 1 before them are staged in LDS once for the group's 64
// channels; every tap j reads the same window shifted by j rows, so no im2col buffer exists.  Packed
// documents are handled per row: the input fragment of output row r at tap j is zeroed when the
// input row lies before r's document start, i.e. when pos[r] + j < taps - 1 (the per-document left
// zero padding of the reference's F.pad).
//
// An output's sum runs over the taps in order, in one chain, in both forms, so results do not depend on
// the form a launch takes.  A launch of few rows is bound by one workgroup's chain of taps on a part of
// the CUs (48 of 256 at 300 rows with 128-row tiles), a large one by the LDS reads of its MFMAs.
// Hence a form of 32 rows a tile, whose waves walk their taps without a barrier, while its workgroups
// are at most one per CU, and one of 128.  A forward of one block holds two launches and took on one
// MI355X (us, at 16 channel groups):
//   rows                                 60    300   500   520   600   700   800   1000  1040
//   this rule                            92    98    106   120   122   130   127   136   142
//   32 rows to twice as many workgroups                    125   127   135   132   138
//   64 rows, two row tiles a workgroup                     123   124   132   130   136
//   128 rows throughout, the channel groups on the grid's slow axis (the only form once)
//                                        103   111   118   120         129         136   144
// Two chains of half the taps each, added at the end, were faster by 1 us below 512 rows and by 6 up to
// 1024, but round differently from one chain.
#include "kernels.hpp"

namespace fcv {
namespace {

constexpr int CG = 64;        // channels per group
constexpr int LDP = CG + 8;   // padded LDS row (f16): 16 consecutive rows hit distinct banks
constexpr int MAX_TAPS = 31;
constexpr int SPITCH = CG + 4;  // fp32 staging row
constexpr int W_BYTES = 2 * CG * LDP * 2;
constexpr int STAGE_BYTES = 4 * 32 * SPITCH * 4;

constexpr int kCUs = 256;

// one output element group of the epilogue: mish(v + bias) to f16, or added to the residual's row
__device__ __forceinline__ void conv_finish(const f32x4& v, const float4& b, const float4& hv,
                                            long at, f16* out_f16, float* h) {
  const float4 y = {mish(v[0] + b.x), mish(v[1] + b.y), mish(v[2] + b.z), mish(v[3] + b.w)};
  if (h)
    *reinterpret_cast<float4*>(h + at) = float4{hv.x + y.x, hv.y + y.y, hv.z + y.z, hv.w + y.w};
  else
    *reinterpret_cast<f16x4*>(out_f16 + at) = f2h4(y.x, y.y, y.z, y.w);
}

// 4 waves x 32 output rows x 64 output channels.  Each tap's 64x64 weight slice streams through an
// LDS double buffer.  (64 rows a wave, for 1 KB of LDS read per MFMA and not 1.5, measured no faster
// from 1100 rows up: two workgroups of 128 rows on a CU hide each other's taps, one of 256 has
// nothing beside it.)  MFMA 32x32x16 with the weights as the A operand, so lane l accumulates output
// row l % 32 and, in register group g of channel tile t, channels 32 t + 8 g + 4 (l / 32) + 0..3.
// The epilogue stages each wave's 32 x 64 block through LDS and reads it back row-major (16 lanes per
// row), so stores are contiguous runs of 128 B (f16 out) or 256 B (fp32 residual); the residual form
// issues all its h loads before its first store.
__global__ __launch_bounds__(256, 2) void conv_kernel(const f16* __restrict__ x, int C,
                                                      const f16* __restrict__ w,
                                                      const float* __restrict__ bias, int taps,
                                                      const int32_t* __restrict__ pos, int rows,
                                                      f16* __restrict__ out_f16,
                                                      float* __restrict__ h,
                                                      const int32_t* __restrict__ rows_live) {
  constexpr int TM = 128;
  constexpr int X_BYTES = (TM + MAX_TAPS - 1) * LDP * 2;
  constexpr int SMEM_BYTES = X_BYTES + W_BYTES > STAGE_BYTES ? X_BYTES + W_BYTES : STAGE_BYTES;
  __shared__ __attribute__((aligned(16))) unsigned char smem[SMEM_BYTES];
  f16 (*sX)[LDP] = reinterpret_cast<f16 (*)[LDP]>(smem);
  f16 (*sW)[CG][LDP] = reinterpret_cast<f16 (*)[CG][LDP]>(smem + X_BYTES);

  if (rows_live) rows = *rows_live;  // live rows of a capacity-sized grid
  const int m0 = blockIdx.y * TM;
  if (m0 >= rows) return;
  const int g = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int halo = taps - 1;

  // stage the input window rows [m0 - halo, m0 + TM) of group g
  const int chunk_c = (tid & 7) * 8;
  for (int r = tid >> 3; r < TM + halo; r += 32) {
    int src = min(max(m0 - halo + r, 0), rows - 1);
    *reinterpret_cast<f16x8*>(&sX[r][chunk_c]) =
        *reinterpret_cast<const f16x8*>(x + (long)src * C + g * CG + chunk_c);
  }

  const f16* wg = w + (long)g * taps * CG * CG;
  const int lw_r = tid >> 3;  // 0..31
  auto fetch = [&](f16x8 (&rw)[2], int j) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      rw[i] = *reinterpret_cast<const f16x8*>(wg + ((long)j * CG + lw_r + 32 * i) * CG + chunk_c);
  };
  auto stash = [&](const f16x8 (&rw)[2], int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<f16x8*>(&sW[buf][lw_r + 32 * i][chunk_c]) = rw[i];
  };

  // output row of this lane (B operand row) and its document position
  const int fr = lane & 31, fh = lane >> 5;
  const int lrow = wave * 32 + fr;
  const int lpos = pos[min(m0 + lrow, rows - 1)];
  const int col_lane = (lane & 15) * 4;  // epilogue: 4 channels of one row per lane
  const float4 bias4 = *reinterpret_cast<const float4*>(bias + g * CG + col_lane);

  f32x16 acc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[t][e] = 0.0f;
  const f16x8 zero8 = {};
  auto tap = [&](int j, int buf) {
    // rows before the row's document start read as zero (per-document causal padding)
    const bool live = lpos + j >= halo;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const f16x8 v = *reinterpret_cast<const f16x8*>(&sX[lrow + j][ks * 16 + fh * 8]);
      const f16x8 xb = live ? v : zero8;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const f16x8 wa = *reinterpret_cast<const f16x8*>(&sW[buf][t * 32 + fr][ks * 16 + fh * 8]);
        acc[t] = mfma32(wa, xb, acc[t]);
      }
    }
  };
  // Weights run two taps ahead of the MFMAs: tap j+1's slice (loaded during tap j-1) is stashed
  // while tap j+2's loads are in flight, so a stash never waits on loads issued in its own tap
  // (a workgroup alone on its CU would otherwise wait out a load round trip every tap).  Taps
  // past the last re-read the last slice, so every path issues the same loads.
  f16x8 ra[2], rb[2];
  fetch(ra, 0);
  stash(ra, 0);
  fetch(ra, min(1, taps - 1));
  __syncthreads();
  for (int j = 0; j < taps; j += 2) {
    fetch(rb, min(j + 2, taps - 1));
    __builtin_amdgcn_sched_barrier(0);
    tap(j, 0);
    stash(ra, 1);
    __syncthreads();
    if (j + 1 < taps) {
      fetch(ra, min(j + 3, taps - 1));
      __builtin_amdgcn_sched_barrier(0);
      tap(j + 1, 1);
      stash(rb, 0);
      __syncthreads();
    }
  }

  // epilogue (the loop's last barrier freed the window and weight buffers)
  float* stage = reinterpret_cast<float*>(smem) + wave * 32 * SPITCH;
  const int col = g * CG + col_lane;
  const int row0 = m0 + wave * 32;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<f32x4*>(stage + fr * SPITCH + t * 32 + q * 8 + fh * 4) = f32x4{
          acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  f32x4 v[8];
  float4 hv[8];
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const int r = p * 4 + (lane >> 4);
    v[p] = *reinterpret_cast<const f32x4*>(stage + r * SPITCH + col_lane);
    const int row = min(row0 + r, rows - 1);
    if (h) hv[p] = *reinterpret_cast<const float4*>(h + (long)row * C + col);
  }
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const int row = row0 + p * 4 + (lane >> 4);
    if (row < rows) conv_finish(v[p], bias4, hv[p], (long)row * C + col, out_f16, h);
  }
}

// The small launches' form: a workgroup owns 32 rows x 64 channels and each of its two waves a 32x32
// tile of them, with the weights straight from global memory three taps ahead (five or seven ahead
// were 1 us slower), so no wave waits for another between the window and the epilogue.
__global__ __launch_bounds__(128, 1) void conv_small_kernel(
    const f16* __restrict__ x, int C, const f16* __restrict__ w, const float* __restrict__ bias,
    int taps, const int32_t* __restrict__ pos, int rows, f16* __restrict__ out_f16,
    float* __restrict__ h, const int32_t* __restrict__ rows_live) {
  constexpr int TM = 32;
  constexpr int X_BYTES = (TM + MAX_TAPS - 1) * LDP * 2;
  constexpr int SUM_BYTES = TM * SPITCH * 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[X_BYTES > SUM_BYTES ? X_BYTES
                                                                                 : SUM_BYTES];
  f16 (*sX)[LDP] = reinterpret_cast<f16 (*)[LDP]>(smem);
  float (*sum)[SPITCH] = reinterpret_cast<float (*)[SPITCH]>(smem);

  if (rows_live) rows = *rows_live;  // live rows of a capacity-sized grid
  const int m0 = blockIdx.y * TM;
  if (m0 >= rows) return;
  const int g = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int fr = lane & 31, fh = lane >> 5;
  const int halo = taps - 1;

  // this wave's first taps' weights: fragment ks of lane l is channel 32 wave + l % 32, inputs
  // 16 ks + 8 (l / 32) + 0..7
  constexpr int PD = 4;
  static_assert(PD % 2 == 0, "a tap's fragment buffer follows its place in the unrolled loop");
  f16x8 wr[PD][4];
  const f16* wg = w + ((long)g * taps * CG + wave * 32 + fr) * CG + fh * 8;
  auto fetch = [&](f16x8 (&f)[4], int j) {
    const f16* src = wg + (long)min(j, taps - 1) * CG * CG;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) f[ks] = *reinterpret_cast<const f16x8*>(src + ks * 16);
  };
#pragma unroll
  for (int u = 0; u < PD - 1; ++u) fetch(wr[u], u);

  const int chunk_c = (tid & 7) * 8;
  for (int r = tid >> 3; r < TM + halo; r += 16) {
    const int src = min(max(m0 - halo + r, 0), rows - 1);
    *reinterpret_cast<f16x8*>(&sX[r][chunk_c]) =
        *reinterpret_cast<const f16x8*>(x + (long)src * C + g * CG + chunk_c);
  }
  const int lpos = pos[min(m0 + fr, rows - 1)];
  // the epilogue's 16 rows a wave, four channels of 4 rows a lane
  const int tr = wave * 16 + (lane >> 4), col_lane = (lane & 15) * 4, col = g * CG + col_lane;
  const float4 bias4 = *reinterpret_cast<const float4*>(bias + col);
  float4 hv[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int row = min(m0 + tr + 4 * p, rows - 1);
    if (h) hv[p] = *reinterpret_cast<const float4*>(h + (long)row * C + col);
  }
  __syncthreads();

  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
  // tap j's input fragments; rows before the row's document start read as zero (per-document causal
  // padding).  They are read a tap ahead, as the weights are fetched PD - 1 ahead.
  f16x8 xb[2][4];
  auto read = [&](f16x8 (&f)[4], int j) {
    const bool live = lpos + j >= halo;
    const f16x8 zero8 = {};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const f16x8 v = *reinterpret_cast<const f16x8*>(&sX[fr + j][ks * 16 + fh * 8]);
      f[ks] = live ? v : zero8;
    }
  };
  read(xb[0], 0);
  for (int jb = 0; jb < taps; jb += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      const int j = jb + u;
      if (j >= taps) break;
      fetch(wr[(u + PD - 1) % PD], j + PD - 1);
      read(xb[(u + 1) & 1], min(j + 1, taps - 1));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) acc = mfma32(wr[u][ks], xb[u & 1][ks], acc);
    }
  }
  __syncthreads();  // every wave has read the window: the sums take its place
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<f32x4*>(&sum[fr][wave * 32 + q * 8 + fh * 4]) =
        f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  __syncthreads();
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int r = tr + 4 * p, row = m0 + r;
    const f32x4 v = *reinterpret_cast<const f32x4*>(&sum[r][col_lane]);
    if (row < rows) conv_finish(v, bias4, hv[p], (long)row * C + col, out_f16, h);
  }
}

}  // namespace

hipError_t conv_causal_mish(const f16* x, int C, const f16* w, const float* bias, int taps,
                            const int32_t* pos, int rows, f16* out_f16, float* h,
                            hipStream_t stream, const int32_t* rows_live) {
  if (rows <= 0) return hipSuccess;
  if (taps < 1 || taps > MAX_TAPS || C % CG != 0) return hipErrorInvalidValue;
  // Channel groups are the grid's fast axis: consecutive workgroups go to the XCDs in turn, so an XCD
  // holds the weights of C/CG / 8 groups in its L2 and reads each once, not all of them.
  // The rule is on the launch's capacity, so that a captured launch and its replays take one form.
  const int groups = C / CG;
  const auto tiles = [&](int tm) { return (rows + tm - 1) / tm; };
  if (tiles(32) * groups <= kCUs)
    hipLaunchKernelGGL(conv_small_kernel, dim3(groups, tiles(32)), dim3(128), 0, stream, x, C, w, bias,
                       taps, pos, rows, out_f16, h, rows_live);
  else
    hipLaunchKernelGGL(conv_kernel, dim3(groups, tiles(128)), dim3(256), 0, stream, x, C, w, bias, taps,
                       pos, rows, out_f16, h, rows_live);
  return hipGetLastError();
}

}  // namespace fcv
