// The HiFT vocoder's causal fp32 convolutions on the f16 matrix cores, at fp32 accuracy.
//
// Every operand is held as a sum of two f16 values, x = hi + lo, scaled by a power of two so that the
// largest finite magnitude lies in [2^14, 2^15): a weight row by its own largest weight (once, when
// the weights are packed), the inputs by the largest of the 32 channels of one row that a chunk
// takes.  Values down to 2^-17 of the largest keep 22 significant bits, smaller ones an absolute error
// of 2^-39 of it.  A product is lo hi + hi lo + hi hi on v_mfma_f32_32x32x16_f16; a step's sum (32
// channels of one tap) starts from zero, and is taken back to the row's scale as it is added to the
// fp32 running sum.  So an output depends on the inputs it reads and on nothing else, as on the fp32
// kernels: not on what else is in its document, later or louder, or on the tile.
// Against 64-bit results the waveform's relative error is 9.4e-6 (8 requests) where
// v_mfma_f32_16x16x4_f32 left 2.6e-5: the operands' rounding adds 1.7e-6, and sums of 16 products at a
// time round less often than sums of 4.  Where one conv's input channels lie up to 2^16 apart, its
// weights the other way, it stays at 9.6e-6; 2^24 apart it is 7.5e-5 (the fp32 form 2.7e-5).
//
// Bound: three f16 MFMAs do a product's work at 16 times the fp32 form's rate each, so the ceiling
// is a third of the f16 peak against the fp32 peak of 157 TFLOP/s.  Measured on one MI355X against
// v_mfma_f32_16x16x4_f32 (hift.hip): 8 requests of 3065 frames 22.6 -> 10.2 ms (91 -> 202 TFLOP/s of
// fp32 work over the whole call), one 68-frame chunk 2.31 -> 0.77 ms (with the small form below and
// launches shared by independent convolutions).  One scale per document in place of one per row and
// chunk was 10.1 and 0.79 ms, but took precision from every row quieter than the loudest.  The large
// form fits its 128 registers only just: seven spilled ones put a wait for every copy into its loop
// (11.0 ms), so the tile's row table stays in LDS.
// What is left of a large launch is latency: the document table, window and residual reads around
// 14 to 88 steps of MFMAs, and LDS reads (1.3 KB per MFMA in the 64x64 tile).  128x128 and 64x256
// tiles (half the weight copies, twice the registers) were no faster, nor were weights loaded straight
// into registers, which needs no barrier between steps.
//
// A workgroup owns TR output rows x TC output channels.  For each 32 input channels it splits a
// window of input rows (the tile's rows and the left context) into LDS once, then walks the taps
// over it: the input is read and split once, not once per tap.  A tap's weights are one
// contiguous block of the packed table, copied straight to LDS (global_load_lds) through a ring
// of NS stages.  Channel chunks outermost (in groups, see kGroups), then taps, then k-steps, then
// the three products: the order of every output's sum is the same in every tile shape, so results
// do not depend on the shape a launch takes.  (Compiled without floating-point contraction, as the
// rounding of an output must not depend on the instantiation either.)
#include <algorithm>
#include <cstdlib>

#include "hift.hpp"
#include "hift_device.hpp"

namespace fcv {
namespace {

constexpr int kRowBytes = 128;  // one row of 32 channels: 4 chunks of hi, 4 of lo, 16 bytes each
constexpr int kMaxHalo = 62;    // largest left context of a tile, in rows
// 64x64 tiles in a launch (all its convolutions, at the call's own rows) under which the small form
// runs.  One call, all small, all 64x64, and by this rule, ms: 24 frames 0.67, 1.11, 0.67; 40 0.73,
// 1.11, 0.73; 68 0.87, 1.12, 0.77; 100 1.03, 1.15, 0.91; 200 1.64, 1.44, 1.25; 286 2.23, 1.66, 1.56;
// 600 4.27, 2.54, 2.53.  (By the capacity's rows, 64 frames at least, 24 frames took 0.74.)
constexpr long kSmallBelow = 256;

// position of 16-byte chunk `chunk` in LDS row `row`: 16 consecutive rows read at one chunk index
// hit 16 distinct 16-byte bank groups
__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// every LDS access of this wave has completed
__device__ __forceinline__ void wait_lgkm0() {
  __builtin_amdgcn_s_waitcnt(0xF | (0x7 << 4) | (0x3 << 14));
}

// |v| as its bits, which order like the values; 0 where v is infinite or NaN
__device__ __forceinline__ uint32_t finite_bits(float v) {
  const uint32_t a = __float_as_uint(v) & 0x7FFFFFFFu;
  return a < 0x7F800000u ? a : 0u;
}
// The scale that brings the magnitude of bits `m` into [2^14, 2^15), as a float's exponent field (that
// of 1 for zero; magnitudes below 2^-86 are raised by 2^100 only)
__device__ __forceinline__ int scale_field(uint32_t m) {
  return m == 0 ? 127 : min(max(268 - (int)(m >> 23), 14), 227);
}
__device__ __forceinline__ float field_to_float(int f) { return __uint_as_float((uint32_t)f << 23); }

// the largest of four bit patterns and those of the other seven lanes of an aligned group of eight
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_max(uint32_t v) {
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xF, 0xF, true));
}
__device__ __forceinline__ uint32_t max_of8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  uint32_t m = max(max(a, b), max(c, d));
  m = dpp_max<0xB1>(m);      // quad_perm [1, 0, 3, 2]
  m = dpp_max<0x4E>(m);      // quad_perm [2, 3, 0, 1]
  return dpp_max<0x141>(m);  // row_half_mirror
}
// A step's sum times this is in units of the weights' scale over 2^15 (kUnscale), in which the weights
// are below 1: the running sum overflows no earlier than the inputs times their number
constexpr float kUnscale = 32768.0f;
__device__ __forceinline__ float step_scale(int field) { return field_to_float(254 - 15 - field); }

// An output's sum is taken over groups of consecutive chunks, each from zero, the groups added in
// order: at most kGroups of group_chunks(chunks).  A small launch gives each group a wave.
constexpr int kGroups = 4;
__device__ __forceinline__ int group_chunks(int chunks) { return (chunks + kGroups - 1) / kGroups; }

// Four values, scaled, as their f16 halves.  A value that is not finite goes into lo alone: beside an
// infinite hi, the other operand's lo, zero or of the other sign, would make NaN of its products.
__device__ __forceinline__ void split4(const f32x4& v, float s, f16x4& hi, f16x4& lo) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float x = v[e] * s;
    const f16 h = (f16)x;
    const bool finite = fabsf(x) <= 3.402823466e38f;
    hi[e] = finite ? h : (f16)0.0f;
    lo[e] = (f16)(finite ? x - (float)h : x);
  }
}

// Splits four values of a window row, whose 32 channels eight lanes hold, and returns the row's scale
// field.  Values that are not finite take the longer way, a wave at a time.
__device__ __forceinline__ int split_row(const f32x4& v, f16x4& hi, f16x4& lo) {
  constexpr uint32_t kAbs = 0x7FFFFFFFu;
  const uint32_t m = max_of8(__float_as_uint(v[0]) & kAbs, __float_as_uint(v[1]) & kAbs,
                             __float_as_uint(v[2]) & kAbs, __float_as_uint(v[3]) & kAbs);
  if (__ballot(m >= 0x7F800000u) != 0) {
    const int field = scale_field(max_of8(finite_bits(v[0]), finite_bits(v[1]), finite_bits(v[2]),
                                          finite_bits(v[3])));
    split4(v, field_to_float(field), hi, lo);
    return field;
  }
  const int field = scale_field(m);
  const float s = field_to_float(field);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float x = v[e] * s;
    hi[e] = (f16)x;
    lo[e] = (f16)(x - (float)hi[e]);
  }
  return field;
}

__device__ __forceinline__ f32x4 load4(const void* q, long i) {
  return *reinterpret_cast<const f32x4*>(static_cast<const float*>(q) + i);
}

// an epilogue's per-channel inputs (the packed ones are padded with zeros to co_pad channels)
struct SplitCols {
  f32x4 bias, winv, alpha, inv_alpha, alpha2, inv_alpha2;
  __device__ __forceinline__ void load(const HiftConv& p, int c) {
    winv = load4(p.winv, c);
    bias = load4(p.winv, p.co_pad + c);
    if (p.snake_out) {
      alpha = load4(p.alpha, c);
      inv_alpha = load4(p.inv_alpha, c);
    }
    if (p.n_snakes) {
      alpha2 = load4(p.snakes[0].alpha, c);
      inv_alpha2 = load4(p.snakes[0].inv_alpha, c);
    }
  }
};

// the rows an epilogue adds to channels c .. c + 3 of output row `row`
struct SplitAdds {
  f32x4 add, acc;
  __device__ __forceinline__ void load(const HiftConv& p, long row, int c) {
    if (p.add) add = load4(p.add, row * p.ld_add + c);
    if (p.mode != HIFT_ACC_WRITE) acc = load4(p.accin, row * p.ldo + c);
  }
};

// the epilogue of channels c .. c + 3 of one row: unscale, bias, residual, resblock sum, Snakes
__device__ __forceinline__ void split_store(const HiftConv& p, const SplitCols& cols,
                                            const SplitAdds& in, long row, int c, const f32x4& acc) {
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = fmaf(acc[e] * cols.winv[e], kUnscale, cols.bias[e]);
  const long i = row * p.ldo + c;
  if (p.add) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = v[e] + in.add[e];
  }
  if (p.mode != HIFT_ACC_WRITE) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = in.acc[e] + v[e];
    if (p.mode == HIFT_ACC_ADD_DIV) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] / p.div;
    }
  }
  if (p.snake_out) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = snake(v[e], cols.alpha[e], cols.inv_alpha[e]);
  }
  *reinterpret_cast<f32x4*>(static_cast<float*>(p.out) + i) = v;
  if (p.n_snakes) {
    f32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = snake(v[e], cols.alpha2[e], cols.inv_alpha2[e]);
    *reinterpret_cast<f32x4*>(p.snakes[0].out + i) = w;
#pragma unroll
    for (int n = 1; n < 4; ++n) {
      if (n >= p.n_snakes) break;
      const f32x4 a = load4(p.snakes[n].alpha, c), ia = load4(p.snakes[n].inv_alpha, c);
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = snake(v[e], a[e], ia[e]);
      *reinterpret_cast<f32x4*>(p.snakes[n].out + i) = w;
    }
  }
}

// The document of a tile's first row, looked up in one round of loads of the table (documents
// past 63: searched in memory).
struct TileDocs {
  int n_docs, rows_out, in_total, d0, in0, out0, out1;
  // false: the tile starts past the live rows
  __device__ __forceinline__ bool load(const HiftDocs* __restrict__ docs, int r0, int lane) {
    n_docs = docs->n;
    const int ta = docs->a[lane], tb = docs->b[lane];
    if (n_docs < 64) {
      rows_out = __builtin_amdgcn_readlane(tb, n_docs);
      in_total = __builtin_amdgcn_readlane(ta, n_docs);
      if (r0 >= rows_out) return false;
      d0 = __builtin_popcountll(__ballot(lane < n_docs && tb <= r0)) - 1;
      in0 = __builtin_amdgcn_readlane(ta, d0);
      out0 = __builtin_amdgcn_readlane(tb, d0);
      out1 = __builtin_amdgcn_readlane(tb, d0 + 1);
    } else {
      rows_out = docs->b[n_docs];
      in_total = docs->a[n_docs];
      if (r0 >= rows_out) return false;
      d0 = doc_of(docs->b, n_docs, r0);
      in0 = docs->a[d0];
      out0 = docs->b[d0];
      out1 = docs->b[d0 + 1];
    }
    return true;
  }
};

// WC x WR waves; each wave MC x MR tiles of 32 channels x 32 rows.  NS weight stages, NI passes of
// window loads (kThreads / 8 rows each).
template <int WC_, int WR_, int MC_, int MR_, int NS_, int NI_>
struct Cfg {
  static constexpr int WC = WC_, WR = WR_, MC = MC_, MR = MR_, NS = NS_, NI = NI_;
  static constexpr int kWaves = WC * WR, kThreads = 64 * kWaves;
  static constexpr int TC = 32 * MC * WC, TR = 32 * MR * WR;
  static constexpr int kWin = NI * kThreads / 8;             // window rows
  static constexpr int kWBytes = TC * kRowBytes;             // one weight stage
  static constexpr int kCopies = kWBytes / 1024 / kWaves;    // weight copies per wave and step
  static constexpr int kXOff = NS * kWBytes;
  static constexpr int kInfoOff = kXOff + (kWin + 1) * kRowBytes;  // + the zero row
  static constexpr int kPitch = 32 * MC + 4;                 // staged epilogue row, in floats
  static constexpr int kStage = 32 * kPitch * 4;             // per wave
  static constexpr int kRemOff = kInfoOff + TR * 16;
  static constexpr int kScaleOff = kRemOff + TR * 4;
  static constexpr int kLds = kScaleOff + (kWin + 1) * 4;
  static constexpr int kMinWaves = kThreads < 256 ? 1 : NI <= 3 ? 4 : 3;  // per SIMD
  static_assert(kWBytes % (1024 * kWaves) == 0, "weight copies");
  static_assert(kStage * kWaves <= kInfoOff, "the epilogue stages in the operand space");
};

template <class C>
__global__ __launch_bounds__(C::kThreads, C::kMinWaves) void split_conv_kernel(
    const HiftJobs jobs) {
  const HiftConv& p = jobs.c[blockIdx.z];
  const HiftDocs* __restrict__ docs = p.docs;
  __shared__ __attribute__((aligned(1024))) char smem[C::kLds];
  char* sX = smem + C::kXOff;
  // per tile row: window row of tap 0, position, document and the window row of the document's first
  // input row, before which a tap reads zeros; then tap 0's remainder (up > 1); then each window
  // row's step_scale
  int4* sInfo = reinterpret_cast<int4*>(smem + C::kInfoOff);
  int* sRem = reinterpret_cast<int*>(smem + C::kRemOff);
  float* sScale = reinterpret_cast<float*>(smem + C::kScaleOff);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave % C::WC, wr = wave / C::WC;
  const int li = lane & 31, hl = lane >> 5;
  const int r0 = blockIdx.x * C::TR;
  TileDocs td;
  if (!td.load(docs, r0, lane)) return;
  const int n_docs = td.n_docs, rows_out = td.rows_out, in_total = td.in_total;
  const int d0 = td.d0, in0 = td.in0, out0 = td.out0, out1 = td.out1;
  const bool one_doc = min(r0 + C::TR, rows_out) <= out1;  // of the tile's rows
  const int co0 = blockIdx.y * C::TC;
  if (co0 >= p.cout) return;
  const int chunks = p.cin_pad / 32;
  const int k = p.k, up = p.up, dil = p.dil;  // (read once: the copies below may write memory)

  // weight copies: step (chunk, tap) is a contiguous block of co_pad rows
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;
  const char* wnext = static_cast<const char*>(p.wsplit) + (long)co0 * kRowBytes;
  const long wstep = (long)p.co_pad * kRowBytes;
  const uint32_t wlane = (uint32_t)(wave * C::kCopies * 1024 + lane * 16);
  const int steps = chunks * k;
  auto issue_w = [&](int stage) {
    const char* src = wnext;
    wnext += wstep;
    const uint32_t dst = lds0 + (uint32_t)stage * C::kWBytes + wave * C::kCopies * 1024;
#pragma unroll
    for (int i = 0; i < C::kCopies; ++i) lds_dma16(src, wlane + i * 1024, dst + i * 1024);
  };

#pragma unroll
  for (int s = 0; s < C::NS - 1; ++s)
    if (s < steps) issue_w(s);

  // the window starts at the first input row any tap of the tile's first row reads
  const int u0 = r0 - out0 - p.pad;
  const int win0 = in0 + (u0 > 0 ? u0 / up : 0);
  for (int t = tid; t < C::TR; t += C::kThreads) {
    const int r = r0 + t;
    int4 v{-(1 << 29), -1, d0, 0};  // rows past the end read the zero row at every tap
    int rem = 0;
    if (r < rows_out) {
      const int d = one_doc ? d0 : doc_of(docs->b, n_docs, r);
      const int base = (one_doc ? in0 : docs->a[d]) - win0;
      v.y = r - (one_doc ? out0 : docs->b[d]);
      v.z = d;
      v.w = max(base, 0);
      int q = v.y - p.pad;
      if (up > 1) {
        const int u = q;
        q = u >= 0 ? u / up : -((-u + up - 1) / up);
        rem = u - q * up;
      }
      v.x = base + q;
    }
    sInfo[t] = v;
    sRem[t] = rem;
  }
  if (tid == 0) sScale[C::kWin] = 1.0f;
  if (tid < 8) *reinterpret_cast<f32x4*>(sX + C::kWin * kRowBytes + tid * 16) = f32x4{0, 0, 0, 0};

  // window loads: pass i, thread tid -> window row i * kThreads / 8 + tid / 8, channels 4 (tid % 8)
  const char* X = reinterpret_cast<const char*>(static_cast<const float*>(p.x) + (long)win0 * p.ldx);
  // (rows of a window past the tile's own may belong to another document: nothing reads them)
  const float slope = p.pro == HIFT_PRO_LEAKY ? p.slope : 1.0f;  // (x 1 is x)
  uint32_t xoff[C::NI];  // bytes from the window's first row
#pragma unroll
  for (int i = 0; i < C::NI; ++i)
    xoff[i] = min(i * (C::kThreads / 8) + (tid >> 3), in_total - 1 - win0) * p.ldx * 4 +
              (tid & 7) * 16;
  f32x4 xr[C::NI];
  auto fetch_x = [&](int c) {
#pragma unroll
    for (int i = 0; i < C::NI; ++i) xr[i] = *reinterpret_cast<const f32x4*>(X + c * 128 + xoff[i]);
  };
  auto stash_x = [&]() {
#pragma unroll
    for (int i = 0; i < C::NI; ++i) {
      f32x4 v = xr[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.0f ? v[e] : v[e] * slope;
      f16x4 hi, lo;
      const int field = split_row(v, hi, lo);
      const int row = i * (C::kThreads / 8) + (tid >> 3);
      if ((tid & 7) == 0) sScale[row] = step_scale(field);
      char* dst = sX + row * kRowBytes + (tid & 1) * 8;
      *reinterpret_cast<f16x4*>(dst + 16 * swz(row, (tid & 7) >> 1)) = hi;
      *reinterpret_cast<f16x4*>(dst + 16 * swz(row, 4 + ((tid & 7) >> 1))) = lo;
    }
  };

  // the step at hand, the sum of the chunk group at hand, and of the groups before it
  f32x16 acc[C::MC][C::MR], group[C::MC][C::MR], total[C::MC][C::MR];
#pragma unroll
  for (int a = 0; a < C::MC; ++a)
#pragma unroll
    for (int b = 0; b < C::MR; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) group[a][b][e] = total[a][b][e] = 0.0f;
  const int per_group = group_chunks(chunks);
  auto end_group = [&]() {
#pragma unroll
    for (int a = 0; a < C::MC; ++a)
#pragma unroll
      for (int b = 0; b < C::MR; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          total[a][b][e] = total[a][b][e] + group[a][b][e];
          group[a][b][e] = 0.0f;
        }
  };

  fetch_x(0);
  __syncthreads();  // the row table
  // Two fragment buffers: the reads of k-step ks + 1 are in flight while the MFMAs of ks run.  A
  // step's second k-step runs after the barrier that publishes the next step, over that step's
  // first reads.  A weight block of 32 channels is 4 KB: k-steps 0 and 1, hi then lo, lane l's 16
  // bytes at 16 l.  In an input row the 16-byte chunk of k-step ks (hi, then lo) sits at byte
  // (16 (hl ^ rot)) ^ 32 ks (^ 64 for lo), rot = (row / 2) % 8.
  f16x8 wh[2][C::MC], wl[2][C::MC], xh[2][C::MR], xl[2][C::MR];
  const uint32_t woff = wc * C::MC * 4096 + lane * 16;
  uint32_t xoff_l[C::MR];
  auto load = [&](int buf, int ks, const char* sW) {
#pragma unroll
    for (int a = 0; a < C::MC; ++a) {
      wh[buf][a] = *reinterpret_cast<const f16x8*>(sW + woff + a * 4096 + ks * 2048);
      wl[buf][a] = *reinterpret_cast<const f16x8*>(sW + woff + a * 4096 + ks * 2048 + 1024);
    }
#pragma unroll
    for (int b = 0; b < C::MR; ++b) {
      xh[buf][b] = *reinterpret_cast<const f16x8*>(sX + (xoff_l[b] ^ (32 * ks)));
      xl[buf][b] = *reinterpret_cast<const f16x8*>(sX + (xoff_l[b] ^ (32 * ks + 64)));
    }
  };
  // a k-step's products, on the sums `from`
  auto mma = [&](int buf, const f32x16 (&from)[C::MC][C::MR]) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int a = 0; a < C::MC; ++a)
#pragma unroll
      for (int b = 0; b < C::MR; ++b) acc[a][b] = mfma32(wl[buf][a], xh[buf][b], from[a][b]);
#pragma unroll
    for (int a = 0; a < C::MC; ++a)
#pragma unroll
      for (int b = 0; b < C::MR; ++b) acc[a][b] = mfma32(wh[buf][a], xl[buf][b], acc[a][b]);
#pragma unroll
    for (int a = 0; a < C::MC; ++a)
#pragma unroll
      for (int b = 0; b < C::MR; ++b) acc[a][b] = mfma32(wh[buf][a], xh[buf][b], acc[a][b]);
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x16 zero[C::MC][C::MR];
#pragma unroll
  for (int a = 0; a < C::MC; ++a)
#pragma unroll
    for (int b = 0; b < C::MR; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) zero[a][b][e] = 0.0f;
  float scale[C::MR];  // of the step at hand
  // a finished step joins its group
  auto fold = [&]() {
#pragma unroll
    for (int a = 0; a < C::MC; ++a)
#pragma unroll
      for (int b = 0; b < C::MR; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          group[a][b][e] = fmaf(acc[a][b][e], scale[b], group[a][b][e]);
  };

  int s = 0, stage_s = 0, in_group = 0;
  for (int c = 0; c < chunks; ++c) {
    int wrow[C::MR], first[C::MR], rem[C::MR];  // this lane's rows
#pragma unroll
    for (int b = 0; b < C::MR; ++b) {
      const int t = (wr * C::MR + b) * 32 + li;
      wrow[b] = sInfo[t].x;
      first[b] = sInfo[t].w;
      rem[b] = sRem[t];
    }
    if (c > 0) {
      // Every wave has read the previous window: a barrier alone does not wait for a wave's reads
      // in flight, and the window is written right after it.
      wait_lgkm0();
      __syncthreads();
      mma(1, acc);
      fold();
      if (++in_group == per_group) {
        end_group();
        in_group = 0;
      }
    }
    stash_x();
    for (int j = 0; j < k; ++j, ++s) {
      // this wave's copies of step s have landed (the later steps' may be in flight), then everyone's
      if (s + C::NS - 2 < steps)
        wait_vm<(C::NS - 2) * C::kCopies>();
      else
        wait_vm<0>();
      wait_lgkm0();  // and this wave's reads of the stage the next copies overwrite
      __syncthreads();
      if (s + C::NS - 1 < steps) issue_w(stage_s == 0 ? C::NS - 1 : stage_s - 1);
      if (j == 0 && c + 1 < chunks) fetch_x(c + 1);

      const char* sW = smem + stage_s * C::kWBytes;
      stage_s = stage_s == C::NS - 1 ? 0 : stage_s + 1;
      float next[C::MR];
#pragma unroll
      for (int b = 0; b < C::MR; ++b) {
        const int row = wrow[b] >= first[b] && wrow[b] < C::kWin ? wrow[b] : C::kWin;
        next[b] = sScale[row];
        xoff_l[b] = row * kRowBytes + 16 * (hl ^ ((row >> 1) & 7));
        // next tap's input row
        if (up > 1) {
          rem[b] += 1;
          const int step = rem[b] == up ? 1 : 0;
          rem[b] = step ? 0 : rem[b];
          wrow[b] += step;
        } else {
          wrow[b] += dil;
        }
      }
      load(0, 0, sW);
      if (j > 0) mma(1, acc);
      load(1, 1, sW);
      if (j > 0) fold();
      mma(0, zero);
#pragma unroll
      for (int b = 0; b < C::MR; ++b) scale[b] = next[b];
    }
  }
  mma(1, acc);
  fold();
  end_group();
  constexpr int LPR = 8 * C::MC;              // lanes per staged output row
  const int cl = (lane % LPR) * 4;            // channel within the wave's columns
  const int c4 = co0 + wc * C::MC * 32 + cl;
  const bool live_c = c4 < p.cout;
  SplitCols cols;
  cols.load(p, live_c ? c4 : 0);
  wait_vm<0>();
  wait_lgkm0();
  __syncthreads();  // the operand space becomes the waves' staging space

  // Epilogue: lane l holds row l % 32 and, in register group g, channels 8 g + 4 (l / 32) + 0..3.
  // Each wave stages 32 rows at a time and reads them back row-major, so loads and stores are
  // whole 128-byte (256-byte) runs of a row.
  float* stage = reinterpret_cast<float*>(smem + wave * C::kStage);
  constexpr int RPI = 64 / LPR, NP = 32 / RPI;  // rows a pass, passes
#pragma unroll
  for (int b = 0; b < C::MR; ++b) {
    const int t0 = (wr * C::MR + b) * 32 + lane / LPR;
    SplitAdds in[NP];  // in flight while the block is staged (out may be the residual itself)
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int t = t0 + i * RPI;
      if (r0 + t < rows_out && live_c)
        in[i].load(p, p.reflect ? (long)r0 + t + sInfo[t].z + 1 : r0 + t, c4);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int a = 0; a < C::MC; ++a)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 v{total[a][b][4 * g], total[a][b][4 * g + 1], total[a][b][4 * g + 2],
                      total[a][b][4 * g + 3]};
        *reinterpret_cast<f32x4*>(stage + li * C::kPitch + a * 32 + g * 8 + hl * 4) = v;
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int t = t0 + i * RPI;
      const int r = r0 + t;
      if (r >= rows_out || !live_c) continue;
      const f32x4 v = *reinterpret_cast<const f32x4*>(stage + (i * RPI + lane / LPR) * C::kPitch + cl);
      const int4 info = sInfo[t];
      const long row = p.reflect ? (long)r + info.z + 1 : r;
      split_store(p, cols, in[i], row, c4, v);
      // reflection padding (1, 0): row 0 of the document repeats the result's row 1
      if (p.reflect && info.y == 1) {
        SplitAdds first;
        first.load(p, (long)r - 1 + info.z, c4);
        split_store(p, cols, first, (long)r - 1 + info.z, c4, v);
      }
    }
  }
}

// The small launches' form: a workgroup owns one 32x32 tile, and each of its kGroups waves sums one
// group of input chunks, on its own window and with its weights loaded straight into registers PD
// steps ahead: no wave waits for another until the sums are added.  A step here is latency, some
// 900 cycles around 192 of MFMAs with one wave on a SIMD (counters of a 68-frame chunk), so the
// shorter chain is what counts.
template <int NI, int PD>
__global__ __launch_bounds__(64 * kGroups, 1) void split_conv_small_kernel(const HiftJobs jobs) {
  constexpr int kWin = NI * 8, kWinBytes = kWin * kRowBytes, kPitch = 36;
  constexpr int kStage = 32 * kPitch * 4;  // a group's 32x32 sums
  constexpr int kScaleOff = kWinBytes + kRowBytes;  // each window row's step_scale, the zero row's too
  constexpr int kOperands = kScaleOff + (kWin + 4) * 4;
  constexpr int kPart = kOperands > kStage ? kOperands : kStage;
  const HiftConv& p = jobs.c[blockIdx.z];
  const HiftDocs* __restrict__ docs = p.docs;
  __shared__ __attribute__((aligned(1024))) char smem[kGroups * kPart];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, hl = lane >> 5;
  const int r0 = blockIdx.x * 32, co0 = blockIdx.y * 32;
  TileDocs td;
  if (!td.load(docs, r0, lane)) return;
  if (co0 >= p.cout) return;
  const bool one_doc = min(r0 + 32, td.rows_out) <= td.out1;
  const int chunks = p.cin_pad / 32, k = p.k, up = p.up, dil = p.dil;
  const int per_group = group_chunks(chunks);
  const int c_begin = wave * per_group, c_end = min(c_begin + per_group, chunks);
  char* win = smem + wave * kPart;
  float* scales = reinterpret_cast<float*>(win + kScaleOff);

  const int u0 = r0 - td.out0 - p.pad;
  const int win0 = td.in0 + (u0 > 0 ? u0 / up : 0);

  if (c_begin < c_end) {
    const char* wbase = static_cast<const char*>(p.wsplit) + (long)(co0 / 32) * 4096;
    const long wstep = (long)p.co_pad * kRowBytes;
    const int s_end = c_end * k;
    f16x8 w[PD][4];
    auto fetch_w = [&](f16x8 (&f)[4], int s) {
      const char* src = wbase + (long)min(s, s_end - 1) * wstep;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        f[i] = *reinterpret_cast<const f16x8*>(src + lane * 16 + i * 1024);
    };
#pragma unroll
    for (int i = 0; i < PD - 1; ++i) fetch_w(w[i], c_begin * k + i);

    // window pass i, lane l: row 8 i + l / 8, channels 4 (l % 8)
    const float* X = static_cast<const float*>(p.x) + (long)win0 * p.ldx + (lane & 7) * 4;
    const float slope = p.pro == HIFT_PRO_LEAKY ? p.slope : 1.0f;  // (x 1 is x)
    int xoff[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) xoff[i] = min(i * 8 + (lane >> 3), td.in_total - 1 - win0) * p.ldx;
    f32x4 xr[NI];
    auto fetch_x = [&](int c) {
#pragma unroll
      for (int i = 0; i < NI; ++i) xr[i] = *reinterpret_cast<const f32x4*>(X + xoff[i] + c * 32);
    };
    auto stash_x = [&]() {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        f32x4 v = xr[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.0f ? v[e] : v[e] * slope;
        f16x4 hi, lo;
        const int field = split_row(v, hi, lo);
        const int row = i * 8 + (lane >> 3);
        if ((lane & 7) == 0) scales[row] = step_scale(field);
        char* dst = win + row * kRowBytes + (lane & 1) * 8;
        *reinterpret_cast<f16x4*>(dst + 16 * swz(row, (lane & 7) >> 1)) = hi;
        *reinterpret_cast<f16x4*>(dst + 16 * swz(row, 4 + ((lane & 7) >> 1))) = lo;
      }
    };
    fetch_x(c_begin);
    // the wave's zero row, and this lane's row: window row and input position of tap 0
    if (lane == 0) scales[kWin] = 1.0f;
    if (lane < 8) *reinterpret_cast<f32x4*>(win + kWinBytes + lane * 16) = f32x4{0, 0, 0, 0};
    int q0 = -(1 << 29), rem0 = 0, wrow0 = 0;
    if (r0 + li < td.rows_out) {
      const int d = one_doc ? td.d0 : doc_of(docs->b, td.n_docs, r0 + li);
      const int u = r0 + li - (one_doc ? td.out0 : docs->b[d]) - p.pad;
      q0 = u;
      if (up > 1) {
        q0 = u >= 0 ? u / up : -((-u + up - 1) / up);
        rem0 = u - q0 * up;
      }
      wrow0 = (one_doc ? td.in0 : docs->a[d]) - win0 + q0;
    }
    stash_x();
    if (c_begin + 1 < c_end) fetch_x(c_begin + 1);

    // the group's sum; the last step's, which is folded behind the next one's MFMAs, and its scale
    f32x16 group, done;
#pragma unroll
    for (int e = 0; e < 16; ++e) group[e] = done[e] = 0.0f;
    float scale = 0.0f;
    auto fold = [&]() {
#pragma unroll
      for (int e = 0; e < 16; ++e) group[e] = fmaf(done[e], scale, group[e]);
    };
    int q = q0, rem = rem0, wrow = wrow0, c = c_begin, j = 0;
    for (int s0 = c_begin * k; s0 < s_end; s0 += PD) {
#pragma unroll
      for (int u = 0; u < PD; ++u) {
        if (s0 + u >= s_end) break;
        if (j == k) {  // the next chunk's window (LDS accesses of one wave stay in order)
          j = 0;
          ++c;
          q = q0; rem = rem0; wrow = wrow0;
          stash_x();
          if (c + 1 < c_end) fetch_x(c + 1);
        }
        fetch_w(w[(u + PD - 1) % PD], s0 + u + PD - 1);
        const bool ok = q >= 0 && (unsigned)wrow < (unsigned)kWin;
        const int row = ok ? wrow : kWin;
        const uint32_t off = row * kRowBytes + 16 * (hl ^ ((row >> 1) & 7));
        const float next = scales[row];
        if (up > 1) {
          rem += 1;
          const int step = rem == up ? 1 : 0;
          rem = step ? 0 : rem;
          q += step;
          wrow += step;
        } else {
          q += dil;
          wrow += dil;
        }
        ++j;
        f32x16 acc;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const f16x8 xh = *reinterpret_cast<const f16x8*>(win + (off ^ (32 * ks)));
          const f16x8 xl = *reinterpret_cast<const f16x8*>(win + (off ^ (32 * ks + 64)));
          acc = mfma32(w[u][2 * ks + 1], xh, acc);
          acc = mfma32(w[u][2 * ks], xl, acc);
          acc = mfma32(w[u][2 * ks], xh, acc);
        }
        fold();
        done = acc;
        scale = next;
      }
    }
    fold();
    // the sums go where the window was: this wave has read it
    float* stage = reinterpret_cast<float*>(win);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 v{group[4 * g], group[4 * g + 1], group[4 * g + 2], group[4 * g + 3]};
      *reinterpret_cast<f32x4*>(stage + li * kPitch + g * 8 + hl * 4) = v;
    }
  }

  // eight rows a wave, eight lanes a row
  constexpr int kRows = 32 / kGroups;
  const int t = wave * kRows + (lane >> 3), r = r0 + t, cl = (lane & 7) * 4, c4 = co0 + cl;
  const bool live = r < td.rows_out && c4 < p.cout;
  SplitCols cols;
  SplitAdds in;
  int d = td.d0, pos = 0;
  long row = r;
  if (live) {
    if (!one_doc) d = doc_of(docs->b, td.n_docs, r);
    pos = r - (one_doc ? td.out0 : docs->b[d]);
    if (p.reflect) row = (long)r + d + 1;
    cols.load(p, c4);
    in.load(p, row, c4);
  }
  wait_lgkm0();
  __syncthreads();
  if (!live) return;
  f32x4 v{0, 0, 0, 0};
  for (int g = 0; g * per_group < chunks; ++g)
    v += *reinterpret_cast<const f32x4*>(smem + g * kPart + (t * kPitch + cl) * 4);
  split_store(p, cols, in, row, c4, v);
  // reflection padding (1, 0): row 0 of the document repeats the result's row 1
  if (p.reflect && pos == 1) {
    SplitAdds first;
    first.load(p, (long)r - 1 + d, c4);
    split_store(p, cols, first, (long)r - 1 + d, c4, v);
  }
}

// One wave per output channel of [co_pad][k][cin] weights: the row's scale from its largest finite
// weight, then both halves in the order the kernels' fragments take them; inv[co] = the inverse scale,
// inv[co_pad + co] = the bias (zero past cout).
__global__ __launch_bounds__(64) void pack_split_kernel(const float* __restrict__ w,
                                                        const float* __restrict__ bias, int cout,
                                                        int co_pad, int k, int cin,
                                                        f16* __restrict__ dst,
                                                        float* __restrict__ inv) {
  const int co = blockIdx.x, lane = threadIdx.x;
  const float* row = w + (long)co * k * cin;
  const int n = k * cin;
  uint32_t m = 0;
  for (int i = lane; i < n; i += 64) m = max(m, finite_bits(row[i]));
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
  const int f = scale_field(m);
  const float s = field_to_float(f);
  if (lane == 0) {
    inv[co] = field_to_float(254 - f);
    inv[co_pad + co] = co < cout ? bias[co] : 0.0f;
  }
  for (int i = lane; i < n / 4; i += 64) {
    const int tap = i * 4 / cin, c = i * 4 - tap * cin;
    f16x4 hi, lo;
    split4(*reinterpret_cast<const f32x4*>(row + i * 4), s, hi, lo);
    // [step][32-channel block][k-step][hi, lo][lane][8]: lane = co % 32 + 32 ((c / 8) % 2)
    f16* out = dst + (((long)(c / 32) * k + tap) * co_pad + (co & ~31)) * 64 +
               ((c >> 4) & 1) * 1024 + ((co & 31) + 32 * ((c >> 3) & 1)) * 8 + (c & 4);
    *reinterpret_cast<f16x4*>(out) = hi;
    *reinterpret_cast<f16x4*>(out + 512) = lo;
  }
}

bool aligned16(const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; }

template <class C>
hipError_t launch(const HiftJobs& jobs, int n, int rows, int cout, hipStream_t stream) {
  static_assert(C::kLds <= 160 * 1024, "LDS");
  const dim3 grid((rows + C::TR - 1) / C::TR, (cout + C::TC - 1) / C::TC, n);
  hipLaunchKernelGGL(split_conv_kernel<C>, grid, dim3(C::kThreads), 0, stream, jobs);
  return hipGetLastError();
}

// input rows a tile of TR output rows reads: its rows and the left context
int window_rows(const HiftConv& p, int tr) {
  return (tr - 1) / p.up + 2 + ((p.k - 1) * p.dil + p.up - 1) / p.up;
}

// the shape with the window passes the launch's widest window needs
template <int WC, int WR, int MC, int MR, int NS, int P1, int P2, int P3>
hipError_t launch_win(const HiftJobs& jobs, int n, int rows, int cout, hipStream_t stream) {
  int need = 0;
  for (int i = 0; i < n; ++i) need = std::max(need, window_rows(jobs.c[i], 32 * MR * WR));
  const int per = 8 * WC * WR;
  if (need <= P1 * per) return launch<Cfg<WC, WR, MC, MR, NS, P1>>(jobs, n, rows, cout, stream);
  if (need <= P2 * per) return launch<Cfg<WC, WR, MC, MR, NS, P2>>(jobs, n, rows, cout, stream);
  if (need <= P3 * per) return launch<Cfg<WC, WR, MC, MR, NS, P3>>(jobs, n, rows, cout, stream);
  return hipErrorInvalidValue;
}

// the small form with the window passes (8 rows each) the launch needs
template <int NI>
hipError_t launch_small_ni(const HiftJobs& jobs, int n, int rows, int cout, hipStream_t stream) {
  const dim3 grid((rows + 31) / 32, (cout + 31) / 32, n);
  hipLaunchKernelGGL((split_conv_small_kernel<NI, 4>), grid, dim3(64 * kGroups), 0, stream, jobs);
  return hipGetLastError();
}
hipError_t launch_small(const HiftJobs& jobs, int n, int rows, int cout, hipStream_t stream) {
  int need = 0;
  for (int i = 0; i < n; ++i) need = std::max(need, window_rows(jobs.c[i], 32));
  if (need <= 4 * 8) return launch_small_ni<4>(jobs, n, rows, cout, stream);
  if (need <= 8 * 8) return launch_small_ni<8>(jobs, n, rows, cout, stream);
  if (need <= 12 * 8) return launch_small_ni<12>(jobs, n, rows, cout, stream);
  return hipErrorInvalidValue;
}

bool launchable(const HiftConv& p) {
  if (!hift_split_eligible(p) || !p.docs || !p.wsplit || !p.winv ||
      p.co_pad % 64 != 0 || p.ldx % 4 != 0 || p.ldo % 4 != 0 || (p.add && p.ld_add % 4 != 0) ||
      !aligned16(p.x) || !aligned16(p.out) || !aligned16(p.add) || !aligned16(p.accin) ||
      !aligned16(p.wsplit) || !aligned16(p.winv) || (long)p.co_pad * kRowBytes >= (1L << 31) ||
      p.n_snakes < 0 || p.n_snakes > 4)
    return false;
  for (int i = 0; i < p.n_snakes; ++i)
    if (!aligned16(p.snakes[i].out)) return false;
  // channels go four at a time: a partial last group writes zeros into the row's padding and has
  // no other row or parameter to read
  return p.cout % 4 == 0 || ((p.cout + 3) / 4 * 4 <= p.ldo && !p.add && !p.snake_out &&
                             !p.n_snakes && p.mode == HIFT_ACC_WRITE);
}

}  // namespace

bool hift_split_eligible(const HiftConv& p) {
  return p.stride == 1 && p.cin_pad % 32 == 0 && p.up >= 1 && p.dil >= 1 &&
         (p.up == 1 || p.dil == 1) && p.pad == (p.k - 1) * p.dil && p.pad <= kMaxHalo &&
         (p.pro == HIFT_PRO_NONE || (p.slope >= -1.0f && p.slope <= 1.0f));
}

size_t hift_split_bytes(int co_pad, int k, int cin) {
  return (size_t)(cin / 32) * k * co_pad * kRowBytes;
}

hipError_t hift_pack_split(const float* w, const float* bias, int cout, int co_pad, int k, int cin,
                           void* dst, float* inv, hipStream_t stream) {
  hipLaunchKernelGGL(pack_split_kernel, dim3(co_pad), dim3(64), 0, stream, w, bias, cout, co_pad, k,
                     cin, static_cast<f16*>(dst), inv);
  return hipGetLastError();
}

hipError_t hift_conv_split(const HiftConv* convs, int n, hipStream_t stream) {
  if (n < 1 || n > kHiftJobs) return hipErrorInvalidValue;
  HiftJobs jobs{};
  int rows = 0, cout = 0;
  long tiles64 = 0;
  for (int i = 0; i < n; ++i) {
    if (!launchable(convs[i])) return hipErrorInvalidValue;
    jobs.c[i] = convs[i];
    rows = std::max(rows, convs[i].rows_out);
    cout = std::max(cout, convs[i].cout);
    tiles64 += (long)((convs[i].rows_live + 63) / 64) * ((convs[i].cout + 63) / 64);
  }
  if (rows <= 0) return hipSuccess;
  // FCV_HIFT_TILE = 32 or 64 forces a tile: a test hook, both must give the same bits
  const char* forced = std::getenv("FCV_HIFT_TILE");
  const int force = forced ? std::atoi(forced) : 0;
  const bool small = force ? force == 32 : tiles64 < kSmallBelow;
  if (small) return launch_small(jobs, n, rows, cout, stream);
  if (cout <= 32) return launch_win<1, 4, 1, 1, 3, 2, 5, 6>(jobs, n, rows, cout, stream);
  return launch_win<2, 2, 1, 1, 3, 2, 3, 4>(jobs, n, rows, cout, stream);
}

}  // namespace fcv
