// Qwen3.5 hybrid text step on the GPU: the engine's float arithmetic
// (crates/coheryn-engine/src/qwen35/execution.rs:257-608, qwen35/kernels.rs:
// 11-269, cpu.rs:31-35,74-124): its f32 products, glibc expf and log1pf
// restated (exp_f32, log1p_f32), no contraction.  The conv, the attention
// scores and the softmax recurrences run in the reference's element order.  The
// f64 sums of the linears, the norms, the gates' q/k squares and the delta rule
// are split over lanes and waves where the reference runs one chain: the same
// bits unless a partial sum rounds in f64 and the difference crosses an f32
// rounding boundary.  Their orders are fixed by the model's shape, so a lane's
// results depend neither on the rows and lanes beside it nor on how its tokens
// are cut into steps.
//
// Layout: activations are row-major f32 per packed row; matrices are BF16
// tiles of 16 outputs (q35_tiled_index); the sequence state lives in slabs
// indexed by sequence slot: K/V rows of the full-attention layers, the
// causal-conv ring and the delta-rule memory of the linear layers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "device.h"
#include "gemm.h"
#include "log1pf.h"
#include "q35.h"

namespace cohx {
namespace {

typedef unsigned int u32x4q __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// kernels.rs:11-24
__device__ __forceinline__ float sigmoid_f32(float x) {
  if (x >= 0.0f) return 1.0f / (1.0f + exp_f32(-x));
  const float e = exp_f32(x);
  return e / (1.0f + e);
}
__device__ __forceinline__ float silu_f32(float x) { return x * sigmoid_f32(x); }
// The same with expf's table staged in LDS (per-lane reads).
__device__ __forceinline__ float sigmoid_f32(float x, const uint64_t *tab) {
  const float e = exp_f32_tab(-fabsf(x), tab);
  return x >= 0.0f ? 1.0f / (1.0f + e) : e / (1.0f + e);
}
__device__ __forceinline__ float silu_f32(float x, const uint64_t *tab) { return x * sigmoid_f32(x, tab); }
__device__ __forceinline__ float softplus_f32(float x, const uint64_t *tab) {
  return fmaxf(x, 0.0f) + log1p_f32(exp_f32_tab(-fabsf(x), tab));
}
__device__ __forceinline__ float softplus_f32(float x) {
  return fmaxf(x, 0.0f) + log1p_f32(exp_f32(-fabsf(x)));
}

// ---------------------------------------------------------------------------
// Token embedding (tensor.rs read_row over BF16: exact widening).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_q35_embed(const uint16_t *__restrict__ embed,
                                                   const uint32_t *__restrict__ tokens, int H,
                                                   float *__restrict__ x) {
  const int r = blockIdx.x;
  const uint16_t *src = embed + (size_t)tokens[r] * H;
  for (int i = threadIdx.x; i < H; i += 256) x[(size_t)r * H + i] = bf_lo(src[i]);
}

// ---------------------------------------------------------------------------
// Norm (kernels.rs:26-52): mean of f32 squares summed in f64, scale =
// 1/sqrt(f32(mean) + eps), y = (x*scale)*(w + zc).  Each thread sums its
// elements (256 apart) in order, then a fixed tree over the workgroup, where
// the reference runs one chain: both round at 2^-53 of the sum, before the
// mean is rounded to f32.  One lane adding 1,024 squares in order took 8.4 us
// of latency a launch (59 us at 4,104 rows); the tree takes 4.8 (8.7).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_q35_norm(const float *__restrict__ x, int ldx,
                                                  const uint32_t *__restrict__ src,
                                                  const float *__restrict__ w, int n, float eps,
                                                  int zc, float *__restrict__ out, int ldo,
                                                  uint32_t *row_err,
                                                  const uint32_t *__restrict__ err_row) {
  __shared__ double red[4];
  const int r = blockIdx.x;
  const float *xr = x + (size_t)(src ? src[r] : r) * ldx;
  bool bad = false;
  // the first kHeld elements per thread (n <= 1024) keep x and the weight in
  // registers across the sum, so the scaling pass issues no loads
  constexpr int kHeld = 4;
  float xv[kHeld], wv[kHeld];
#pragma unroll
  for (int c = 0; c < kHeld; c++) {
    const int i = threadIdx.x + c * 256;
    xv[c] = i < n ? xr[i] : 0.0f;
    wv[c] = i < n ? w[i] : 0.0f;
  }
  double ss = -0.0;
#pragma unroll
  for (int c = 0; c < kHeld; c++)
    if ((int)threadIdx.x + c * 256 < n) {
      ss += (double)(xv[c] * xv[c]);
      bad |= !finitef(xv[c]);
    }
  for (int i = threadIdx.x + kHeld * 256; i < n; i += 256) {
    const float v = xr[i];
    ss += (double)(v * v);
    bad |= !finitef(v);
  }
  const double mean = block_sum_f64<256>(ss, red) / (double)n;
  bad |= !(__builtin_isfinite(mean) && finitef((float)mean));
  const float scale = 1.0f / sqrtf((float)mean + eps), add = zc ? 1.0f : 0.0f;
#pragma unroll
  for (int c = 0; c < kHeld; c++) {
    const int i = threadIdx.x + c * 256;
    if (i < n) {
      const float y = (xv[c] * scale) * (wv[c] + add);
      out[(size_t)r * ldo + i] = y;
      bad |= !finitef(y);
    }
  }
  for (int i = threadIdx.x + kHeld * 256; i < n; i += 256) {
    const float y = (xr[i] * scale) * (w[i] + add);
    out[(size_t)r * ldo + i] = y;
    bad |= !finitef(y);
  }
  if (bad) atomicOr(&row_err[err_row ? err_row[r] : r], kErrRequest);
}

// ---------------------------------------------------------------------------
// BF16 matvec (tensor.rs:380-406 -> cpu::dot): out[r][o] = f32(sum_k
// f64(f32(w[o][k] * x[r][k]))).  A workgroup owns one tile of 16 outputs x kR
// rows.  Chunk c of 64 inputs is of class c % 8: eight waves take a class each,
// four waves the two classes w and w + 4.  Within a chunk each 16-lane row of
// the wave takes 16 inputs: lane l brings the weights of output l % 16 (two
// 16-byte loads, coalesced in the tile layout).  The rows' inputs pass through
// a strip of LDS of the wave's own (256 contiguous bytes a row, no barrier: a
// wave's LDS operations stay in order) and come back as 16-byte broadcasts.
//   The order of the sums: a chain per class and 16-lane row, class c + class
// c + 4, then those by class and row.  It is the same in every instance, so an
// output does not depend on the rows beside it.  The reference adds the
// products in one chain; they are f32 values of 24 bits, so a partial f64 sum
// rounds only where a product is 2^-29 of it or smaller, by 2^-53 of its size,
// before the dot is rounded to f32.
//   What bounds it: vector issue, an f32 multiply, a widening and an f64 add
// per product, 4.6 ns a wave and SIMD, issued as pinned groups of products,
// widenings and adds over four or eight rows (left alone, the compiler sends
// every triple through one temporary and each add waits for its widening;
// taking the inputs from the lanes by DPP, without LDS, cost 5.9 ns).  One
// chain per output left a decode step waiting on 1,024 to 3,584 dependent adds
// in every linear.  Sixteen rows are held to 128 registers, four waves a SIMD
// (head at 16 rows 330 us; 352 with 154 registers and three waves).
//   kQ35Swiglu: gate tile blockIdx.x and up tile blockIdx.x + up_off / 16
// (up_off passed in valid_rows, F in ldo's place as the output count) over the
// same inputs; h = (g / (1 + exp(-g))) * u (the SwiGLU pass's expression) to
// out [R][F].
//   Measured at 16 rows (us a launch, one chain per output before): o 7.3 and
// down 10.0 (22.4 each), mix 17.1 (22.2), gate+up 15.0 (18.3), head 330 (343);
// o and down at 96 rows 28 on average (228).
// ---------------------------------------------------------------------------
template <int kEpi, int kR, int kW, bool kTail>
__global__ __launch_bounds__(64 * kW, kR == 16 && kEpi != kQ35Swiglu && !kTail ? 4 : 1) void k_q35_mv(
    const uint16_t *__restrict__ w, int valid_rows, int K, const float *__restrict__ x, int ldx, int R, float *out,
    int ldo, unsigned long long *__restrict__ part, uint32_t *row_err, const uint32_t *__restrict__ err_row) {
  constexpr bool kGlu = kEpi == kQ35Swiglu;
  constexpr int kTiles = kGlu ? 2 : 1;
  __shared__ double s_sum[kW][kTiles][kR][kWave];
  static_assert(sizeof(float) * kR * kWave <= sizeof(s_sum[0]), "the wave's input strip");
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  float *strip = reinterpret_cast<float *>(s_sum[wave]);  // [kR][64], until the sums take its place
  const int o16 = lane % 16, koff = 16 * (lane / 16);
  const int tile = blockIdx.x, r0 = blockIdx.y * kR, nc = (K + 63) / 64;
  const u32x4q *wt[kTiles];
  wt[0] = reinterpret_cast<const u32x4q *>(w) + (size_t)tile * (K / 8) * 16 + o16;
  if constexpr (kGlu) wt[1] = wt[0] + (size_t)(valid_rows / 16) * (K / 8) * 16;
  const float *xr[kR];
#pragma unroll
  for (int r = 0; r < kR; r++) xr[r] = x + (size_t)min(r0 + r, R - 1) * ldx;  // rows past R: unused
  constexpr int kA = 8 / kW;  // classes of chunks per wave
  double sums[kA][kTiles][kR];
#pragma unroll
  for (int k = 0; k < kA; k++)
#pragma unroll
    for (int m = 0; m < kTiles; m++)
#pragma unroll
      for (int r = 0; r < kR; r++) sums[k][m][r] = -0.0;
  struct Step {
    u32x4q w[kTiles][2];
    float x[kR];
  };
  // branch-free: chunks past the last load it again (unused); inputs past K
  // (kTail: K not a multiple of 64) become weight +0 and input -0, whose
  // product -0 changes no sum
  auto load = [&](Step &st, int c) {
    const int k = 64 * min(c, nc - 1) + koff;
#pragma unroll
    for (int m = 0; m < kTiles; m++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const bool in = !kTail || k + 8 * i < K;
        st.w[m][i] = wt[m][(size_t)(in ? k / 8 + i : 0) * 16];
        if (!in) st.w[m][i] = u32x4q{0u, 0u, 0u, 0u};
      }
#pragma unroll
    for (int r = 0; r < kR; r++) {
      const int kx = 64 * min(c, nc - 1) + lane;
      const bool in = !kTail || kx < K;
      st.x[r] = xr[r][in ? kx : 0];
      if (!in) st.x[r] = -0.0f;
    }
  };
  auto use = [&](const Step &st, double (&acc)[kTiles][kR]) {
#pragma unroll
    for (int r = 0; r < kR; r++) strip[r * kWave + lane] = st.x[r];
    constexpr int kG = kR == 8 ? 8 : 4;
#pragma unroll
    for (int q = 0; q < 4; q++) {  // inputs 4 q .. + 3 of the lane's 16
      float wf[kTiles][4];
#pragma unroll
      for (int m = 0; m < kTiles; m++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
          wf[m][2 * i] = bf_lo(st.w[m][q / 2][q % 2 * 2 + i]);
          wf[m][2 * i + 1] = bf_hi(st.w[m][q / 2][q % 2 * 2 + i]);
        }
#pragma unroll
      for (int g = 0; g < kR; g += kG) {
        float4 xv[kG];
#pragma unroll
        for (int r = 0; r < kG; r++) xv[r] = *reinterpret_cast<const float4 *>(strip + (g + r) * kWave + koff + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int m = 0; m < kTiles; m++) {
            float pr[kG];
            double wd[kG];
#pragma unroll
            for (int r = 0; r < kG; r++)
              pr[r] = wf[m][e] * (e == 0 ? xv[r].x : e == 1 ? xv[r].y : e == 2 ? xv[r].z : xv[r].w);
            pin_vgprs(pr);
#pragma unroll
            for (int r = 0; r < kG; r++) wd[r] = (double)pr[r];
            pin_vgprs(wd);
#pragma unroll
            for (int r = 0; r < kG; r++) acc[m][g + r] += wd[r];
          }
      }
      // the sums stay here: sunk past the loop's branch, their terms would
      // all be live at once (512 registers and scratch where K is ragged)
#pragma unroll
      for (int m = 0; m < kTiles; m++) pin_vgprs(acc[m]);
    }
  };
  Step a, b;  // two register sets, one loading while the other is used
  load(a, wave);
  for (int c = wave; c < nc; c += 2 * kW) {
    load(b, c + kW);
    use(a, sums[0]);
    if (c + kW < nc) {
      load(a, c + 2 * kW);
      use(b, sums[kA - 1]);
    }
  }
  // each wave's sums take its own strip's place; the fence keeps its reads of
  // the strip (another type, which the compiler need not order) ahead of them
  asm volatile("" ::: "memory");
#pragma unroll
  for (int m = 0; m < kTiles; m++)
#pragma unroll
    for (int r = 0; r < kR; r++)
      s_sum[wave][m][r][lane] = kA == 1 ? sums[0][m][r] : sums[0][m][r] + sums[kA - 1][m][r];
  __syncthreads();
  for (int idx = wave * kWave + (int)__lane_id(); idx < kR * 16; idx += 64 * kW) {
    const int br = idx / 16, oo = idx % 16, r = r0 + br, o = tile * 16 + oo;
    float v[kTiles];
#pragma unroll
    for (int m = 0; m < kTiles; m++) {
      double sum = -0.0;
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const double part = s_sum[i][m][br][q * 16 + oo];
          sum += kA == 1 ? part + s_sum[i + kW - 4][m][br][q * 16 + oo] : part;
        }
      v[m] = (float)sum;
    }
    bool bad = !finitef(v[0]);
    if constexpr (kGlu) {
      const bool ok = r < R && o < ldo;  // ldo: the output count F
      bad |= !finitef(v[kTiles - 1]);
      if (ok) out[(size_t)r * ldo + o] = (v[0] / (1.0f + exp_f32(-v[0]))) * v[kTiles - 1];
      if (ok && bad) atomicOr(&row_err[r], kErrNonFinite);
    } else {
      const bool ok = r < R && o < valid_rows;
      if constexpr (kEpi == kQ35Argmax) {
        unsigned long long key = ok ? argmax_key(v[0], o) : 0ull;
#pragma unroll
        for (int m = 8; m >= 1; m >>= 1) {
          const unsigned long long other = __shfl_xor(key, m, 16);
          key = other > key ? other : key;
        }
        if (ok && out) out[(size_t)r * ldo + o] = v[0];
        if (r < R && oo == 0) part[(size_t)r * gridDim.x + tile] = key;
      } else if (ok) {
        float *p = out + (size_t)r * ldo + o;
        *p = kEpi == kQ35Residual ? *p + v[0] : v[0];
      }
      if (ok && bad) atomicOr(&row_err[err_row ? err_row[r] : r], kErrNonFinite);
    }
  }
}

// cpu.rs:74-78 swiglu
__global__ __launch_bounds__(256) void k_q35_swiglu(const float *__restrict__ gu, int ldgu, int F,
                                                    int up_off, float *__restrict__ h, int ldh) {
  const int r = blockIdx.y;
  for (int f = blockIdx.x * 256 + threadIdx.x; f < F; f += gridDim.x * 256) {
    const float g = gu[(size_t)r * ldgu + f], u = gu[(size_t)r * ldgu + up_off + f];
    h[(size_t)r * ldh + f] = (g / (1.0f + exp_f32(-g))) * u;
  }
}

// ---------------------------------------------------------------------------
// Causal depthwise conv (kernels.rs:54-120).  An output needs its channel's
// last K inputs only, so a lane's tokens are cut into segments of kConvSeg: a
// workgroup takes 256 channels of one segment, its first taps coming from the
// rows before the segment (from the ring for a lane's first tokens).  The ring
// is in time order, oldest first, from slot position % kernel on, which is the
// reference's slot order (cursor + 1 + i) % kernel after the new input is
// written (every layer steps once per token).  The lane's first segment alone
// reads the ring and, when its tokens are done, leaves the lane's last inputs
// in it.
//   What bounds it: one read and one write of the rows.  One thread per
// channel walking its lane's tokens waited on memory once per eight tokens:
// 332 us a launch at 16 lanes of 64-449 tokens, 64 now (143 with run-time
// widths and expf's table in constant memory).
// ---------------------------------------------------------------------------
constexpr int kMaxConv = 8, kConvSeg = 32;
template <int kK>  // the kernel width, or 0: any up to kMaxConv
__global__ __launch_bounds__(256) void k_q35_conv(Q35Lanes L, const float *__restrict__ mix,
                                                  int ldm, const float *__restrict__ w, int C,
                                                  int K_, float *hist, size_t hist_seq,
                                                  float *__restrict__ out, int ldo,
                                                  uint32_t *row_err) {
  constexpr int kTaps = kK ? kK : kMaxConv;
  const int K = kK ? kK : K_;
  __shared__ uint64_t s_tab[32];
  if (threadIdx.x < 32) s_tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  __syncthreads();
  const int ln = blockIdx.x, ch = blockIdx.y * 256 + threadIdx.x;
  const uint32_t first = L.first[ln], n = L.n[ln], start = L.start[ln];
  const uint32_t seg = blockIdx.z * kConvSeg, end = min(n, seg + kConvSeg);
  if (ch >= C || seg >= n) return;
  float *h = hist + (size_t)L.seq[ln] * hist_seq + (size_t)ch * K;
  const int c0 = (int)(start % (uint32_t)K);
  const float *mc = mix + ch;
  // the K inputs before token seg, oldest first: ring entries (of which the
  // oldest is dropped by the first token) or earlier rows
  static_assert(kConvSeg >= kMaxConv, "a later segment's taps are rows of the lane");
  float tap[kTaps], wv[kTaps];
#pragma unroll
  for (int i = 0; i < kTaps; i++) {
    tap[i] = i >= K ? 0.0f : seg == 0 ? h[(c0 + i) % K] : mc[(size_t)(first + seg - K + i) * ldm];
    wv[i] = i < K ? w[(size_t)ch * K + i] : 0.0f;
  }
  // the inputs load a group of kAhead tokens at a time, the next group
  // requested before the current one is folded in
  constexpr int kAhead = 8;
  float cur[kAhead], nxt[kAhead];
#pragma unroll
  for (int j = 0; j < kAhead; j++) cur[j] = seg + j < end ? mc[(size_t)(first + seg + j) * ldm] : 0.0f;
  for (uint32_t t0 = seg; t0 < end; t0 += kAhead) {
#pragma unroll
    for (int j = 0; j < kAhead; j++) {
      const uint32_t tn = t0 + kAhead + j;
      nxt[j] = tn < end ? mc[(size_t)(first + tn) * ldm] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < kAhead; j++) {
      if (t0 + j >= end) break;
      const uint32_t row = first + t0 + j;
      const float in = cur[j];
#pragma unroll
      for (int i = 0; i < kTaps - 1; i++)
        if (i < K - 1) tap[i] = tap[i + 1];
#pragma unroll
      for (int i = 0; i < kTaps; i++)
        if (i == K - 1) tap[i] = in;
      double sum = -0.0;
#pragma unroll
      for (int i = 0; i < kTaps; i++)
        if (i < K) sum += (double)(tap[i] * wv[i]);
      const float y = silu_f32((float)sum, s_tab);
      out[(size_t)row * ldo + ch] = y;
      if (!finitef(in) || !finitef(y)) atomicOr(&row_err[row], kErrRequest);
    }
#pragma unroll
    for (int j = 0; j < kAhead; j++) cur[j] = nxt[j];
  }
  if (seg != 0) return;
  // the lane's last K inputs: rows, or what is left of the ring before them
  // (n < K, where the lane is this one segment and tap holds them)
  const int c1 = (int)((start + n) % (uint32_t)K);
#pragma unroll
  for (int i = 0; i < kTaps; i++)
    if (i < K) h[(c1 + i) % K] = n >= (uint32_t)K ? mc[(size_t)(first + n - K + i) * ldm] : tap[i];
}

// ---------------------------------------------------------------------------
// Gated delta rule (kernels.rs:122-214) in three passes.
// Gates, per (row, value head): the q/k norms (f64 sums of f32 squares),
// q_scale = (1/sqrt(qn + 1e-6))/sqrt(key_dim), k_scale =
// 1/sqrt(kn + 1e-6), decay = exp(log_decay) with log_decay = -exp(A_log) *
// softplus(a + dt_bias), beta = sigmoid(b) (execution.rs:376-388).
// ---------------------------------------------------------------------------
// One wave per (row, value head), the squares added as a tree over the
// channels, neighbours first (the fused mixer's order): 44 us at 4,104 rows x
// 16 heads, 74 with one lane of a workgroup running the whole sum.
template <int kN>  // over aligned groups of kN lanes, the same bits in each lane
__device__ __forceinline__ double pairs_sum(double v) {
#pragma unroll
  for (int m = 1; m < kN; m <<= 1) v += __shfl_xor(v, m, kWave);
  return v;
}
__global__ __launch_bounds__(256) void k_q35_gates(const float *__restrict__ conv, int ldc,
                                                   int keys, const float *__restrict__ mix,
                                                   int ldm, int a_off, int b_off,
                                                   const float *__restrict__ a_log,
                                                   const float *__restrict__ dt, int KH, int VH,
                                                   int KD, int pairs, float4 *__restrict__ gates,
                                                   uint32_t *row_err) {
  const int pair = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (pair >= pairs) return;
  const int row = pair / VH, h = pair % VH;
  const int src = (h / (VH / KH)) * KD;
  const float *cr = conv + (size_t)row * ldc, *mr = mix + (size_t)row * ldm;
  const float av = mr[a_off + h], bv = mr[b_off + h];
  double q2 = -0.0, k2 = -0.0;
  if (2 * lane < KD) {  // KD <= 128; rows and channel offsets are even
    const float2 q = *reinterpret_cast<const float2 *>(cr + src + 2 * lane);
    const float2 k = *reinterpret_cast<const float2 *>(cr + keys + src + 2 * lane);
    q2 = (double)(q.x * q.x) + (double)(q.y * q.y);
    k2 = (double)(k.x * k.x) + (double)(k.y * k.y);
  }
  const float qn = (float)pairs_sum<kWave>(q2), kn = (float)pairs_sum<kWave>(k2);
  if (lane == 0) {
    const float ld = -exp_f32(a_log[h]) * softplus_f32(av + dt[h]);
    const float beta = sigmoid_f32(bv);
    gates[(size_t)row * VH + h] = make_float4((1.0f / sqrtf(qn + 1e-6f)) / sqrtf((float)KD),
                                              1.0f / sqrtf(kn + 1e-6f), exp_f32(ld), beta);
    if (!finitef(qn) || !finitef(kn) || !finitef(ld) || !finitef(beta) || ld > 0.0f ||
        !(beta >= 0.0f && beta <= 1.0f))
      atomicOr(&row_err[row], kErrRequest);
  }
}

// Sum of v over aligned groups of kP lanes (1, 2, 4 or 8), the same bits in
// each lane: neighbours, then pairs, then fours.
template <int kCtrl>
__device__ __forceinline__ double dpp_f64(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, kCtrl, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), kCtrl, 0xf, 0xf, false);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
template <int kP>
__device__ __forceinline__ double parts_sum(double v) {
  if constexpr (kP >= 2) v += dpp_f64<0xB1>(v);   // quad_perm [1,0,3,2]
  if constexpr (kP >= 4) v += dpp_f64<0x4E>(v);   // quad_perm [2,3,0,1]
  if constexpr (kP >= 8) v += dpp_f64<0x141>(v);  // row_half_mirror
  return v;
}

// The recurrence over prompt chunks.  kP lanes own one state column, 16 keys
// each (in registers across the lane's tokens); a workgroup of 256 threads
// owns 256 / kP columns of one (lane, value head).  Per token the cells decay,
// the prediction sum_i f64(cell * k_i*k_scale) runs in key order from +0.0
// within each lane's 16 keys and over the lanes in a fixed tree, corr =
// (v_j - f32(pred)) * beta, then the cells take k_i*k_scale*corr and the read
// sum_i f64(cell * q_i*q_scale) gives the head's raw output.  (The reference
// runs each f64 sum as one chain, kernels.rs:122-214.  Its terms are f32
// products of 24 bits, so a partial sum rounds only where a term is 2^-29 of
// it or smaller, by 2^-53 of its size, before the sum is rounded to f32.)
//   What bounds it: vector issue, five f32 and four f64 operations a cell and
// token (about 0.9 us a token and CU at full rate).  One thread per column,
// two waves a CU, took 3.0 us a token; sixteen waves a CU cover the
// operations' latencies.  The key vectors, values and gates of kT tokens are
// staged in LDS at a time, the next kT requested while they are used, so there
// is one barrier per kT tokens.  Workgroups of one column group start at
// another lane (blockIdx.z), so a CU's share mixes long and short lanes.
// Measured at 16 lanes of 64-449 tokens: 1,345 -> 444 us a launch.
template <int kKD>
__global__ __launch_bounds__(256) void k_q35_delta(Q35Lanes L, const float *__restrict__ conv,
                                                   int ldc, int keys,
                                                   const float4 *__restrict__ gates, int KH,
                                                   int VH, int VD, float *state, size_t state_seq,
                                                   float *__restrict__ o_out, int ldo,
                                                   uint32_t *row_err) {
  constexpr int kP = kKD / 16, kC = 256 / kP;  // lanes per column, columns per workgroup
  constexpr int kT = 8;                        // tokens per stage
  constexpr int kSK = 2 * kKD * kT / 256, kSV = kC * kT / 256;  // staged key and value words per thread
  // keys as [quad][lane of the column][4]: the kP lanes of a column read
  // consecutive 16-byte words
  __shared__ __align__(16) float s_k[2][kT][kKD], s_q[2][kT][kKD], s_v[2][kT][kC];
  __shared__ float4 s_g[2][kT];
  const int tid = threadIdx.x, h = blockIdx.y;
  const int nl = gridDim.x, ln = (int)(blockIdx.x + blockIdx.z * (nl / gridDim.z)) % nl;
  const uint32_t first = L.first[ln], n = L.n[ln];
  if (!n) return;
  const int src = (h / (VH / KH)) * kKD, j0 = blockIdx.z * kC;
  const int part = tid % kP, c = tid / kP, j = j0 + c;
  const bool active = j < VD;
  float *S = state + (size_t)L.seq[ln] * state_seq + (size_t)h * kKD * VD + (active ? j : 0);
  float col[16];
#pragma unroll
  for (int i = 0; i < 16; i++) col[i] = active ? S[(size_t)(16 * part + i) * VD] : 0.0f;
  // word e = tid + 256 i of a stage's keys: token e / (2 kKD), then q and k channels
  float rk[kSK], rs[kSK], rv[kSV];
  float4 rg = make_float4(0.f, 0.f, 0.f, 0.f);
  auto fetch = [&](uint32_t t0) {
#pragma unroll
    for (int i = 0; i < kSK; i++) {
      const int e = tid + 256 * i, t = e / (2 * kKD), ch = e % (2 * kKD);
      const size_t row = first + min(t0 + t, n - 1);
      rk[i] = conv[row * ldc + (ch < kKD ? src + ch : keys + src + ch - kKD)];
      const float4 &g = gates[row * VH + h];
      rs[i] = ch < kKD ? g.x : g.y;
    }
#pragma unroll
    for (int i = 0; i < kSV; i++) {
      const int e = tid + 256 * i, t = e / kC, cc = e % kC;
      const size_t row = first + min(t0 + t, n - 1);
      rv[i] = j0 + cc < VD ? conv[row * ldc + 2 * keys + h * VD + j0 + cc] : 0.0f;
    }
    if (tid < kT) rg = gates[(size_t)(first + min(t0 + tid, n - 1)) * VH + h];
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < kSK; i++) {
      const int e = tid + 256 * i, t = e / (2 * kKD), ch = e % (2 * kKD), k = ch % kKD;
      const int at = ((k % 16 / 4) * kP + k / 16) * 4 + k % 4;
      (ch < kKD ? s_q : s_k)[buf][t][at] = rk[i] * rs[i];
    }
#pragma unroll
    for (int i = 0; i < kSV; i++) {
      const int e = tid + 256 * i;
      s_v[buf][e / kC][e % kC] = rv[i];
    }
    if (tid < kT) s_g[buf][tid] = rg;
  };
  fetch(0);
  stash(0);
  __syncthreads();
  int buf = 0;
  for (uint32_t t0 = 0; t0 < n; t0 += kT) {
    const bool more = t0 + kT < n;
    if (more) fetch(t0 + kT);
    const int nt = (int)min((uint32_t)kT, n - t0);
    for (int t = 0; t < nt; t++) {
      const float4 gt = s_g[buf][t];
      const float v = s_v[buf][t][c], decay = gt.z, beta = gt.w;
      float kk[16], qq[16];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float4 a = *reinterpret_cast<const float4 *>(&s_k[buf][t][(u * kP + part) * 4]);
        const float4 b = *reinterpret_cast<const float4 *>(&s_q[buf][t][(u * kP + part) * 4]);
        kk[4 * u] = a.x; kk[4 * u + 1] = a.y; kk[4 * u + 2] = a.z; kk[4 * u + 3] = a.w;
        qq[4 * u] = b.x; qq[4 * u + 1] = b.y; qq[4 * u + 2] = b.z; qq[4 * u + 3] = b.w;
      }
      double pred = 0.0;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        col[i] *= decay;
        pred += (double)(col[i] * kk[i]);
      }
      pred = parts_sum<kP>(pred);
      const float corr = (v - (float)pred) * beta;
      double rd = 0.0;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        col[i] += kk[i] * corr;
        rd += (double)(col[i] * qq[i]);
      }
      const float o = (float)parts_sum<kP>(rd);
      // a non-finite cell makes its read product non-finite (inf * 0 is NaN),
      // and no f64 sum brings an inf or NaN term back to a finite value, so o
      // is non-finite whenever any updated cell is: o covers the cells' check
      if (active && part == 0) {
        const size_t row = first + t0 + t;
        o_out[row * ldo + h * VD + j] = o;
        if (!finitef(o) || !finitef(v)) atomicOr(&row_err[row], kErrRequest);
      }
    }
    if (more) stash(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  if (active) {
#pragma unroll
    for (int i = 0; i < 16; i++) S[(size_t)(16 * part + i) * VD] = col[i];
  }
}

// ---------------------------------------------------------------------------
// The whole linear-attention mixer of one (lane, value head) in one
// workgroup, token after token (execution.rs:357-411): the causal conv of the
// head's q, k (its key head's channels) and v channels, the q/k norms and
// gates, the delta-rule column updates, and the output norm times SiLU(z).
// kP lanes own one state column, kKD / kP keys each.  The arithmetic of each
// stage and the order of each sum are the separate kernels' (sums of 16 keys,
// then a tree over them), so a lane's results do not depend on which of the two
// runs it.  (One thread per column with ordered sums took 19 us a
// launch at 16 one-token lanes x 16 heads, most of it waiting on one lane's
// adds; this takes 15.  Whole waves hold one part of the columns, so the state
// streams in 256-byte rows and the partial sums meet in LDS: with the lanes of
// a column side by side, in 32-byte pieces and DPP sums, it took 18.)
// Used when every value head has its own key head: a workgroup then owns all
// the conv channels it reads and writes back (with shared key heads the ring
// would be read by one workgroup after another had advanced it).  Conv
// kernels up to kFusedConv taps.
// ---------------------------------------------------------------------------
constexpr int kFusedConv = 4;
struct ConvTaps {
  float tap[kFusedConv], w[kFusedConv];
};
__device__ __forceinline__ void conv_load(ConvTaps &c, const float *h, const float *w, int K,
                                          int c0) {
#pragma unroll
  for (int i = 0; i < kFusedConv; i++) {
    c.tap[i] = i < K ? h[(c0 + i) % K] : 0.0f;
    c.w[i] = i < K ? w[i] : 0.0f;
  }
}
__device__ __forceinline__ float conv_step(ConvTaps &c, float in, int K, const uint64_t *tab) {
#pragma unroll
  for (int i = 0; i < kFusedConv - 1; i++)
    if (i < K - 1) c.tap[i] = c.tap[i + 1];
#pragma unroll
  for (int i = 0; i < kFusedConv; i++)
    if (i == K - 1) c.tap[i] = in;
  double sum = -0.0;
#pragma unroll
  for (int i = 0; i < kFusedConv; i++)
    if (i < K) sum += (double)(c.tap[i] * c.w[i]);
  return silu_f32((float)sum, tab);
}
__device__ __forceinline__ void conv_store(const ConvTaps &c, float *h, int K, int c1) {
#pragma unroll
  for (int i = 0; i < kFusedConv; i++)
    if (i < K) h[(c1 + i) % K] = c.tap[i];
}

template <int kKD, int kP>
__global__ __launch_bounds__(1024) void k_q35_linear(
    Q35Lanes L, const float *__restrict__ mix, int ldm, int keys, int z_off, int a_off, int b_off,
    const float *__restrict__ conv_w, int K, float *hist, size_t hist_seq,
    const float *__restrict__ a_log, const float *__restrict__ dt,
    const float *__restrict__ norm_w, int KH, int VH, int VD, float eps, float *state,
    size_t state_seq, float *__restrict__ tgt, int ldt, uint32_t *row_err) {
  constexpr int kCells = kKD / kP, kHalves = kCells / 16;  // keys per thread, in sums of 16
  constexpr int kN = kKD < kWave ? kKD : kWave;   // channels of one norm partial
  __shared__ __align__(16) float s_q[kKD], s_k[kKD], s_v[256];
  __shared__ double s_p[2][1024];
  __shared__ double s_sq[1024 / kN], s_o[256];
  __shared__ float s_decay, s_beta;
  __shared__ int s_bad;
  __shared__ uint64_t s_tab[32];
  const int ln = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  if (tid < 32) s_tab[tid] = kExp2Tab[tid];
  const int rep = VH / KH, src = (h / rep) * kKD;
  const uint32_t first = L.first[ln], n = L.n[ln], start = L.start[ln];
  const uint32_t seq = L.seq[ln];
  float *hs = hist + (size_t)seq * hist_seq;
  const int c0 = (int)(start % (uint32_t)K);
  // conv roles: thread tid brings q channel tid, k channel tid - kKD or v
  // channel tid - 2 kKD (the launch gives at least 2 kKD + VD threads)
  const bool has_c = tid < 2 * kKD + VD;
  const int ch = tid < kKD ? src + tid : tid < 2 * kKD ? keys + src + tid - kKD : 2 * keys + h * VD + tid - 2 * kKD;
  // the first token's small inputs are requested before the state: loads
  // complete in order, and the conv and the gate then run under the state's
  ConvTaps ct;
  if (has_c) conv_load(ct, hs + (size_t)ch * K, conv_w + (size_t)ch * K, K, c0);
  const bool gate = tid == (int)blockDim.x - 1;
  float in = 0.0f, a_in = 0.0f, b_in = 0.0f;
  auto small = [&](uint32_t t) {
    const float *mr = mix + (size_t)(first + t) * ldm;
    if (has_c) in = mr[ch];
    if (gate) {
      a_in = mr[a_off + h];
      b_in = mr[b_off + h];
    }
  };
  if (n) small(0);
  const float al = gate ? a_log[h] : 0.0f, dtb = gate ? dt[h] : 0.0f;
  __builtin_amdgcn_sched_barrier(0);
  // delta roles: part `part` of state column j
  // (whole waves of one part, so a wave's state loads are contiguous)
  const int vdp = (VD + kWave - 1) / kWave * kWave;
  const int part = __builtin_amdgcn_readfirstlane(tid / vdp), j = tid % vdp;
  const bool active = j < VD && part < kP;
  float *S = state + (size_t)seq * state_seq + (size_t)h * kKD * VD + (active ? j : 0);
  float col[kCells];
#pragma unroll
  for (int i = 0; i < kCells; i++) col[i] = active ? S[(size_t)(kCells * part + i) * VD] : 0.0f;
  const float nw = active ? norm_w[j] : 0.0f;
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();  // s_tab
  // a column's partial sums meet in LDS and are added in parts_sum's order
  auto all_parts = [&](int which, const double (&v)[kHalves]) {
    double p[kP];
    p[0] = kHalves == 1 ? v[0] : v[0] + v[kHalves - 1];
    if constexpr (kP > 1) {
      s_p[which][tid] = p[0];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kP; i++) p[i] = s_p[which][i * vdp + j];
#pragma unroll
      for (int m = 1; m < kP; m <<= 1)
#pragma unroll
        for (int i = 0; i < kP; i += 2 * m) p[i] += p[i + m];
    }
    return p[0];
  };
  for (uint32_t t = 0; t < n; t++) {
    const uint32_t row = first + t;
    const float *mr = mix + (size_t)row * ldm;
    const float z = active ? mr[z_off + h * VD + j] : 0.0f;
    bool bad = false;
    // causal conv + SiLU (kernels.rs:54-120)
    float y = 0.0f;
    if (has_c) {
      y = conv_step(ct, in, K, s_tab);
      bad |= !finitef(in) || !finitef(y);
      if (tid < 2 * kKD) {
        (tid < kKD ? s_q : s_k)[tid % kKD] = y;
      } else {
        s_v[tid - 2 * kKD] = y;
      }
    }
    // q/k norms: a tree over each kN channels, then (128 keys) two in order
    const double sq = pairs_sum<kN>((double)(y * y));
    if (tid % kN == 0) s_sq[tid / kN] = sq;
    if (gate) {
      const float ld = -exp_f32_tab(al, s_tab) * softplus_f32(a_in + dtb, s_tab);
      const float beta = sigmoid_f32(b_in, s_tab);
      s_decay = exp_f32_tab(ld, s_tab);
      s_beta = beta;
      s_bad = !finitef(ld) || !finitef(beta) || ld > 0.0f || !(beta >= 0.0f && beta <= 1.0f);
    }
    if (t + 1 < n) small(t + 1);
    __syncthreads();
    constexpr int kNP = kKD / kN;
    double qs = s_sq[0], ks = s_sq[kNP];
    if constexpr (kNP == 2) {
      qs += s_sq[1];
      ks += s_sq[3];
    }
    const float qn = (float)qs, kn = (float)ks;
    bad |= !finitef(qn) || !finitef(kn);
    const float q_scale = (1.0f / sqrtf(qn + 1e-6f)) / sqrtf((float)kKD), k_scale = 1.0f / sqrtf(kn + 1e-6f);
    // the delta rule on state column j (kernels.rs:122-214), as in k_q35_delta
    float o = 0.0f;
    {
      const float decay = s_decay, beta = s_beta, v = s_v[min(j, VD - 1)];
      double pred[kHalves] = {};
      float kk[kCells];
#pragma unroll
      for (int u = 0; u < kCells / 4; u++) {
        const float4 a = *reinterpret_cast<const float4 *>(&s_k[part % kP * kCells + 4 * u]);
        kk[4 * u] = a.x * k_scale; kk[4 * u + 1] = a.y * k_scale;
        kk[4 * u + 2] = a.z * k_scale; kk[4 * u + 3] = a.w * k_scale;
      }
#pragma unroll
      for (int i = 0; i < kCells; i++) {
        col[i] *= decay;
        pred[i / 16] += (double)(col[i] * kk[i]);
      }
      const float corr = (v - (float)all_parts(0, pred)) * beta;
      double rd[kHalves] = {};
#pragma unroll
      for (int u = 0; u < kCells / 4; u++) {
        const float4 a = *reinterpret_cast<const float4 *>(&s_q[part % kP * kCells + 4 * u]);
        const float qq[4] = {a.x * q_scale, a.y * q_scale, a.z * q_scale, a.w * q_scale};
#pragma unroll
        for (int e = 0; e < 4; e++) {
          col[4 * u + e] += kk[4 * u + e] * corr;
          rd[u / 4] += (double)(col[4 * u + e] * qq[e]);
        }
      }
      // a non-finite updated cell makes o non-finite (its read product is
      // inf or NaN, and no f64 sum returns from those), so o covers the cells
      o = (float)all_parts(1, rd);
      bad |= active && !finitef(o);
    }
    // output norm over the head (zero_centered false) times SiLU(z) (execution.rs:397-411)
    // its sum as in k_q35_headnorm, by every wave
    if (active && part == 0) s_o[j] = (double)(o * o);
    __syncthreads();
    double os = -0.0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int i = tid % kWave + c * kWave;
      if (i < VD) os += s_o[i];
    }
    const double mean = wave_sum_f64(os) / (double)VD;
    bad |= !(__builtin_isfinite(mean) && finitef((float)mean));
    if (active && part == 0) {
      const float yo = ((o * (1.0f / sqrtf((float)mean + eps))) * (nw + 0.0f)) * silu_f32(z, s_tab);
      tgt[(size_t)row * ldt + h * VD + j] = yo;
      bad |= !finitef(yo);
    }
    if (bad || (tid == 0 && s_bad)) atomicOr(&row_err[row], kErrRequest);
    __syncthreads();  // the LDS stages are rewritten by the next token
  }
  const int c1 = (int)((start + n) % (uint32_t)K);
  if (has_c) conv_store(ct, hs + (size_t)ch * K, K, c1);
  if (active) {
#pragma unroll
    for (int i = 0; i < kCells; i++) S[(size_t)(kCells * part + i) * VD] = col[i];
  }
}

// Per value head: the output norm (zero_centered false) times SiLU(z)
// (execution.rs:397-411), one wave per (row, value head), its sum as in the
// gates: 73 -> 35 us at 4,104 rows x 16 heads.
__global__ __launch_bounds__(256) void k_q35_headnorm(const float *__restrict__ o_in, int ldo,
                                                      const float *__restrict__ mix, int ldm,
                                                      int z_off, const float *__restrict__ w, int VH,
                                                      int VD, int pairs, float eps, float *__restrict__ tgt,
                                                      int ldt, uint32_t *row_err) {
  __shared__ uint64_t s_tab[32];
  if (threadIdx.x < 32) s_tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  __syncthreads();
  const int pair = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (pair >= pairs) return;
  const int row = pair / VH, h = pair % VH;
  constexpr int kHeld = 4;  // VD <= 256
  float o[kHeld], z[kHeld], nw[kHeld];
  double ss = -0.0;
#pragma unroll
  for (int c = 0; c < kHeld; c++) {
    const int j = lane + c * kWave;
    const bool in = j < VD;
    o[c] = in ? o_in[(size_t)row * ldo + h * VD + j] : 0.0f;
    z[c] = in ? mix[(size_t)row * ldm + z_off + h * VD + j] : 0.0f;
    nw[c] = in ? w[j] : 0.0f;
  }
#pragma unroll
  for (int c = 0; c < kHeld; c++)
    if (lane + c * kWave < VD) ss += (double)(o[c] * o[c]);
  const double mean = wave_sum_f64(ss) / (double)VD;
  bool bad = !(__builtin_isfinite(mean) && finitef((float)mean));
  const float scale = 1.0f / sqrtf((float)mean + eps);
#pragma unroll
  for (int c = 0; c < kHeld; c++) {
    const int j = lane + c * kWave;
    if (j < VD) {
      const float y = ((o[c] * scale) * (nw[c] + 0.0f)) * silu_f32(z[c], s_tab);
      tgt[(size_t)row * ldt + h * VD + j] = y;
      bad |= !finitef(y);
    }
  }
  if (bad) atomicOr(&row_err[row], kErrRequest);
}

// ---------------------------------------------------------------------------
// Full-attention q/k preparation (execution.rs:436-497): per head the
// zero-centred norm, then the partial rotary embedding (kernels.rs:226-268)
// from the host table (cos, sin) of angle pos * base^(-2i/rotary); q and its
// gate to the q/z buffers, k and v appended to the sequence's cache rows.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_q35_qk(Q35Rows Rw, const float *__restrict__ mix,
                                                int ldm, int k_off, int v_off,
                                                const float *__restrict__ q_norm,
                                                const float *__restrict__ k_norm, int NH, int NKV,
                                                int D, int rotary, float eps,
                                                const float2 *__restrict__ rope, float *q,
                                                float *z, int ldq, float *kc, float *vc,
                                                size_t cache_seq, uint32_t *row_err) {
  __shared__ float y[kQ35MaxHeadDim];
  __shared__ double red[kQ35MaxHeadDim / kWave];
  const int row = blockIdx.x, hh = blockIdx.y, d = threadIdx.x;
  const uint32_t pos = Rw.pos[row], seq = Rw.seq[row];
  const bool is_q = hh < NH;
  const int kh = hh - NH, kvw = NKV * D;
  const float *srcp = mix + (size_t)row * ldm + (is_q ? hh * 2 * D : k_off + kh * D);
  const float xv = d < D ? srcp[d] : 0.0f;
  // the f64 sum of squares: a tree per wave, then the waves in order
  const double part = wave_sum_f64(d < D ? (double)(xv * xv) : -0.0);
  if (d % kWave == 0) red[d / kWave] = part;
  __syncthreads();
  double sum = red[0];
  for (int i = 1; i < (int)blockDim.x / kWave; i++) sum += red[i];
  const double mean = sum / (double)D;
  const float scale = 1.0f / sqrtf((float)mean + eps);
  bool bad = (d < D && !finitef(xv)) || !(__builtin_isfinite(mean) && finitef((float)mean));
  if (d < D) {
    y[d] = (xv * scale) * ((is_q ? q_norm : k_norm)[d] + 1.0f);
    bad |= !finitef(y[d]);
  }
  __syncthreads();
  float *dst = is_q ? q + (size_t)row * ldq + hh * D
                    : kc + (size_t)seq * cache_seq + (size_t)pos * kvw + kh * D;
  const int half = rotary / 2;
  if (d < half) {
    const float a = y[d], b = y[d + half];
    const float2 cs = rope[(size_t)pos * half + d];
    const float ra = a * cs.x - b * cs.y, rb = b * cs.x + a * cs.y;
    dst[d] = ra;
    dst[d + half] = rb;
    bad |= !finitef(ra) || !finitef(rb);
  } else if (d >= rotary && d < D) {
    dst[d] = y[d];
  }
  if (d < D) {
    if (is_q)
      z[(size_t)row * ldq + hh * D + d] = mix[(size_t)row * ldm + hh * 2 * D + D + d];
    else
      vc[(size_t)seq * cache_seq + (size_t)pos * kvw + kh * D + d] =
          mix[(size_t)row * ldm + v_off + kh * D + d];
  }
  if (bad) atomicOr(&row_err[row], kErrRequest);
}

// ---------------------------------------------------------------------------
// Attention scores s_t = f32(sum_i f64(q_i * k_t,i)) / sqrt(D) (cpu.rs:80-124
// dot products), every (row, head, key) an independent ordered chain: a
// workgroup takes one row, one KV group and 256/G keys, the G heads of the
// group side by side so each K load serves them all.  Scores go to
// sc[row][head][key].
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_q35_scores(Q35Rows Rw, const float *__restrict__ q,
                                                    int ldq, const float *__restrict__ kc,
                                                    size_t cache_seq, int NH, int NKV, int D,
                                                    float *__restrict__ sc, int ldsc) {
  __shared__ __align__(16) float qs[kQ35MaxGroup * kQ35MaxHeadDim];
  const int row = blockIdx.x, kvh = blockIdx.y, G = NH / NKV, kb = 256 / G;
  const int kv = (int)Rw.pos[row] + 1, t0 = blockIdx.z * kb;
  if (t0 >= kv) return;
  const uint32_t seq = Rw.seq[row];
  const int kvw = NKV * D;
  const float *qg = q + (size_t)row * ldq + (size_t)kvh * G * D;
  for (int i = threadIdx.x; i < G * D; i += 256) qs[i] = qg[i];
  __syncthreads();
  const int hg = threadIdx.x % G, t = t0 + (int)threadIdx.x / G;
  if (t >= kv || (int)threadIdx.x >= kb * G) return;
  const float4 *kr =
      reinterpret_cast<const float4 *>(kc + (size_t)seq * cache_seq + (size_t)t * kvw + kvh * D);
  const float4 *qh = reinterpret_cast<const float4 *>(qs + hg * D);
  double a = -0.0;
  const int n4 = D / 4;
  for (int i0 = 0; i0 < n4; i0 += 8) {
    float4 kk[8];
#pragma unroll
    for (int j = 0; j < 8; j++) kk[j] = i0 + j < n4 ? kr[i0 + j] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      if (i0 + j < n4) {
        const float4 qq = qh[i0 + j];
        a += (double)(qq.x * kk[j].x);
        a += (double)(qq.y * kk[j].y);
        a += (double)(qq.z * kk[j].z);
        a += (double)(qq.w * kk[j].w);
      }
    }
  }
  sc[((size_t)row * NH + kvh * G + hg) * ldsc + t] = (float)a / sqrtf((float)D);
}

// ---------------------------------------------------------------------------
// Online-softmax attention (cpu.rs:80-124) in the reference's exact order.
// The running maximum m_t is a prefix maximum (exact in any order), so the
// maxima and both exponentials old_t = exp(m_{t-1} - m_t), new_t =
// exp(s_t - m_t) are formed in parallel from the scores; the two f32
// recurrences den = den*old + new and o_d = o_d*old + new*v_d then run in key
// order, one thread per output element (and one for the denominator), V
// loads running kAhead keys ahead.  The output is o/den times sigmoid(gate)
// (execution.rs:506-508).
// ---------------------------------------------------------------------------
template <int kAhead>
__global__ __launch_bounds__(576) void k_q35_attn(Q35Rows Rw, const float *__restrict__ scores,
                                                  int ldsc, const float *__restrict__ z, int ldq,
                                                  const float *__restrict__ vc, size_t cache_seq,
                                                  int NH, int NKV, int D, int maxc4,
                                                  float *__restrict__ out, int ldo) {
  extern __shared__ __align__(16) float sm[];
  float *sc = sm, *mx = sc + maxc4, *old = mx + maxc4, *seg = old + maxc4;
  __shared__ float s_den;
  const int row = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, nt = blockDim.x;
  const int dthreads = nt - kWave;  // the last wave runs the denominator
  const uint32_t pos = Rw.pos[row], seq = Rw.seq[row];
  const int kv = (int)pos + 1, kvh = h / (NH / NKV), kvw = NKV * D;
  const float *V = vc + (size_t)seq * cache_seq + kvh * D;
  const float *srow = scores + ((size_t)row * NH + h) * ldsc;
  __shared__ uint64_t s_tab[32];  // expf's table, read per lane in the exponent loops
  if (tid < 32) s_tab[tid] = kExp2Tab[tid];
  for (int t = tid; t < kv; t += nt) sc[t] = srow[t];
  __syncthreads();
  // prefix maxima: contiguous segments, then an exclusive scan of segment maxima
  const int per = (kv + nt - 1) / nt, lo = min(kv, tid * per), hi = min(kv, lo + per);
  float m = -__builtin_inff();
  for (int t = lo; t < hi; t++) {
    m = fmaxf(m, sc[t]);
    mx[t] = m;
  }
  // exclusive prefix maxima of the segment maxima (a maximum is exact in any
  // order): a shuffle scan within each wave, then the earlier waves' totals
  // (the block is whole waves)
  const int lane = tid % kWave, wave = tid / kWave;
  float inc = m;
#pragma unroll
  for (int d = 1; d < kWave; d *= 2) {
    const float u = __shfl_up(inc, d, kWave);
    if (lane >= d) inc = fmaxf(inc, u);
  }
  float base = __shfl_up(inc, 1, kWave);
  if (lane == 0) base = -__builtin_inff();
  if (lane == kWave - 1) seg[wave] = inc;
  __syncthreads();
  for (int i = 0; i < wave; i++) base = fmaxf(base, seg[i]);
  for (int t = lo; t < hi; t++) mx[t] = fmaxf(base, mx[t]);
  __syncthreads();
  for (int t = lo; t < hi; t++) {
    const float prev = t ? mx[t - 1] : -__builtin_inff();
    old[t] = exp_f32_tab(prev - mx[t], s_tab);
  }
  __syncthreads();
  for (int t = lo; t < hi; t++) sc[t] = exp_f32_tab(sc[t] - mx[t], s_tab);  // new_t
  __syncthreads();
  if (tid == dthreads) {
    float den = 0.0f;
    int t = 0;
    if constexpr (kAhead > 8) {
      // whole groups of 8 keys, the next group's factors loading while the
      // current one is folded in
      float4 of[2], nf[2], on[2], nn[2];
      auto get = [&](float4 (&o4)[2], float4 (&n4)[2], int g) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
          o4[u] = *reinterpret_cast<const float4 *>(old + 8 * g + 4 * u);
          n4[u] = *reinterpret_cast<const float4 *>(sc + 8 * g + 4 * u);
        }
      };
      const int full = kv / 8;
      if (full) get(of, nf, 0);
      for (int g = 0; g < full; g++) {
        get(on, nn, min(g + 1, full - 1));
#pragma unroll
        for (int u = 0; u < 2; u++) {
          den = den * of[u].x + nf[u].x;
          den = den * of[u].y + nf[u].y;
          den = den * of[u].z + nf[u].z;
          den = den * of[u].w + nf[u].w;
          of[u] = on[u];
          nf[u] = nn[u];
        }
      }
      t = full * 8;
    }
    for (; t < kv; t++) den = den * old[t] + sc[t];
    s_den = den;
  }
  float o = 0.0f;
  if (tid < D) {
    if constexpr (kAhead == 8) {
      // whole groups of 8 keys without branches, the next group's V values
      // loading while the current group is folded in; then the tail
      const float *vp = V + tid;
      const int full = kv / 8;
      float cur[8], nxt[8];
#pragma unroll
      for (int j = 0; j < 8; j++) cur[j] = full ? vp[(size_t)j * kvw] : 0.0f;
      for (int g = 0; g < full; g++) {
        const int tn = min(g + 1, full - 1) * 8;
#pragma unroll
        for (int j = 0; j < 8; j++) nxt[j] = vp[(size_t)(tn + j) * kvw];
        const float4 o0 = *reinterpret_cast<const float4 *>(old + 8 * g);
        const float4 o1 = *reinterpret_cast<const float4 *>(old + 8 * g + 4);
        const float4 n0 = *reinterpret_cast<const float4 *>(sc + 8 * g);
        const float4 n1 = *reinterpret_cast<const float4 *>(sc + 8 * g + 4);
        o = o * o0.x + n0.x * cur[0];
        o = o * o0.y + n0.y * cur[1];
        o = o * o0.z + n0.z * cur[2];
        o = o * o0.w + n0.w * cur[3];
        o = o * o1.x + n1.x * cur[4];
        o = o * o1.y + n1.y * cur[5];
        o = o * o1.z + n1.z * cur[6];
        o = o * o1.w + n1.w * cur[7];
#pragma unroll
        for (int j = 0; j < 8; j++) cur[j] = nxt[j];
      }
      for (int t = full * 8; t < kv; t++) o = o * old[t] + sc[t] * vp[(size_t)t * kvw];
    } else {
      // groups of kAhead keys, the next group's V values loading while the
      // current group is folded in; a last, partial group folds its own keys
      const float *vp = V + tid;
      const int groups = (kv + kAhead - 1) / kAhead;
      float cur[kAhead], nxt[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; j++) cur[j] = vp[(size_t)min(j, kv - 1) * kvw];
      for (int g = 0; g < groups; g++) {
        const int t0 = g * kAhead;
#pragma unroll
        for (int j = 0; j < kAhead; j++) nxt[j] = vp[(size_t)min(t0 + kAhead + j, kv - 1) * kvw];
#pragma unroll
        for (int u = 0; u < kAhead; u += 4) {
          if (t0 + u >= kv) break;
          const float4 of = *reinterpret_cast<const float4 *>(old + t0 + u);
          const float4 nf = *reinterpret_cast<const float4 *>(sc + t0 + u);
          o = o * of.x + nf.x * cur[u];
          if (t0 + u + 1 < kv) o = o * of.y + nf.y * cur[u + 1];
          if (t0 + u + 2 < kv) o = o * of.z + nf.z * cur[u + 2];
          if (t0 + u + 3 < kv) o = o * of.w + nf.w * cur[u + 3];
        }
#pragma unroll
        for (int j = 0; j < kAhead; j++) cur[j] = nxt[j];
      }
    }
  }
  __syncthreads();
  if (tid < D) {
    const float gate = z[(size_t)row * ldq + h * D + tid];
    out[(size_t)row * ldo + h * D + tid] = (o / s_den) * sigmoid_f32(gate);
  }
}

// ---------------------------------------------------------------------------
// Packed-prefill regime (steps of 128+ rows): the linears run on the
// matrix-core GEMM (gemm.h) over the tiled BF16 matrices.  An f32 activation x enters
// as hi = bf16(x) and lo = bf16(x - hi) (round to nearest even), so hi + lo
// is x to a relative 2^-17 or better, every product of two bfloat16 values is
// exact in f32, and the f32 sums of hi . w + lo . w are what differ from the
// reference's f64 dot (cpu.rs:31-48).  Thread = 4 consecutive inputs.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_q35_split(const float *__restrict__ x, int ldx, int K,
                                                   uint16_t *__restrict__ hi, uint16_t *__restrict__ lo) {
  const int r = blockIdx.y, k = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (k >= K) return;
  const float4 v = *reinterpret_cast<const float4 *>(x + (size_t)r * ldx + k);
  const float f[4] = {v.x, v.y, v.z, v.w};
  uint16_t h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const __bf16 bh = (__bf16)f[i];
    const __bf16 bl = (__bf16)(f[i] - (float)bh);
    h[i] = __builtin_bit_cast(uint16_t, bh);
    l[i] = __builtin_bit_cast(uint16_t, bl);
  }
  *reinterpret_cast<uint2 *>(hi + (size_t)r * K + k) =
      make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
  *reinterpret_cast<uint2 *>(lo + (size_t)r * K + k) =
      make_uint2(l[0] | (uint32_t)l[1] << 16, l[2] | (uint32_t)l[3] << 16);
}

// Copies of a snapshot (cohx_seq_fork): piece blockIdx.y, 16-byte words.
__global__ __launch_bounds__(256) void k_q35_copy(Q35Copy c) {
  const Q35Copy::Piece p = c.piece[blockIdx.y];
  const u32x4q *src = reinterpret_cast<const u32x4q *>(p.src);
  u32x4q *dst = reinterpret_cast<u32x4q *>(p.dst);
  const size_t n = p.floats / 4, step = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) dst[i] = src[i];
  for (size_t i = n * 4 + (size_t)blockIdx.x * 256 + threadIdx.x; i < p.floats; i += step) p.dst[i] = p.src[i];
}

}  // namespace

// ---- launchers ---------------------------------------------------------------

void q35_copy(hipStream_t s, const Q35Copy &c, int pieces) {
  hipLaunchKernelGGL(k_q35_copy, dim3(64, pieces), dim3(256), 0, s, c);
}

void q35_embed(hipStream_t s, int rows, const uint16_t *embed, const uint32_t *tokens, int H,
               float *x) {
  hipLaunchKernelGGL(k_q35_embed, dim3(rows), dim3(256), 0, s, embed, tokens, H, x);
}

void q35_norm(hipStream_t s, int rows, const float *x, int ldx, const uint32_t *src,
              const float *w, int n, float eps, int zc, float *out, int ldo, uint32_t *row_err,
              const uint32_t *err_row) {
  hipLaunchKernelGGL(k_q35_norm, dim3(rows), dim3(256), 0, s, x, ldx, src, w, n, eps, zc, out,
                     ldo, row_err, err_row);
}

int q35_matvec_blocks(int rows_w) { return (rows_w + 15) / 16; }

// Rows per workgroup (kR) and waves that split K (kW).  More rows share each
// weight load and widening, but the grid has to fill the CUs: at 16 rows o and
// down (64 tiles) take 7.3 and 10.0 us as four rows on eight waves, 10.0 and
// 14.6 as eight; gate+up (224 pairs) 15.0 as eight rows on four waves, 15.2 as
// four, 18.9 as sixteen; mix (514 tiles) 17.1, 17.2 and 20.1; the head (15,520
// tiles) 330 as sixteen, 346 as eight, 399 as four.  The sums are the same in all.
template <int kEpi>
static void mv(hipStream_t s, const uint16_t *w, int tiles, int valid_rows, int K, const float *x, int ldx, int R,
               float *out, int ldo, unsigned long long *part, uint32_t *row_err, const uint32_t *err_row) {
  auto go = [&](auto kr, auto kw) {
    constexpr int kR = decltype(kr)::value, kW = decltype(kw)::value;
    const dim3 grid(tiles, (R + kR - 1) / kR);
    if (K % 64 == 0)
      hipLaunchKernelGGL((k_q35_mv<kEpi, kR, kW, false>), grid, dim3(64 * kW), 0, s, w, valid_rows, K, x, ldx, R, out,
                         ldo, part, row_err, err_row);
    else
      hipLaunchKernelGGL((k_q35_mv<kEpi, kR, kW, true>), grid, dim3(64 * kW), 0, s, w, valid_rows, K, x, ldx, R, out,
                         ldo, part, row_err, err_row);
  };
  using std::integral_constant;
  const int g8 = tiles * ((R + 7) / 8), g4 = tiles * ((R + 3) / 4);
  if (R > 8 && tiles * ((R + 15) / 16) >= 4096)
    go(integral_constant<int, 16>{}, integral_constant<int, 4>{});
  else if (R > 4 && g8 >= 448)
    go(integral_constant<int, 8>{}, integral_constant<int, 4>{});
  else if (g4 >= 448)
    go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
  else
    go(integral_constant<int, 4>{}, integral_constant<int, 8>{});
}

void q35_matvec(hipStream_t s, int epi, const uint16_t *w, int rows_w, int valid_rows, int K,
                const float *x, int ldx, int R, float *out, int ldo, unsigned long long *part,
                uint32_t *row_err, const uint32_t *err_row) {
  const int tiles = rows_w / 16;
  if (epi == kQ35Store)
    mv<kQ35Store>(s, w, tiles, valid_rows, K, x, ldx, R, out, ldo, part, row_err, err_row);
  else if (epi == kQ35Residual)
    mv<kQ35Residual>(s, w, tiles, valid_rows, K, x, ldx, R, out, ldo, part, row_err, err_row);
  else
    mv<kQ35Argmax>(s, w, tiles, valid_rows, K, x, ldx, R, out, ldo, part, row_err, err_row);
}

void q35_matvec_swiglu(hipStream_t s, const uint16_t *w, int up_off, int F, int K, const float *x,
                       int ldx, int R, float *h, uint32_t *row_err) {
  mv<kQ35Swiglu>(s, w, up_off / 16, up_off, K, x, ldx, R, h, F, nullptr, row_err, nullptr);
}

void q35_split_bf16(hipStream_t s, int rows, int K, const float *x, int ldx, uint16_t *hi, uint16_t *lo) {
  hipLaunchKernelGGL(k_q35_split, dim3((K / 4 + 255) / 256, rows), dim3(256), 0, s, x, ldx, K, hi, lo);
}

// Tiles measured on the Qwen3.5 prompt-chunk shapes (4,096 rows, hi and lo
// products counted): 128 x 128 on eight waves of 64 features x 32 rows with
// two K steps in flight (mix 8,224 x 1024: 170 us; gate+up 7,168 x 1024:
// 130 us; out K 2048: 41 us; down K 3584: 63 us; on four waves of 64 x 64:
// 181, 128, 48, 72).
void q35_gemm_split(hipStream_t s, bool accumulate, const uint16_t *w, int N, int K, const uint16_t *hi,
                    const uint16_t *lo, int rows, float *out, int ldo, uint32_t *row_err) {
  using namespace gemm;
  Args g{};
  g.w = w;
  g.w_tiled = 1;
  g.x = hi;
  g.xlo = lo;
  g.N = N;
  g.K = K;
  g.M = rows;
  g.ldx = K;
  g.out = out;
  g.ldo = ldo;
  g.row_err = row_err;
  const dim3 grid(tile_order(g, N, 128, 128));
  constexpr int lds = lds_bytes<2, 4, 4, 2, true, kStore>();
  if (accumulate)
    hipLaunchKernelGGL((k_gemm<kBF16, true, 2, 4, 4, 2, 2, kAccumulate>), grid, dim3(512), lds, s, g);
  else
    hipLaunchKernelGGL((k_gemm<kBF16, true, 2, 4, 4, 2, 2, kStore>), grid, dim3(512), lds, s, g);
}

void q35_swiglu(hipStream_t s, int rows, const float *gu, int ldgu, int F, int up_off, float *h,
                int ldh) {
  hipLaunchKernelGGL(k_q35_swiglu, dim3((F + 255) / 256, rows), dim3(256), 0, s, gu, ldgu, F,
                     up_off, h, ldh);
}

void q35_conv(hipStream_t s, int lanes, int max_tokens, Q35Lanes L, const float *mix, int ldm, const float *w,
              int C, int K, float *hist, size_t hist_seq, float *out, int ldo, uint32_t *row_err) {
  const dim3 grid(lanes, (C + 255) / 256, (max_tokens + kConvSeg - 1) / kConvSeg);
  if (K == 4)
    hipLaunchKernelGGL(k_q35_conv<4>, grid, dim3(256), 0, s, L, mix, ldm, w, C, K, hist, hist_seq, out, ldo, row_err);
  else
    hipLaunchKernelGGL(k_q35_conv<0>, grid, dim3(256), 0, s, L, mix, ldm, w, C, K, hist, hist_seq, out, ldo, row_err);
}

bool q35_linear_fused(int conv_kernel, int key_heads, int value_heads) {
  return conv_kernel <= kFusedConv && key_heads == value_heads;
}

void q35_linear(hipStream_t s, int lanes, Q35Lanes L, const float *mix, int ldm, int keys,
                int z_off, int a_off, int b_off, const float *conv_w, int K, float *hist,
                size_t hist_seq, const float *a_log, const float *dt, const float *norm_w,
                int key_heads, int value_heads, int key_dim, int value_dim, float eps,
                float *state, size_t state_seq, float *tgt, int ldt, uint32_t *row_err) {
  const dim3 grid(lanes, value_heads);
  // a column's lanes: 16 keys each, or 32 where 128 keys x more than 128
  // columns would pass 1,024 threads
  auto go = [&](auto kd, auto parts) {
    constexpr int kKD = decltype(kd)::value, kP = decltype(parts)::value;
    const int vdp = (value_dim + kWave - 1) / kWave * kWave;
    const int threads = (std::max(vdp * kP, 2 * kKD + value_dim) + kWave - 1) / kWave * kWave;
    hipLaunchKernelGGL((k_q35_linear<kKD, kP>), grid, dim3(threads), 0, s, L, mix, ldm, keys, z_off, a_off, b_off,
                       conv_w, K, hist, hist_seq, a_log, dt, norm_w, key_heads, value_heads, value_dim, eps, state,
                       state_seq, tgt, ldt, row_err);
  };
  using std::integral_constant;
  switch (key_dim) {
    case 16: return go(integral_constant<int, 16>{}, integral_constant<int, 1>{});
    case 32: return go(integral_constant<int, 32>{}, integral_constant<int, 2>{});
    case 64: return go(integral_constant<int, 64>{}, integral_constant<int, 4>{});
    case 128:
      if (value_dim <= 128) return go(integral_constant<int, 128>{}, integral_constant<int, 8>{});
      return go(integral_constant<int, 128>{}, integral_constant<int, 4>{});
    default: return;
  }
}

bool q35_delta_supported(int key_dim, int value_dim) {
  return (key_dim == 16 || key_dim == 32 || key_dim == 64 || key_dim == 128) && value_dim >= 1 &&
         value_dim <= 256;
}

void q35_delta(hipStream_t s, int rows, int lanes, Q35Lanes L, const float *conv, int ldc, int keys,
               const float *mix, int ldm, int z_off, int a_off, int b_off, const float *a_log,
               const float *dt, const float *norm_w, int key_heads, int value_heads, int key_dim,
               int value_dim, float eps, float *state, size_t state_seq, float4 *gates,
               float *o_raw, float *tgt, int ldt, uint32_t *row_err) {
  const int pairs = rows * value_heads;
  hipLaunchKernelGGL(k_q35_gates, dim3((pairs + 3) / 4), dim3(256), 0, s, conv, ldc, keys, mix, ldm, a_off, b_off,
                     a_log, dt, key_heads, value_heads, key_dim, pairs, gates, row_err);
#define L_(KD)                                                                                 \
  case KD:                                                                                     \
    hipLaunchKernelGGL(k_q35_delta<KD>, dim3(lanes, value_heads, (value_dim + 4096 / KD - 1) / (4096 / KD)), \
                       dim3(256), 0, s, L, conv, ldc, keys, gates, key_heads, value_heads, value_dim, state, \
                       state_seq, o_raw, ldt, row_err);                                        \
    break;
  switch (key_dim) {
    L_(16) L_(32) L_(64) L_(128)
    default: break;
  }
#undef L_
  hipLaunchKernelGGL(k_q35_headnorm, dim3((pairs + 3) / 4), dim3(256), 0, s, o_raw, ldt, mix, ldm, z_off, norm_w,
                     value_heads, value_dim, pairs, eps, tgt, ldt, row_err);
}

void q35_qk(hipStream_t s, int rows, Q35Rows Rw, const float *mix, int ldm, int k_off, int v_off,
            const float *q_norm, const float *k_norm, int heads, int kv_heads, int D, int rotary,
            float eps, const float2 *rope, float *q, float *z, int ldq, float *kc, float *vc,
            size_t cache_seq, uint32_t *row_err) {
  const int threads = ((D + kWave - 1) / kWave) * kWave;
  hipLaunchKernelGGL(k_q35_qk, dim3(rows, heads + kv_heads), dim3(threads), 0, s, Rw, mix, ldm,
                     k_off, v_off, q_norm, k_norm, heads, kv_heads, D, rotary, eps, rope, q, z,
                     ldq, kc, vc, cache_seq, row_err);
}

void q35_attention(hipStream_t s, int rows, Q35Rows Rw, const float *q, const float *z, int ldq,
                   const float *kc, const float *vc, size_t cache_seq, int heads, int kv_heads,
                   int D, int max_context, float *scores, float *out, int ldo) {
  const int G = heads / kv_heads, kb = 256 / G;
  hipLaunchKernelGGL(k_q35_scores, dim3(rows, kv_heads, (max_context + kb - 1) / kb), dim3(256), 0,
                     s, Rw, q, ldq, kc, cache_seq, heads, kv_heads, D, scores, max_context);
  const int threads = ((D + kWave - 1) / kWave) * kWave + kWave;
  const int maxc4 = (max_context + 3) / 4 * 4;
  const size_t lds = (size_t)(3 * maxc4 + threads) * sizeof(float);
  // few rows: the walk over the keys waits on memory, so 32 keys' V values are
  // in flight per thread (16 decode rows over 32-448 keys: 35 -> 25 us); many rows
  // hide that among themselves and keep the smaller form's occupancy
  if (rows * heads <= 1024)
    hipLaunchKernelGGL(k_q35_attn<32>, dim3(rows, heads), dim3(threads), lds, s, Rw, scores, max_context,
                       z, ldq, vc, cache_seq, heads, kv_heads, D, maxc4, out, ldo);
  else
    hipLaunchKernelGGL(k_q35_attn<8>, dim3(rows, heads), dim3(threads), lds, s, Rw, scores, max_context,
                       z, ldq, vc, cache_seq, heads, kv_heads, D, maxc4, out, ldo);
}

}  // namespace cohx
