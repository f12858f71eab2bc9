// Fused elementwise kernels of the Qwen3 decoder around the sparse
// layer-step (its caller: nanovllm/models/qwen3.py).
//
// One launch each for what the reference runs as a chain of small tensor
// ops, with the same rounding points (fp32 arithmetic, bf16 where the
// reference stores a bf16 tensor):
//  * rmsnorm_kernel: RMSNorm, optionally after the residual add
//    (nanovllm/layers/layernorm.py:17-44): s = x (+ r) in fp32,
//    r' = bf16(s), y = bf16(bf16(s * rsqrt(mean(s^2) + eps)) * w);
//  * qk_norm_rope_kernel: per-head RMSNorm of q and k, then rotate-half RoPE
//    in fp32 with the products and sums rounded separately, as separate
//    tensor ops round them (nanovllm/models/qwen3.py:99-110,
//    nanovllm/layers/rotary_embedding.py:6-50); v is copied out of the
//    fused projection output so that q, k and v are contiguous;
//  * silu_mul_kernel: SiLU(gate) * up (nanovllm/layers/activation.py:6-11),
//    bf16(bf16(g / (1 + e^-g)) * u).
//  * gemv_kernel: the decode-time projections (nn.Linear without bias on
//    1-4 rows, nanovllm/layers/linear.py) as an HBM-bound matrix-vector
//    product, fp32 accumulation, bf16 output; norm_gemv_kernel: the RMSNorm of
//    one row in front of it, in the same launch.
// The sums of squares are taken in a fixed order of this kernel's own, so
// a result can differ from a tensor library's reduction by an fp32 rounding.
#include <algorithm>

#include "nkv_common.h"

namespace nkv {
namespace {

constexpr int kNormThreads = 256;
constexpr int kNormChunks = 4;  // 8-element chunks per thread: rows of up to 8192
constexpr int kMaxNormWidth = kNormThreads * kNormChunks * 8;

// Two floats rounded to bf16 (nearest even, NaN stays NaN) in one conversion
// instruction: the integer form of f32_to_bf16 is about seven per value, which
// bounded the elementwise kernels (us: RMSNorm + residual 1 x 2560 3.8 -> 2.8,
// 3000 x 2560 17.9 -> 15.9; SiLU-mul 3000 x 9728 37.5 -> 34.7, 5.0 TB/s).
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  return make_uint4(pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7]));
}

// f rounded to bf16, as fp32
__device__ __forceinline__ void round8(float (&f)[8]) { unpack8(pack8(f), f); }

__device__ __forceinline__ float round_bf16(float f) { return bf16_to_f32(f32_to_bf16(f)); }

// The pieces of a row's RMSNorm, thread t of kNormThreads holding chunks t,
// t + kNormThreads, ...: chunk c as fp32 (x, plus the residual, whose bf16 sum
// goes to ro) with its squares added to ss in order, ...
__device__ __forceinline__ void norm_load(const uint4& x, const uint4* rr, uint4* ro, int c, float (&v)[8], float& ss) {
  unpack8(x, v);
  if (rr) {
    float r[8];
    unpack8(rr[c], r);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += r[e];
  }
  if (ro) ro[c] = pack8(v);
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
}
// ... rsqrt(mean(s^2) + eps) over the workgroup's partial sums (one barrier), ...
__device__ __forceinline__ float norm_scale(float ss, float* s_part, int wave, int lane, int n, float eps) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  if (lane == 0) s_part[wave] = ss;
  __syncthreads();
  float tot = 0.0f;
#pragma unroll
  for (int i = 0; i < kNormThreads / kWave; ++i) tot += s_part[i];
  return rsqrtf(tot / static_cast<float>(n) + eps);
}
// ... and bf16(bf16(s * r) * w).
__device__ __forceinline__ uint4 norm_apply(const float (&v)[8], float r, const uint4& w) {
  float wf[8], o[8];
  unpack8(w, wf);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = v[e] * r;
  round8(o);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] *= wf[e];
  return pack8(o);
}

// One workgroup per row.
__global__ __launch_bounds__(kNormThreads) void rmsnorm_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ res, const uint16_t* __restrict__ w,
    uint16_t* __restrict__ y, uint16_t* __restrict__ res_out, int n, float eps) {
  __shared__ float s_part[kNormThreads / kWave];
  const int64_t row = blockIdx.x;
  const int nc = n >> 3;
  const uint4* xr = reinterpret_cast<const uint4*>(x + row * n);
  const uint4* rr = res ? reinterpret_cast<const uint4*>(res + row * n) : nullptr;
  uint4* ro = res_out ? reinterpret_cast<uint4*>(res_out + row * n) : nullptr;
  float v[kNormChunks][8];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < kNormChunks; ++j) {
    const int c = threadIdx.x + j * kNormThreads;
    if (c < nc) norm_load(xr[c], rr, ro, c, v[j], ss);
  }
  const float r = norm_scale(ss, s_part, threadIdx.x / kWave, threadIdx.x & (kWave - 1), n, eps);
  const uint4* wr = reinterpret_cast<const uint4*>(w);
  uint4* yr = reinterpret_cast<uint4*>(y + row * n);
#pragma unroll
  for (int j = 0; j < kNormChunks; ++j) {
    const int c = threadIdx.x + j * kNormThreads;
    if (c < nc) yr[c] = norm_apply(v[j], r, wr[c]);
  }
}

// Eight lanes per (token, head) of the fused q|k|v projection output: lane i
// holds dims 8 i .. + 7 and 64 + 8 i .. + 7, eight rotate-half RoPE pairs, as
// two 16-byte pieces, so a wavefront streams 8 consecutive heads (2 KiB).
// The squares are summed over the pairs (d, d + 64), then over d by halving
// distances (32, 16, 8 across lanes, 4, 2, 1 inside), the order of
// qk_norm_rope_kernel: the same bits.  Bound by reading qkv and writing q, k
// and v once: 3000 tokens x 48 heads 45.3 -> 18.7 us (cold, 74 MB: 3.9 TB/s).
constexpr int kRopeThreads = 256;
constexpr int kRopeRows = 64;   // fewer rows: one wavefront per head
__global__ __launch_bounds__(kRopeThreads) void qk_norm_rope8_kernel(
    const uint16_t* __restrict__ qkv, uint32_t units, int hq, int hkv, const uint16_t* __restrict__ qw,
    const uint16_t* __restrict__ kw, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
    int max_pos, const int64_t* __restrict__ positions, float eps, uint16_t* __restrict__ q,
    uint16_t* __restrict__ k, uint16_t* __restrict__ v) {
#pragma clang fp contract(off)
  const uint32_t unit = blockIdx.x * (kRopeThreads / 8) + (threadIdx.x >> 3);
  const int i = threadIdx.x & 7;
  const int nh = hq + 2 * hkv;
  const uint32_t at = min(unit, units - 1);
  const int64_t t = at / static_cast<uint32_t>(nh);
  const int head = static_cast<int>(at % static_cast<uint32_t>(nh));
  const uint4* src = reinterpret_cast<const uint4*>(qkv + static_cast<int64_t>(at) * kHeadDim);
  const uint4 xa = src[i], xb = src[8 + i];
  const bool isq = head < hq, isv = head >= hq + hkv;
  int64_t pos = positions[t];
  pos = pos < 0 ? 0 : (pos >= max_pos ? max_pos - 1 : pos);
  const float4* ct = reinterpret_cast<const float4*>(cos_t + pos * (kHeadDim / 2) + 8 * i);
  const float4* st = reinterpret_cast<const float4*>(sin_t + pos * (kHeadDim / 2) + 8 * i);
  const float4 c0 = ct[0], c1 = ct[1], s0 = st[0], s1 = st[1];
  const uint4* wv = reinterpret_cast<const uint4*>(isq ? qw : kw);
  float a[8], b[8], wa[8], wb[8], ss[8];
  unpack8(xa, a);
  unpack8(xb, b);
  unpack8(wv[i], wa);
  unpack8(wv[8 + i], wb);
#pragma unroll
  for (int e = 0; e < 8; ++e) ss[e] = a[e] * a[e] + b[e] * b[e];
#pragma unroll
  for (int o = 4; o > 0; o >>= 1)
#pragma unroll
    for (int e = 0; e < 8; ++e) ss[e] += __shfl_xor(ss[e], o);
#pragma unroll
  for (int o = 4; o > 0; o >>= 1)
#pragma unroll
    for (int e = 0; e < o; ++e) ss[e] += ss[e + o];
  if (unit >= units) return;   // (after the shuffles)
  if (isv) {
    uint4* dst = reinterpret_cast<uint4*>(v + (t * hkv + (head - hq - hkv)) * kHeadDim);
    dst[i] = xa;
    dst[8 + i] = xb;
    return;
  }
  const float r = rsqrtf(ss[0] * (1.0f / kHeadDim) + eps);
  const float cc[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  const float sn[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
  auto scaled = [&](float (&x)[8], const float (&w)[8]) {   // bf16(bf16(x r) w)
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= r;
    round8(x);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= w[e];
    round8(x);
  };
  scaled(a, wa);
  scaled(b, wb);
  float y1[8], y2[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    y1[e] = a[e] * cc[e] - b[e] * sn[e];
    y2[e] = b[e] * cc[e] + a[e] * sn[e];
  }
  uint4* dst = reinterpret_cast<uint4*>(isq ? q + (t * hq + head) * kHeadDim : k + (t * hkv + (head - hq)) * kHeadDim);
  dst[i] = pack8(y1);
  dst[8 + i] = pack8(y2);
}

// The same for a few tokens, where a wavefront per head is as fast, and for
// operands that are not 16-byte aligned: lane l holds dims l and l + 64.
constexpr int kRopeWaves = 4;
__global__ __launch_bounds__(kRopeWaves * kWave) void qk_norm_rope_kernel(
    const uint16_t* __restrict__ qkv, int hq, int hkv, const uint16_t* __restrict__ qw,
    const uint16_t* __restrict__ kw, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
    int max_pos, const int64_t* __restrict__ positions, float eps, uint16_t* __restrict__ q,
    uint16_t* __restrict__ k, uint16_t* __restrict__ v) {
#pragma clang fp contract(off)
  const int64_t t = blockIdx.x;
  const int nh = hq + 2 * hkv;
  const int head = blockIdx.y * kRopeWaves + static_cast<int>(threadIdx.x / kWave);
  if (head >= nh) return;
  const int lane = threadIdx.x & (kWave - 1);
  const uint16_t* src = qkv + (t * nh + head) * kHeadDim;
  if (head >= hq + hkv) {
    uint16_t* dst = v + (t * hkv + (head - hq - hkv)) * kHeadDim;
    dst[lane] = src[lane];
    dst[lane + 64] = src[lane + 64];
    return;
  }
  const bool isq = head < hq;
  const float a0 = bf16_to_f32(src[lane]);
  const float b0 = bf16_to_f32(src[lane + 64]);
  float ss = a0 * a0 + b0 * b0;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  const float r = rsqrtf(ss * (1.0f / kHeadDim) + eps);
  const uint16_t* wv = isq ? qw : kw;
  const float a = round_bf16(round_bf16(a0 * r) * bf16_to_f32(wv[lane]));
  const float b = round_bf16(round_bf16(b0 * r) * bf16_to_f32(wv[lane + 64]));
  int64_t pos = positions[t];
  pos = pos < 0 ? 0 : (pos >= max_pos ? max_pos - 1 : pos);
  const float c = cos_t[pos * (kHeadDim / 2) + lane];
  const float s = sin_t[pos * (kHeadDim / 2) + lane];
  const float y1 = a * c - b * s;
  const float y2 = b * c + a * s;
  uint16_t* dst = isq ? q + (t * hq + head) * kHeadDim : k + (t * hkv + (head - hq)) * kHeadDim;
  dst[lane] = f32_to_bf16(y1);
  dst[lane + 64] = f32_to_bf16(y2);
}

// One thread per 8 outputs.
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gu, uint16_t* __restrict__ out,
                                                       int64_t chunks, int inter) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= chunks) return;
  const int per_row = inter >> 3;
  const int64_t row = i / per_row;
  const int c = static_cast<int>(i % per_row);
  const uint16_t* g0 = gu + row * 2 * inter;
  float g[8], u[8], o[8];
  unpack8(reinterpret_cast<const uint4*>(g0)[c], g);
  unpack8(reinterpret_cast<const uint4*>(g0 + inter)[c], u);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = g[e] / (1.0f + expf(-g[e]));
  round8(o);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] *= u[e];
  reinterpret_cast<uint4*>(out + row * inter)[c] = pack8(o);
}

// y[m][r] = sum_k x[m][k] w[r][k] (nn.Linear without bias) for up to 4 rows
// of x.  A workgroup owns ROWS weight rows; its 4 wavefronts take a quarter
// of k each, every lane streaming one 16-byte chunk of each row per
// iteration with the matching x chunk (L1 / L2 hits); fp32 fma
// accumulation, a wavefront sum, then the 4 quarters summed through LDS in
// wavefront order.  One chunk per row in flight keeps the wave small (more
// resident wavefronts per CU), which on gfx950 streams the weights faster
// than deeper per-wave unrolling: 5.5-5.8 TB/s on a 19456 x 2560 matrix
// against 2.7 TB/s with 8 chunks per row in flight.  HBM-bound: the weight
// matrix is read once.  The per-lane chunk order and the reduction order
// depend only on k, so a row's sum is the same for every ROWS.
constexpr int kGemvRows = 2;      // plain GEMV: rows per workgroup
constexpr int kGemvSiluRows = 4;  // gate|up: 2 gate rows + the 2 matching up rows

__device__ __forceinline__ float dot8(const uint4& a, const uint4& b, float acc) {
  float fa[8], fb[8];
  unpack8(a, fa);
  unpack8(b, fb);
#pragma unroll
  for (int e = 0; e < 8; ++e) acc = __builtin_fmaf(fa[e], fb[e], acc);
  return acc;
}

// SILU: w is the fused gate|up weight [2 n][k]; the workgroup's rows are gate
// rows r0 .. r0 + ROWS/2 - 1 and the matching up rows n + r0 ..; the epilogue
// writes bf16(bf16(silu(bf16 g)) * bf16 u) for rows r0 .. of y [m][n] (the
// rounding points of a bf16 GEMM followed by nkv_silu_mul).
template <int MR, int ROWS, bool SILU = false>
__global__ __launch_bounds__(256) void gemv_kernel(const uint16_t* __restrict__ w, const uint16_t* __restrict__ x,
                                                   uint16_t* __restrict__ y, int n, int k) {
  constexpr int kOut = SILU ? ROWS / 2 : ROWS;  // output rows per workgroup
  __shared__ float s_red[4][MR][ROWS];
  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int r0 = blockIdx.x * kOut;
  const int nc = k >> 3;
  const int cbeg = static_cast<int>(static_cast<int64_t>(nc) * wave / 4);
  const int cend = static_cast<int>(static_cast<int64_t>(nc) * (wave + 1) / 4);
  const uint4* wr[ROWS];
#pragma unroll
  for (int j = 0; j < ROWS; ++j) {
    // rows past n re-read the last row (not stored)
    const int r = SILU ? min(r0 + j % kOut, n - 1) + (j / kOut) * n : min(r0 + j, n - 1);
    wr[j] = reinterpret_cast<const uint4*>(w + static_cast<int64_t>(r) * k);
  }
  const uint4* xv = reinterpret_cast<const uint4*>(x);
  float acc[MR][ROWS];
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int j = 0; j < ROWS; ++j) acc[m][j] = 0.0f;
  for (int c = cbeg + lane; c < cend; c += kWave) {
    uint4 a[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; ++j) a[j] = wr[j][c];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const uint4 xm = xv[static_cast<int64_t>(m) * nc + c];
#pragma unroll
      for (int j = 0; j < ROWS; ++j) acc[m][j] = dot8(a[j], xm, acc[m][j]);
    }
  }
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int j = 0; j < ROWS; ++j)
#pragma unroll
      for (int o = kWave / 2; o > 0; o >>= 1) acc[m][j] += __shfl_xor(acc[m][j], o);
  if (lane == 0)
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
      for (int j = 0; j < ROWS; ++j) s_red[wave][m][j] = acc[m][j];
  __syncthreads();
  if (threadIdx.x >= MR * kOut) return;
  const int m = threadIdx.x / kOut, j = threadIdx.x % kOut;
  if (r0 + j >= n) return;
  const float v = s_red[0][m][j] + s_red[1][m][j] + s_red[2][m][j] + s_red[3][m][j];
  if constexpr (SILU) {
    const float g = round_bf16(v);
    const float u = round_bf16(s_red[0][m][kOut + j] + s_red[1][m][kOut + j] + s_red[2][m][kOut + j] +
                               s_red[3][m][kOut + j]);
    y[static_cast<int64_t>(m) * n + r0 + j] = f32_to_bf16(round_bf16(g / (1.0f + expf(-g))) * u);
  } else {
    y[static_cast<int64_t>(m) * n + r0 + j] = f32_to_bf16(v);
  }
}

template <int MR>
void launch_gemv_silu(const uint16_t* w, const uint16_t* x, uint16_t* y, int n, int k, hipStream_t s) {
  constexpr int rows_per_wg = kGemvSiluRows / 2;
  hipLaunchKernelGGL((gemv_kernel<MR, kGemvSiluRows, true>), dim3((n + rows_per_wg - 1) / rows_per_wg), dim3(256), 0,
                     s, w, x, y, n, k);
}

template <int MR>
void launch_gemv(const uint16_t* w, const uint16_t* x, uint16_t* y, int n, int k, hipStream_t s) {
  hipLaunchKernelGGL((gemv_kernel<MR, kGemvRows>), dim3((n + kGemvRows - 1) / kGemvRows), dim3(256), 0, s, w, x, y, n,
                     k);
}

// Sum of x over the wavefront, in every lane, without the LDS pipeline: row
// rotations within 16 lanes, then the row swaps.
__device__ __forceinline__ float wave_sum(float x) {
  x += row_ror<8>(x);
  x += row_ror<4>(x);
  x += row_ror<2>(x);
  x += row_ror<1>(x);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// RMSNorm (+ residual add) of one row and the GEMV of the normalised row in
// one launch, for decode steps, where a norm launch of its own costs 4.2-4.9
// us.  In a captured chain over 1.2 GB of distinct weights, norm + gemv_kernel
// against this (us): 6144 rows of k = 512 7.1 / 4.1, 1024 7.5 / 5.2, 1536
// 8.1 / 6.5, 2048 9.0 / 7.9, 2560 11.4 / 9.3, 3072 12.3 / 10.8, 4096 14.5 /
// 13.3; gate|up of 6 k rows, k = 1024 7.4 / 5.4, 2048 13.7 / 10.8, 2560 19.7 /
// 16.4, 3072 25.5 / 22.3, 4096 38.7 / 37.0 (no size between them is slower).
// The gain ends where a row's chunks fill the registers: k = 4096 holds 156
// of the 168 of three wavefronts a SIMD, so longer rows take the two launches.
// Resident workgroups (one round) take a row pair per wavefront at a time --
// two consecutive rows, or with SILU a gate row and its up row -- the pair's
// NCH = ceil(k / 512) chunks a lane all in flight at once (a second pair in
// flight behind them spills or halves the residency: 12.7 and 28 us).
// Each workgroup computes the norm once, as rmsnorm_kernel does (the same
// bits), while its first pair is in flight.  (The norm as a prologue of
// gemv_kernel's thousands of small workgroups cost more than the launch it
// saved: q|k|v 13.6 against 12.2 us, gate|up 34 against 24.)
struct GemvNorm {
  const uint16_t* x;
  const uint16_t* res;   // residual added first, or null
  const uint16_t* w;     // norm weight
  uint16_t* res_out;     // bf16(x + res), or null
  float eps;
};
constexpr int kNgThreads = kNormThreads;
constexpr int kNgWaves = kNgThreads / kWave;
// resident wavefronts per SIMD the kernel is built for and launched with
constexpr int norm_gemv_waves(int nch) { return nch <= 5 ? 4 : 3; }

template <int NCH, bool SILU>
__global__ __launch_bounds__(kNgThreads, norm_gemv_waves(NCH)) void norm_gemv_kernel(
    const uint16_t* __restrict__ w, const GemvNorm a, uint16_t* __restrict__ y, int n, int k) {
  __shared__ uint4 s_x[NCH * kWave];
  __shared__ float s_part[kNormThreads / kWave];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x & (kWave - 1);
  const int nc = k >> 3;
  const int units = SILU ? n : (n + 1) >> 1;
  const int stride = gridDim.x * kNgWaves;
  int u = blockIdx.x * kNgWaves + wave;
  uint4 b[2][NCH];
  auto load = [&](int unit) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = SILU ? unit + j * n : min(2 * unit + j, n - 1);
      const uint4* wr = reinterpret_cast<const uint4*>(w + static_cast<int64_t>(row) * k);
#pragma unroll
      for (int i = 0; i < NCH; ++i) b[j][i] = wr[min(i * kWave + lane, nc - 1)];   // past the row: its last chunk, masked below
    }
  };
  load(min(u, units - 1));

  // the normalised row, zero-padded to NCH chunks a lane
  {
    const uint4* xr = reinterpret_cast<const uint4*>(a.x);
    const uint4* rr = reinterpret_cast<const uint4*>(a.res);
    const uint4* nw = reinterpret_cast<const uint4*>(a.w);
    uint4* ro = blockIdx.x == 0 ? reinterpret_cast<uint4*>(a.res_out) : nullptr;
    constexpr int kMine = (NCH * kWave + kNormThreads - 1) / kNormThreads;
    float v[kMine][8];
    uint4 wv[kMine];
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
      const int d = threadIdx.x + i * kNormThreads;
      if (d < nc) {
        wv[i] = nw[d];
        norm_load(xr[d], rr, ro, d, v[i], ss);
      }
    }
    const float r = norm_scale(ss, s_part, wave, lane, k, a.eps);
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
      const int d = threadIdx.x + i * kNormThreads;
      if (d < nc)
        s_x[d] = norm_apply(v[i], r, wv[i]);
      else if (d < NCH * kWave)
        s_x[d] = make_uint4(0u, 0u, 0u, 0u);
    }
    __syncthreads();
  }
  uint4 xv[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) xv[i] = s_x[i * kWave + lane];

  const bool in_row = (NCH - 1) * kWave + lane < nc;   // of the lane's last chunk
  auto finish = [&](int unit) {
    float acc[2] = {0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)   // (a masked chunk: an infinite weight times x = 0 would be NaN)
        acc[j] = dot8(i + 1 < NCH ? b[j][i] : and_mask(b[j][i], in_row), xv[i], acc[j]);
    const float v0 = wave_sum(acc[0]), v1 = wave_sum(acc[1]);
    if (lane != 0) return;
    if constexpr (SILU) {
      const float g = round_bf16(v0), up = round_bf16(v1);
      y[unit] = f32_to_bf16(round_bf16(g / (1.0f + expf(-g))) * up);
    } else {
      y[2 * unit] = f32_to_bf16(v0);
      if (2 * unit + 1 < n) y[2 * unit + 1] = f32_to_bf16(v1);
    }
  };
  while (u < units) {
    finish(u);
    u += stride;
    if (u < units) load(u);
  }
}

// Whether a row of k elements fits the norm GEMV's registers, and its launch.
constexpr int kNgMaxK = 8 * 8 * kWave;
template <bool SILU>
int launch_norm_gemv(const uint16_t* w, const GemvNorm& a, uint16_t* y, int n, int k, hipStream_t s) {
  const int cus = device_cus();
  const int units = SILU ? n : (n + 1) / 2;
  auto go = [&](auto kern, int waves) {   // waves per SIMD = workgroups per CU
    const int grid = std::min(waves * (cus > 0 ? cus : 256), (units + kNgWaves - 1) / kNgWaves);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kNgThreads), 0, s, w, a, y, n, k);
  };
  switch ((k / 8 + kWave - 1) / kWave) {
    case 1: go(norm_gemv_kernel<1, SILU>, norm_gemv_waves(1)); return 0;
    case 2: go(norm_gemv_kernel<2, SILU>, norm_gemv_waves(2)); return 0;
    case 3: go(norm_gemv_kernel<3, SILU>, norm_gemv_waves(3)); return 0;
    case 4: go(norm_gemv_kernel<4, SILU>, norm_gemv_waves(4)); return 0;
    case 5: go(norm_gemv_kernel<5, SILU>, norm_gemv_waves(5)); return 0;
    case 6: go(norm_gemv_kernel<6, SILU>, norm_gemv_waves(6)); return 0;
    case 7: go(norm_gemv_kernel<7, SILU>, norm_gemv_waves(7)); return 0;
    case 8: go(norm_gemv_kernel<8, SILU>, norm_gemv_waves(8)); return 0;
    default: return -1;   // k beyond kNgMaxK: refused by the entry points
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace nkv

using namespace nkv;

extern "C" int nkv_rmsnorm(const uint16_t* x, const uint16_t* residual, const uint16_t* weight, uint16_t* out,
                           uint16_t* residual_out, int rows, int n, float eps, void* stream) {
  NKV_CHECK_ARG(x != nullptr && weight != nullptr && out != nullptr, "nkv_rmsnorm: x, weight and out must be non-NULL");
  NKV_CHECK_ARG(rows >= 1, "nkv_rmsnorm: rows must be >= 1 (got %d)", rows);
  NKV_CHECK_ARG(n >= 8 && n % 8 == 0 && n <= kMaxNormWidth, "nkv_rmsnorm: n must be a multiple of 8 in [8, %d] (got %d)",
                kMaxNormWidth, n);
  NKV_CHECK_ARG(aligned16(x) && aligned16(weight) && aligned16(out) && (!residual || aligned16(residual)) &&
                    (!residual_out || aligned16(residual_out)),
                "nkv_rmsnorm: every buffer must be 16-byte aligned");
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(rows), dim3(kNormThreads), 0, reinterpret_cast<hipStream_t>(stream), x,
                     residual, weight, out, residual_out, n, eps);
  return launch_status("nkv_rmsnorm");
}

extern "C" int nkv_qk_norm_rope(const uint16_t* qkv, int rows, int num_heads, int num_kv_heads, const uint16_t* q_weight,
                                const uint16_t* k_weight, const float* cos_table, const float* sin_table,
                                int max_position, const int64_t* positions, float eps, uint16_t* q, uint16_t* k,
                                uint16_t* v, void* stream) {
  NKV_CHECK_ARG(qkv != nullptr && q_weight != nullptr && k_weight != nullptr && cos_table != nullptr &&
                    sin_table != nullptr && positions != nullptr && q != nullptr && k != nullptr && v != nullptr,
                "nkv_qk_norm_rope: every pointer must be non-NULL");
  NKV_CHECK_ARG(rows >= 1 && num_heads >= 1 && num_kv_heads >= 1 && max_position >= 1,
                "nkv_qk_norm_rope: rows, heads and max_position must be >= 1");
  const int nh = num_heads + 2 * num_kv_heads;
  // us, one wavefront per head / eight lanes per head, 48 heads: 1 row 2.30 /
  // 2.38, 64 rows 2.87 / 2.90, 300 rows 5.8 / 4.2, 3000 rows 45 / 18.7
  const int64_t units = static_cast<int64_t>(rows) * nh;
  if (rows >= kRopeRows && units < INT32_MAX && aligned16(qkv) && aligned16(q_weight) && aligned16(k_weight) && aligned16(cos_table) && aligned16(sin_table) &&
      aligned16(q) && aligned16(k) && aligned16(v)) {
    constexpr int per = kRopeThreads / 8;
    hipLaunchKernelGGL(qk_norm_rope8_kernel, dim3(static_cast<unsigned>((units + per - 1) / per)), dim3(kRopeThreads),
                       0, reinterpret_cast<hipStream_t>(stream), qkv, static_cast<uint32_t>(units), num_heads, num_kv_heads, q_weight,
                       k_weight, cos_table, sin_table, max_position, positions, eps, q, k, v);
    return launch_status("nkv_qk_norm_rope");
  }
  hipLaunchKernelGGL(qk_norm_rope_kernel, dim3(rows, (nh + kRopeWaves - 1) / kRopeWaves), dim3(kRopeWaves * kWave), 0,
                     reinterpret_cast<hipStream_t>(stream), qkv, num_heads, num_kv_heads, q_weight, k_weight,
                     cos_table, sin_table, max_position, positions, eps, q, k, v);
  return launch_status("nkv_qk_norm_rope");
}

extern "C" int nkv_silu_mul(const uint16_t* gate_up, uint16_t* out, int rows, int intermediate, void* stream) {
  NKV_CHECK_ARG(gate_up != nullptr && out != nullptr, "nkv_silu_mul: gate_up and out must be non-NULL");
  NKV_CHECK_ARG(rows >= 1 && intermediate >= 8 && intermediate % 8 == 0,
                "nkv_silu_mul: rows >= 1 and intermediate a positive multiple of 8 (got %d, %d)", rows, intermediate);
  NKV_CHECK_ARG(aligned16(gate_up) && aligned16(out), "nkv_silu_mul: buffers must be 16-byte aligned");
  const int64_t chunks = static_cast<int64_t>(rows) * (intermediate / 8);
  hipLaunchKernelGGL(silu_mul_kernel, dim3(static_cast<unsigned>((chunks + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), gate_up, out, chunks, intermediate);
  return launch_status("nkv_silu_mul");
}

extern "C" int nkv_gemv(const uint16_t* weight, const uint16_t* x, uint16_t* y, int m, int n, int k, void* stream) {
  NKV_CHECK_ARG(weight != nullptr && x != nullptr && y != nullptr, "nkv_gemv: weight, x and y must be non-NULL");
  NKV_CHECK_ARG(m >= 1 && m <= 4, "nkv_gemv: m must be in [1, 4] (got %d)", m);
  NKV_CHECK_ARG(n >= 1 && k >= 8 && k % 8 == 0, "nkv_gemv: n >= 1 and k a positive multiple of 8 (got %d, %d)", n, k);
  NKV_CHECK_ARG(aligned16(weight) && aligned16(x), "nkv_gemv: weight and x must be 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (m) {
    case 1: launch_gemv<1>(weight, x, y, n, k, s); break;
    case 2: launch_gemv<2>(weight, x, y, n, k, s); break;
    case 3: launch_gemv<3>(weight, x, y, n, k, s); break;
    default: launch_gemv<4>(weight, x, y, n, k, s); break;
  }
  return launch_status("nkv_gemv");
}

extern "C" int nkv_gemv_silu_mul(const uint16_t* gate_up_weight, const uint16_t* x, uint16_t* y, int m,
                                 int intermediate, int k, void* stream) {
  NKV_CHECK_ARG(gate_up_weight != nullptr && x != nullptr && y != nullptr,
                "nkv_gemv_silu_mul: gate_up_weight, x and y must be non-NULL");
  NKV_CHECK_ARG(m >= 1 && m <= 4, "nkv_gemv_silu_mul: m must be in [1, 4] (got %d)", m);
  NKV_CHECK_ARG(intermediate >= 1 && k >= 8 && k % 8 == 0,
                "nkv_gemv_silu_mul: intermediate >= 1 and k a positive multiple of 8 (got %d, %d)", intermediate, k);
  NKV_CHECK_ARG(aligned16(gate_up_weight) && aligned16(x), "nkv_gemv_silu_mul: weight and x must be 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (m) {
    case 1: launch_gemv_silu<1>(gate_up_weight, x, y, intermediate, k, s); break;
    case 2: launch_gemv_silu<2>(gate_up_weight, x, y, intermediate, k, s); break;
    case 3: launch_gemv_silu<3>(gate_up_weight, x, y, intermediate, k, s); break;
    default: launch_gemv_silu<4>(gate_up_weight, x, y, intermediate, k, s); break;
  }
  return launch_status("nkv_gemv_silu_mul");
}

namespace {

// Whether two ranges of bytes have none in common (NULL: no range).
bool apart(const void* a, int64_t na, const void* b, int64_t nb) {
  const char *pa = static_cast<const char*>(a), *pb = static_cast<const char*>(b);
  return !a || !b || pa + na <= pb || pb + nb <= pa;
}

int check_norm_gemv(const char* who, const uint16_t* weight, const uint16_t* x, const uint16_t* residual,
                    const uint16_t* norm_weight, const uint16_t* residual_out, const uint16_t* y, int n, int k) {
  NKV_CHECK_ARG(weight != nullptr && x != nullptr && norm_weight != nullptr && y != nullptr,
                "%s: weight, x, norm_weight and y must be non-NULL", who);
  NKV_CHECK_ARG(n >= 1 && k >= 8 && k % 8 == 0 && k <= kNgMaxK,
                "%s: n >= 1 and k a multiple of 8 in [8, %d] (got %d, %d)", who, kNgMaxK, n, k);
  NKV_CHECK_ARG(aligned16(weight) && aligned16(x) && aligned16(norm_weight) && (!residual || aligned16(residual)) &&
                    (!residual_out || aligned16(residual_out)),
                "%s: every input and residual_out must be 16-byte aligned", who);
  // every workgroup reads x, residual and norm_weight for itself while others
  // write y and one writes residual_out
  const int64_t row = 2 * static_cast<int64_t>(k), out = 2 * static_cast<int64_t>(n);
  for (const uint16_t* in : {x, residual, norm_weight}) {
    NKV_CHECK_ARG(apart(y, out, in, row), "%s: y must not overlap x, residual or norm_weight", who);
    NKV_CHECK_ARG(apart(residual_out, row, in, row), "%s: residual_out must not overlap x, residual or norm_weight", who);
  }
  NKV_CHECK_ARG(apart(y, out, residual_out, row), "%s: y must not overlap residual_out", who);
  return NKV_OK;
}

}  // namespace

extern "C" int nkv_norm_gemv(const uint16_t* weight, const uint16_t* x, const uint16_t* residual,
                             const uint16_t* norm_weight, float eps, uint16_t* y, uint16_t* residual_out, int n, int k,
                             void* stream) {
  const int rc = check_norm_gemv("nkv_norm_gemv", weight, x, residual, norm_weight, residual_out, y, n, k);
  if (rc != NKV_OK) return rc;
  launch_norm_gemv<false>(weight, GemvNorm{x, residual, norm_weight, residual_out, eps}, y, n, k,
                          reinterpret_cast<hipStream_t>(stream));
  return launch_status("nkv_norm_gemv");
}

extern "C" int nkv_norm_gemv_silu_mul(const uint16_t* gate_up_weight, const uint16_t* x, const uint16_t* residual,
                                      const uint16_t* norm_weight, float eps, uint16_t* y, uint16_t* residual_out,
                                      int intermediate, int k, void* stream) {
  const int rc = check_norm_gemv("nkv_norm_gemv_silu_mul", gate_up_weight, x, residual, norm_weight, residual_out, y,
                                 intermediate, k);
  if (rc != NKV_OK) return rc;
  launch_norm_gemv<true>(gate_up_weight, GemvNorm{x, residual, norm_weight, residual_out, eps}, y, intermediate, k,
                         reinterpret_cast<hipStream_t>(stream));
  return launch_status("nkv_norm_gemv_silu_mul");
}
