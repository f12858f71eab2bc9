// HBM store maintenance: appending prefill chunks to the history (with the
// int8 schemes), building block representatives, updating the recent window
// and computing prefill query summaries.  These run once per prefill chunk
// (or verify commit), not per decode step.
#include <algorithm>

#include "nkv_common.h"

namespace nkv {
namespace {

constexpr int kStoreThreads = 256;

// bf16 value a over fp32 value d, correctly rounded to fp32, from inv = 1.0 / d
// in fp64.  The product's relative error is below 2^-52, and a / d is at least
// 2^-49 away from every midpoint of two fp32 values (a nonzero difference
// a - m d of an 8-bit, a 25-bit and a 24-bit significand; a quotient with
// exactly 25 bits would need a product m d of at least 25 bits to equal a), so
// the second rounding lands where the quotient's own would.  Three
// instructions against about ten of an fp32 division.
__device__ __forceinline__ float div_bf16(float a, double inv) {
  return static_cast<float>(static_cast<double>(a) * inv);
}

// ---------------------------------------------------------------------------
// int8 K scale from the first chunk: m12_runtime.py:463-467
//   k_scale[h][d] = max(amax_t |k[t][h][d]|, 1e-8) / 127
// One workgroup per (32 dims of one KV head, layer): 4 lanes cover the 64
// bytes of a row, 256 row groups the tokens, and the maxima meet in LDS, so no
// cleared buffer, atomics or second pass (one launch instead of three:
// 2048 tokens, one layer, 25.4 -> 7.6 us).
// SPLIT: blockIdx.z's part of the tokens, its maxima folded into the cleared
// buffer (non-negative floats order as their bits do); k_scale_finish_kernel
// then turns them into scales.
// ---------------------------------------------------------------------------
constexpr int kScaleThreads = 1024;
constexpr int kScaleDims = 32;
template <bool SPLIT>
__global__ __launch_bounds__(kScaleThreads) void k_scale_kernel(const uint16_t* __restrict__ k, int64_t kv_ls, int T,
                                                                int hkv, float* __restrict__ k_scale) {
  __shared__ uint32_t s_max[kScaleDims];
  const int c = threadIdx.x & 3;
  const int d0 = blockIdx.x * kScaleDims + 8 * c;   // column of [hkv * 128]
  const int layer = blockIdx.y;
  if (threadIdx.x < kScaleDims) s_max[threadIdx.x] = 0u;
  const uint16_t* src = k + kv_ls * layer + d0;
  const int64_t ld = static_cast<int64_t>(hkv) * kHeadDim;
  float m[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int kStep = kScaleThreads / 4, kUnroll = 4;
  int lo = 0, hi = T;
  if constexpr (SPLIT) {
    lo = static_cast<int>(static_cast<int64_t>(T) * blockIdx.z / gridDim.z);
    hi = static_cast<int>(static_cast<int64_t>(T) * (blockIdx.z + 1) / gridDim.z);
  }
  for (int t = lo + (threadIdx.x >> 2); t < hi; t += kStep * kUnroll) {
    uint4 v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)   // past the end: the last row again
      v[u] = *reinterpret_cast<const uint4*>(src + min(t + u * kStep, hi - 1) * ld);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      float f[8];
      unpack8(v[u], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) m[e] = fmaxf(m[e], fabsf(f[e]));
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int o = 4; o < kWave; o <<= 1) m[e] = fmaxf(m[e], __shfl_xor(m[e], o));
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) < 4)
#pragma unroll
    for (int e = 0; e < 8; ++e) atomicMax(&s_max[8 * c + e], __float_as_uint(m[e]));   // non-negative floats
  __syncthreads();
  if (threadIdx.x < kScaleDims) {
    float* dst = k_scale + static_cast<int64_t>(layer) * ld + blockIdx.x * kScaleDims + threadIdx.x;
    if constexpr (SPLIT)
      atomicMax(reinterpret_cast<uint32_t*>(dst), s_max[threadIdx.x]);
    else
      *dst = fmaxf(__uint_as_float(s_max[threadIdx.x]), 1e-8f) / 127.0f;
  }
}

__global__ __launch_bounds__(kStoreThreads) void k_scale_clear_kernel(float* __restrict__ k_scale, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kStoreThreads + threadIdx.x;
  if (i < n) k_scale[i] = 0.0f;
}

__global__ __launch_bounds__(kStoreThreads) void k_scale_finish_kernel(float* __restrict__ k_scale, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kStoreThreads + threadIdx.x;
  if (i < n) k_scale[i] = fmaxf(k_scale[i], 1e-8f) / 127.0f;
}

// ---------------------------------------------------------------------------
// A prefill chunk into the store: one wavefront per (block, KV head, layer)
// reads the block's keys and values once and writes whichever of these the
// call asks for:
//   HIST: the history block (bf16, or quantised), the sink and the recent
//         window's share of the block's tokens;
//   REPS: the block's representatives (m12_runtime.py:354-395).
// Bound by memory: K and V are read and written once, 64 KiB a wavefront in
// 1 KiB instructions (4 token rows x 256 B), all loads in flight before the
// first store; one wavefront per workgroup so that the 17 KiB of LDS the
// representatives need allow several per CU.  36 layers x 4096 tokens, bf16:
// 248 us for 1.2 GB (4.9 TB/s, the rate of a large copy) against 575 us for
// separate history, representative and recent-window kernels, which read K
// twice with 16-byte pieces of a row per lane and held 33 KiB of LDS a
// wavefront; one layer x 1501 tokens 34.3 -> 12.1 us, a chain of dependent
// sums and selections in one wavefront (1.5 us of it was argmax by LDS
// shuffles).
// ---------------------------------------------------------------------------
struct StoreArgs {
  const uint16_t* k;
  const uint16_t* v;
  int64_t kv_ls;
  int T, start_block, hkv, cap, r;
  void* hist_k;
  void* hist_v;
  int64_t hist_ls;
  const float* k_scale;
  float* v_scale;
  uint16_t* k_tscale;
  uint16_t* v_tscale;
  uint16_t* sink_k;
  uint16_t* sink_v;
  int64_t sink_ls;
  int S, sink_n;              // the first sink_n tokens go to the sink
  uint16_t* rec_k;
  uint16_t* rec_v;
  int64_t rec_ls;
  int R, rec_lo, rec_n, rec_slot;   // tokens rec_lo .. + rec_n go to ring slots rec_slot .. (mod R)
  uint16_t* reps;
  int64_t reps_ls;
};

// int8 codes of 8 values: clamp(round-half-even(x / s), -127, 127)
__device__ __forceinline__ uint2 quant8(const float (&x)[8], const double (&inv)[8]) {
  uint32_t w[2] = {0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float r = rintf(div_bf16(x[e], inv[e]));
    r = fminf(fmaxf(r, -127.0f), 127.0f);
    w[e >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(static_cast<int8_t>(static_cast<int>(r)))) << (8 * (e & 3));
  }
  return make_uint2(w[0], w[1]);
}

__device__ __forceinline__ float amax8(const uint4& c) {
  float f[8];
  unpack8(c, f);
  float m = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(f[e]));
  return m;
}

constexpr int kRawRow = 17;               // 16-byte chunks per key row in LDS (one of padding)
constexpr int kDirRow = kBlock + 1;       // floats per key row of half the directions in LDS

// The largest x of the wavefront in every lane, without the LDS pipeline (row
// rotations within 16 lanes, then the row swaps), and the first lane holding
// it; lane 0 where every x is NaN.
__device__ __forceinline__ int first_argmax(float x) {
  float m = x;
  m = fmaxf(m, row_ror<8>(m));
  m = fmaxf(m, row_ror<4>(m));
  m = fmaxf(m, row_ror<2>(m));
  m = fmaxf(m, row_ror<1>(m));
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  m = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  m = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
  const unsigned long long at = __ballot(x == m);
  return at ? __builtin_ctzll(at) : 0;
}

// Representatives of the 64 keys whose chunks this wavefront holds (kv[i]: key
// 4 i + lane / 16, dims 8 (lane & 15) .. + 7); lane l then owns key l.  The
// first is the first argmax of the cosine to the mean direction, the others
// the first argmin of the largest cosine to the chosen ones; every sum runs
// in ascending order in one lane.
__device__ __forceinline__ void pick_reps(const uint4 (&kv)[16], uint4* s_raw, int lane, int r,
                                          const uint16_t* kl, int64_t row_ld, int t0, int T, uint16_t* dst) {
  float* s_dir = reinterpret_cast<float*>(s_raw);
  float* s_mean = s_dir + kBlock * kDirRow;
  const int ln = lane & 15, lg = lane >> 4;
#pragma unroll
  for (int i = 0; i < 16; ++i) s_raw[(4 * i + lg) * kRawRow + ln] = kv[i];
  wave_lds_sync();
  // normalise this lane's key (F.normalize: x / max(||x||, 1e-12))
  float x[kHeadDim];
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    float f[8];
    unpack8(s_raw[lane * kRawRow + c], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[8 * c + e] = f[e];
  }
  float ss = 0.0f;
#pragma unroll
  for (int d = 0; d < kHeadDim; ++d) ss = __builtin_fmaf(x[d], x[d], ss);
  const double inv = 1.0 / static_cast<double>(fmaxf(sqrtf(ss), 1e-12f));
#pragma unroll
  for (int d = 0; d < kHeadDim; ++d) x[d] = div_bf16(x[d], inv);

  // mean direction over the block's keys, 64 dims at a time through LDS
  float m[2] = {0.0f, 0.0f};
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    wave_lds_sync();   // the keys (the other half) have been read
#pragma unroll
    for (int d = 0; d < kBlock; ++d) s_dir[lane * kDirRow + d] = x[kBlock * half + d];
    wave_lds_sync();
#pragma unroll 16
    for (int tt = 0; tt < kBlock; ++tt) m[half] += s_dir[tt * kDirRow + lane];
  }
  m[0] *= (1.0f / kBlock);
  m[1] *= (1.0f / kBlock);
  float mss = m[0] * m[0] + m[1] * m[1];
  for (int o = 32; o > 0; o >>= 1) mss += __shfl_xor(mss, o);
  const float mden = fmaxf(sqrtf(mss), 1e-12f);
  s_mean[lane] = m[0] / mden;
  s_mean[lane + 64] = m[1] / mden;
  wave_lds_sync();

  // cosine of this lane's key to the direction at `row` (every lane reads the
  // same LDS address)
  auto cosine = [&](const float* row) {
    float c = 0.0f;
#pragma unroll
    for (int d = 0; d < kHeadDim; d += 4) {
      const float4 w = *reinterpret_cast<const float4*>(row + d);
      c = __builtin_fmaf(x[d], w.x, c);
      c = __builtin_fmaf(x[d + 1], w.y, c);
      c = __builtin_fmaf(x[d + 2], w.z, c);
      c = __builtin_fmaf(x[d + 3], w.w, c);
    }
    return c;
  };
  // chosen keys: lane group g keeps the picks of representatives g and 4 + g
  int pick0 = 0, pick1 = 0;
  const int bi = first_argmax(cosine(s_mean));
  if (lg == 0) pick0 = bi;
  int last = bi;
  bool is_chosen = (lane == bi);
  float maxcos = -INFINITY;
  for (int step = 1; step < r; ++step) {
    wave_lds_sync();   // the previous direction has been read
    if (lane == last) {
#pragma unroll
      for (int d = 0; d < kHeadDim; d += 4)
        *reinterpret_cast<float4*>(s_dir + d) = make_float4(x[d], x[d + 1], x[d + 2], x[d + 3]);
    }
    wave_lds_sync();
    maxcos = fmaxf(maxcos, cosine(s_dir));
    const float val = is_chosen ? fmaxf(maxcos, 2.0f) : maxcos;
    const int vi = first_argmax(-val);   // the first smallest
    if (lg == (step & 3)) (step < 4 ? pick0 : pick1) = vi;
    last = vi;
    is_chosen = is_chosen || (lane == vi);
  }
  // the raw bf16 keys, one round trip for all of them
  auto write_rep = [&](int j, int tok) {
    if (j < r)
      reinterpret_cast<uint4*>(dst + static_cast<int64_t>(j) * kHeadDim)[ln] =
          and_mask(reinterpret_cast<const uint4*>(kl + min(t0 + tok, T - 1) * row_ld)[ln], t0 + tok < T);
  };
  write_rep(lg, pick0);
  if (r > 4) write_rep(4 + lg, pick1);
}

template <int FMT, bool HIST, bool REPS>
__global__ __launch_bounds__(kWave) void store_block_kernel(const StoreArgs a) {
  __shared__ uint4 s_raw[REPS ? kBlock * kRawRow : 1];   // keys, then half the directions + the mean
  const int b = blockIdx.x, h = blockIdx.y, layer = blockIdx.z;
  const int lane = threadIdx.x;
  const int ln = lane & 15, lg = lane >> 4;
  const int t0 = b * kBlock;
  const int blk = a.start_block + b;
  const int64_t row_ld = static_cast<int64_t>(a.hkv) * kHeadDim;
  const int64_t src = a.kv_ls * layer + static_cast<int64_t>(h) * kHeadDim + 8 * ln;
  const int lh = layer * a.hkv + h;

  // K (and V): chunk ln of rows 4 i + lg; rows past the chunk re-read its last
  // row and count as zeros
  uint4 kv[16], vv[16];
#pragma unroll
  for (int i = 0; i < 16; ++i)
    kv[i] = *reinterpret_cast<const uint4*>(a.k + src + min(t0 + 4 * i + lg, a.T - 1) * row_ld);
  if constexpr (HIST) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      vv[i] = *reinterpret_cast<const uint4*>(a.v + src + min(t0 + 4 * i + lg, a.T - 1) * row_ld);
  }
  if (t0 + kBlock > a.T) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      kv[i] = and_mask(kv[i], t0 + 4 * i + lg < a.T);
      if constexpr (HIST) vv[i] = and_mask(vv[i], t0 + 4 * i + lg < a.T);
    }
  }

  if constexpr (HIST) {
    // sink: the first min(S, T) tokens of the first chunk (m12_runtime.py:482-486)
    if (t0 < a.sink_n) {
      const int64_t o = a.sink_ls * layer + static_cast<int64_t>(h) * a.S * kHeadDim + 8 * ln;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = t0 + 4 * i + lg;
        if (t < a.sink_n) {
          *reinterpret_cast<uint4*>(a.sink_k + o + static_cast<int64_t>(t) * kHeadDim) = kv[i];
          *reinterpret_cast<uint4*>(a.sink_v + o + static_cast<int64_t>(t) * kHeadDim) = vv[i];
        }
      }
    }
    // recent window: this block's share of the chunk's last tokens
    if (t0 + kBlock > a.rec_lo && t0 < a.rec_lo + a.rec_n) {
      const int64_t o = a.rec_ls * layer + static_cast<int64_t>(h) * a.R * kHeadDim + 8 * ln;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int x = t0 + 4 * i + lg - a.rec_lo;
        if (x >= 0 && x < a.rec_n) {
          const int64_t at = o + static_cast<int64_t>((a.rec_slot + x) % a.R) * kHeadDim;
          *reinterpret_cast<uint4*>(a.rec_k + at) = kv[i];
          *reinterpret_cast<uint4*>(a.rec_v + at) = vv[i];
        }
      }
    }
    const int64_t row = a.hist_ls * layer + (static_cast<int64_t>(h) * a.cap + blk) * kBlock * kHeadDim + 8 * ln;
    if constexpr (FMT == NKV_KV_BF16) {
      uint16_t* dk = static_cast<uint16_t*>(a.hist_k) + row;
      uint16_t* dv = static_cast<uint16_t*>(a.hist_v) + row;
#pragma unroll
      for (int i = 0; i < 16; ++i) *reinterpret_cast<uint4*>(dk + (4 * i + lg) * kHeadDim) = kv[i];
#pragma unroll
      for (int i = 0; i < 16; ++i) *reinterpret_cast<uint4*>(dv + (4 * i + lg) * kHeadDim) = vv[i];
    } else {
      int8_t* dk = static_cast<int8_t*>(a.hist_k) + row;
      int8_t* dv = static_cast<int8_t*>(a.hist_v) + row;
      double ki[8], vi[8];
      if constexpr (FMT == NKV_KV_INT8_CHANNEL) {
        const float* ks = a.k_scale + static_cast<int64_t>(lh) * kHeadDim + 8 * ln;
#pragma unroll
        for (int e = 0; e < 8; ++e) ki[e] = 1.0 / static_cast<double>(ks[e]);
        // V: per-(block, head) scale over all 64 x 128 values (m12_runtime.py:469-474)
        float am = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) am = fmaxf(am, amax8(vv[i]));
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
        const float vs = fmaxf(am, 1e-8f) / 127.0f;
        if (lane == 0) a.v_scale[static_cast<int64_t>(lh) * a.cap + blk] = vs;
        const double inv = 1.0 / static_cast<double>(vs);
#pragma unroll
        for (int e = 0; e < 8; ++e) vi[e] = inv;
      }
      const int64_t ti = (static_cast<int64_t>(lh) * a.cap + blk) * kBlock;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if constexpr (FMT == NKV_KV_INT8_TOKEN) {
          // per-token fp16 scales: s = fp16(max(amax_d |x| / 127, 2^-24)) over
          // the row's 16 lanes
          float ak = amax8(kv[i]), av = amax8(vv[i]);
#pragma unroll
          for (int o = 1; o < 16; o <<= 1) {
            ak = fmaxf(ak, __shfl_xor(ak, o));
            av = fmaxf(av, __shfl_xor(av, o));
          }
          const __half hk = __float2half_rn(fmaxf(ak / 127.0f, 5.9604644775390625e-08f));
          const __half hv = __float2half_rn(fmaxf(av / 127.0f, 5.9604644775390625e-08f));
          if (ln == 0) {
            a.k_tscale[ti + 4 * i + lg] = __half_as_ushort(hk);
            a.v_tscale[ti + 4 * i + lg] = __half_as_ushort(hv);
          }
          const double ik = 1.0 / static_cast<double>(__half2float(hk));
          const double iv = 1.0 / static_cast<double>(__half2float(hv));
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            ki[e] = ik;
            vi[e] = iv;
          }
        }
        float f[8];
        unpack8(kv[i], f);
        *reinterpret_cast<uint2*>(dk + (4 * i + lg) * kHeadDim) = quant8(f, ki);
        unpack8(vv[i], f);
        *reinterpret_cast<uint2*>(dv + (4 * i + lg) * kHeadDim) = quant8(f, vi);
      }
    }
  }
  if constexpr (REPS) {
    uint16_t* dst = a.reps + a.reps_ls * layer + (static_cast<int64_t>(h) * a.cap + blk) * a.r * kHeadDim;
    pick_reps(kv, s_raw, lane, a.r, a.k + a.kv_ls * layer + static_cast<int64_t>(h) * kHeadDim, row_ld, t0, a.T, dst);
  }
}

// Selected int8 history blocks as bf16(code * scale): one workgroup per (block,
// KV head, layer), 16 codes a thread and load.  Bound by
// launch and latency for one layer (32 blocks x 8 heads: 4 MB read, 8 MB
// written), by memory for many; it takes the in-LDS conversion, its two extra
// barriers a segment included, out of every query tile of a long chunk.
template <int FMT>
__global__ __launch_bounds__(kStoreThreads) void history_bf16_kernel(
    const int8_t* __restrict__ hist_k, const int8_t* __restrict__ hist_v, int64_t hist_ls,
    const float* __restrict__ k_scale, const float* __restrict__ v_scale, const uint16_t* __restrict__ k_tscale,
    const uint16_t* __restrict__ v_tscale, int hkv, int cap, const int32_t* __restrict__ ids, int64_t ids_ls, int n_hist,
    uint16_t* __restrict__ out_k, uint16_t* __restrict__ out_v, int32_t* __restrict__ out_ids) {
  const int i = blockIdx.x, h = blockIdx.y, layer = blockIdx.z;
  const int blk = ids[ids_ls * layer + i];
  const bool ok = blk >= 0 && blk < cap;
  if (h == 0 && threadIdx.x == 0) out_ids[static_cast<int64_t>(layer) * n_hist + i] = ok ? i : -1;
  if (!ok) return;   // nothing attends it
  const int lh = layer * hkv + h;
  const int64_t src = hist_ls * layer + (static_cast<int64_t>(h) * cap + blk) * kBlock * kHeadDim;
  const int64_t dst = (static_cast<int64_t>(lh) * n_hist + i) * kBlock * kHeadDim;
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  constexpr int kPer = kBlock * kHeadDim / 16 / kStoreThreads;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int c = j * kStoreThreads + threadIdx.x;   // 16-code chunk of the block
    const int row = c >> 3, d0 = (c & 7) * 16;
    const uint4 kq = *reinterpret_cast<const uint4*>(hist_k + src + 16 * c);
    const uint4 vq = *reinterpret_cast<const uint4*>(hist_v + src + 16 * c);
    float ks[16], vs;
    if constexpr (FMT == NKV_KV_INT8_CHANNEL) {
#pragma unroll
      for (int e = 0; e < 16; ++e) ks[e] = k_scale[static_cast<int64_t>(lh) * kHeadDim + d0 + e];
      vs = v_scale[static_cast<int64_t>(lh) * cap + blk];
    } else {
      const int64_t t = (static_cast<int64_t>(lh) * cap + blk) * kBlock + row;
      const float k1 = f16_bits_to_f32(k_tscale[t]);
#pragma unroll
      for (int e = 0; e < 16; ++e) ks[e] = k1;
      vs = f16_bits_to_f32(v_tscale[t]);
    }
    auto put = [&](const uint4& q, auto scale, uint16_t* out) {
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
      uint32_t o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t two = w[e >> 1] >> (16 * (e & 1));
        const bf16x2 b = {static_cast<__bf16>(static_cast<float>(static_cast<int8_t>(two & 0xffu)) * scale(2 * e)),
                          static_cast<__bf16>(static_cast<float>(static_cast<int8_t>((two >> 8) & 0xffu)) *
                                              scale(2 * e + 1))};
        o[e] = __builtin_bit_cast(uint32_t, b);
      }
      uint4* p = reinterpret_cast<uint4*>(out + dst + 16 * c);
      p[0] = make_uint4(o[0], o[1], o[2], o[3]);
      p[1] = make_uint4(o[4], o[5], o[6], o[7]);
    };
    put(kq, [&](int e) { return ks[e]; }, out_k);
    put(vq, [&](int) { return vs; }, out_v);
  }
}

template <bool HIST, bool REPS>
void launch_store(int fmt, int num_layers, const StoreArgs& a, hipStream_t s) {
  const dim3 grid((a.T + kBlock - 1) / kBlock, a.hkv, num_layers);
  if (!HIST || fmt == NKV_KV_BF16)
    hipLaunchKernelGGL((store_block_kernel<NKV_KV_BF16, HIST, REPS>), grid, dim3(kWave), 0, s, a);
  else if (fmt == NKV_KV_INT8_CHANNEL)
    hipLaunchKernelGGL((store_block_kernel<NKV_KV_INT8_CHANNEL, HIST, REPS>), grid, dim3(kWave), 0, s, a);
  else
    hipLaunchKernelGGL((store_block_kernel<NKV_KV_INT8_TOKEN, HIST, REPS>), grid, dim3(kWave), 0, s, a);
}

// ---------------------------------------------------------------------------
// Recent window on the logical buffer.  Carry moves logical [X, X + carry) ->
// [0, carry) with X = old_len - carry >= 0: with X = 0 nothing moves, and the
// new tokens are spread over workgroups of 64 (one per KV head, layer and 64
// tokens).  With X > 0 one workgroup per KV head and layer moves the slots in
// ascending 64-token chunks with a barrier between each chunk's reads and
// writes (a chunk's writes land below every later chunk's sources, so the
// forward copy never reads a clobbered slot), then stores the new tokens.  The
// runtimes move their ring start and always ask for X = 0; X > 0 is for
// callers of nkv_recent_update that keep theirs.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kStoreThreads) void recent_update_kernel(
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, int64_t kv_ls, int src_lo,
    int n_src, int ring_start, int old_len, int carry, int hkv, int R,
    uint16_t* __restrict__ rk, uint16_t* __restrict__ rv, int64_t rec_ls) {
  const int h = blockIdx.x;
  const int layer = blockIdx.y;
  const int tl = threadIdx.x >> 4;   // token of a group of 16
  const int c = threadIdx.x & 15;    // 16-byte chunk of the row
  uint4* rkl = reinterpret_cast<uint4*>(rk + rec_ls * layer + static_cast<int64_t>(h) * R * kHeadDim);
  uint4* rvl = reinterpret_cast<uint4*>(rv + rec_ls * layer + static_cast<int64_t>(h) * R * kHeadDim);
  const int X = old_len - carry;
  if (X > 0) {
    for (int base = 0; base < carry; base += kBlock) {
      auto slot = [&](int j, int shift) { return (ring_start + shift + min(base + 16 * j + tl, carry - 1)) % R * 16 + c; };
      const uint4 a0 = rkl[slot(0, X)], a1 = rkl[slot(1, X)], a2 = rkl[slot(2, X)], a3 = rkl[slot(3, X)];
      const uint4 b0 = rvl[slot(0, X)], b1 = rvl[slot(1, X)], b2 = rvl[slot(2, X)], b3 = rvl[slot(3, X)];
      __syncthreads();
      auto put = [&](int j, const uint4& a, const uint4& b) {
        if (base + 16 * j + tl < carry) {
          rkl[slot(j, 0)] = a;
          rvl[slot(j, 0)] = b;
        }
      };
      put(0, a0, b0);
      put(1, a1, b1);
      put(2, a2, b2);
      put(3, a3, b3);
      __syncthreads();
    }
  }
  for (int i = blockIdx.z * kBlock + tl; i < n_src; i += kStoreThreads / 16) {
    if (X == 0 && i >= (static_cast<int>(blockIdx.z) + 1) * kBlock) break;   // the next workgroup's tokens
    const int dst = (ring_start + carry + i) % R;
    const int64_t o = kv_ls * layer + (static_cast<int64_t>(src_lo + i) * hkv + h) * kHeadDim;
    rkl[dst * 16 + c] = reinterpret_cast<const uint4*>(k + o)[c];
    rvl[dst * 16 + c] = reinterpret_cast<const uint4*>(v + o)[c];
  }
}

// ---------------------------------------------------------------------------
// Query summaries: bf16 RNE of the fp64 mean (prefill_query_summaries).
// The fp64 sum of bf16 values is exact at these lengths; the quotient is
// rounded to fp32 with round-to-odd and then to bf16 with RNE, which equals a
// single rounding of the fp64 quotient to bf16.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint16_t f64_to_bf16(double x) {
  float f = __double2float_rz(x);
  if (static_cast<double>(f) != x && isfinite(f)) f = __uint_as_float(__float_as_uint(f) | 1u);
  return f32_to_bf16(f);
}

__global__ __launch_bounds__(kStoreThreads) void query_mean_kernel(
    const uint16_t* __restrict__ q, int64_t q_ls, int T, int nelem, int nseg,
    uint16_t* __restrict__ out, int64_t out_ls) {
  const int e = blockIdx.x * kStoreThreads + threadIdx.x;
  const int s = blockIdx.y;
  const int layer = blockIdx.z;
  if (e >= nelem) return;
  const int base = T / nseg, extra = T % nseg;
  const int lo = s * base + min(s, extra);
  const int hi = lo + base + (s < extra ? 1 : 0);
  const uint16_t* ql = q + q_ls * layer;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  int t = lo;
  for (; t + 3 < hi; t += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[u] += static_cast<double>(bf16_to_f32(ql[static_cast<int64_t>(t + u) * nelem + e]));
  }
  for (; t < hi; ++t) acc[0] += static_cast<double>(bf16_to_f32(ql[static_cast<int64_t>(t) * nelem + e]));
  const double sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  out[out_ls * layer + static_cast<int64_t>(s) * nelem + e] = f64_to_bf16(sum / static_cast<double>(hi - lo));
}

// The same means with 16-byte loads: a workgroup of NT threads owns CL chunks
// of 8 elements and splits the segment's tokens over NT / CL thread groups,
// each with 8 rows in flight; the groups' fp64 partial sums meet in registers
// and LDS.  The sums are exact in fp64 (bf16 values of any realistic exponent
// spread), so the result does not depend on the order and equals
// query_mean_kernel's.
// Bound by reading the queries once.  <256, 16> reads 256-byte row pieces:
// 36 layers x 4096 tokens x 32 heads 1.2 GB in 231-250 us (4.8-5.2 TB/s).
// One layer gives only 32 such workgroups, each streaming 1 MiB: <1024, 8>
// puts twice the workgroups with four times the loads in flight each on it
// (4096 x 32 heads, one layer, cold: 30.0 -> 18.2 us; 64- and 32-byte pieces
// 18.0 and 25.1 us, but 24.8 and 50.2 against 19.7 us for two layers).
constexpr int kQmUnroll = 8;
template <int NT, int CL>
__global__ __launch_bounds__(NT) void query_mean8_kernel(
    const uint16_t* __restrict__ q, int64_t q_ls, int T, int nelem, int nseg,
    uint16_t* __restrict__ out, int64_t out_ls) {
  constexpr int kGroups = NT / CL;
  constexpr int kWaves = NT / kWave;
  __shared__ double s_part[kWaves][CL * 8];
  const int cl = threadIdx.x % CL;
  const int grp = threadIdx.x / CL;
  const int nc = nelem >> 3;
  const int c = blockIdx.x * CL + cl;
  const int s = blockIdx.y;
  const int layer = blockIdx.z;
  const int base = T / nseg, extra = T % nseg;
  const int lo = s * base + min(s, extra);
  const int hi = lo + base + (s < extra ? 1 : 0);
  double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  auto add = [&](const uint4& v) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[2 * i] += static_cast<double>(bf16_lo(w[i]));
      acc[2 * i + 1] += static_cast<double>(bf16_hi(w[i]));
    }
  };
  if (c < nc) {
    const uint4* ql = reinterpret_cast<const uint4*>(q + q_ls * layer);
    int t = lo + grp;
    for (; t + (kQmUnroll - 1) * kGroups < hi; t += kQmUnroll * kGroups) {
      uint4 v[kQmUnroll];
#pragma unroll
      for (int u = 0; u < kQmUnroll; ++u) v[u] = ql[static_cast<int64_t>(t + u * kGroups) * nc + c];
#pragma unroll
      for (int u = 0; u < kQmUnroll; ++u) add(v[u]);
    }
    for (; t < hi; t += kGroups) add(ql[static_cast<int64_t>(t) * nc + c]);
  }
  // the wavefront's groups, then the workgroup's wavefronts
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int o = CL; o < kWave; o <<= 1) acc[e] += __shfl_xor(acc[e], o);
  if ((threadIdx.x & (kWave - 1)) < CL)
#pragma unroll
    for (int e = 0; e < 8; ++e) s_part[threadIdx.x / kWave][cl * 8 + e] = acc[e];
  __syncthreads();
  if (threadIdx.x < CL * 8) {
    const int c2 = blockIdx.x * CL + threadIdx.x / 8;
    if (c2 < nc) {
      double sum = 0.0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) sum += s_part[w][threadIdx.x];
      out[out_ls * layer + static_cast<int64_t>(s) * nelem + c2 * 8 + threadIdx.x % 8] =
          f64_to_bf16(sum / static_cast<double>(hi - lo));
    }
  }
}

}  // namespace
}  // namespace nkv

using namespace nkv;

namespace {

// The history / sink part of a chunk's arguments (checked), with the int8 K
// scale computed on the way if asked for.
int fill_store_args(const char* who, const nkv_store* st, int layer0, int num_layers, const uint16_t* k,
                    const uint16_t* v, int64_t kv_layer_stride, int T, int start_block, StoreArgs* out) {
  const int rc = check_store(st, layer0, num_layers);
  if (rc != NKV_OK) return rc;
  NKV_CHECK_ARG(T >= 1, "%s: T must be >= 1 (got %d)", who, T);
  const int nblk = (T + kBlock - 1) / kBlock;
  NKV_CHECK_ARG(start_block >= 0 && start_block + nblk <= st->cap_blocks, "%s: blocks [%d, %d) exceed cap_blocks %d",
                who, start_block, start_block + nblk, st->cap_blocks);
  const int hkv = st->num_kv_heads;
  StoreArgs& a = *out;
  a = StoreArgs{};
  a.k = k;
  a.v = v;
  a.kv_ls = kv_layer_stride;
  a.T = T;
  a.start_block = start_block;
  a.hkv = hkv;
  a.cap = st->cap_blocks;
  a.r = st->r;
  a.hist_ls = static_cast<int64_t>(hkv) * st->cap_blocks * kBlock * kHeadDim;
  const int64_t elem = st->kv_format == NKV_KV_BF16 ? 2 : 1;
  a.hist_k = static_cast<char*>(st->hist_k) + layer0 * a.hist_ls * elem;
  a.hist_v = static_cast<char*>(st->hist_v) + layer0 * a.hist_ls * elem;
  const int64_t ts_ls = static_cast<int64_t>(hkv) * st->cap_blocks * kBlock;
  a.k_scale = st->k_scale ? st->k_scale + static_cast<int64_t>(layer0) * hkv * kHeadDim : nullptr;
  a.v_scale = st->v_scale ? st->v_scale + static_cast<int64_t>(layer0) * hkv * st->cap_blocks : nullptr;
  a.k_tscale = st->k_tscale ? st->k_tscale + layer0 * ts_ls : nullptr;
  a.v_tscale = st->v_tscale ? st->v_tscale + layer0 * ts_ls : nullptr;
  a.S = st->sink_tokens;
  a.sink_ls = static_cast<int64_t>(hkv) * st->sink_tokens * kHeadDim;
  a.sink_k = st->sink_k ? static_cast<uint16_t*>(st->sink_k) + layer0 * a.sink_ls : nullptr;
  a.sink_v = st->sink_v ? static_cast<uint16_t*>(st->sink_v) + layer0 * a.sink_ls : nullptr;
  a.R = st->recent_tokens;
  a.rec_ls = static_cast<int64_t>(hkv) * a.R * kHeadDim;
  a.rec_k = static_cast<uint16_t*>(st->recent_k) + layer0 * a.rec_ls;
  a.rec_v = static_cast<uint16_t*>(st->recent_v) + layer0 * a.rec_ls;
  a.reps_ls = static_cast<int64_t>(hkv) * st->cap_blocks * st->r * kHeadDim;
  a.reps = static_cast<uint16_t*>(st->reps) + layer0 * a.reps_ls;
  return NKV_OK;
}

// A long chunk of few (layer, KV head) pairs gives a few workgroups that each
// stream all of its tokens: from 8192 tokens on they are split over up to 512
// workgroups, for two more launches (us, whole / split: one layer, 8 heads,
// 4096 tokens 11.5 / 11.4, 8192 19.2 / 12.6, 65536 203 / 42; one head, 4096
// tokens 8.6 / 7.8, 8192 13.8 / 9.4, 65536 83 / 11; four layers of 8 heads,
// 4096 tokens 17.2 / 17.4, 16384 57 / 45).
constexpr int kScaleSplitRows = 8192;
constexpr int kScalePartRows = 2048;
constexpr int kScaleWorkgroups = 512;

int launch_k_scale(const nkv_store* st, int layer0, int num_layers, const uint16_t* k, int64_t kv_layer_stride, int T,
                   hipStream_t s) {
  const int hkv = st->num_kv_heads;
  float* dst = st->k_scale + static_cast<int64_t>(layer0) * hkv * kHeadDim;
  const int64_t n = static_cast<int64_t>(num_layers) * hkv * kHeadDim;
  const int64_t wgs = n / kScaleDims;
  const int parts = static_cast<int>(std::min<int64_t>((T + kScalePartRows - 1) / kScalePartRows,
                                                       std::max<int64_t>(1, kScaleWorkgroups / wgs)));
  if (T < kScaleSplitRows || parts < 2) {
    hipLaunchKernelGGL(k_scale_kernel<false>, dim3(hkv * kHeadDim / kScaleDims, num_layers), dim3(kScaleThreads), 0, s,
                       k, kv_layer_stride, T, hkv, dst);
  } else {
    const dim3 all(static_cast<unsigned>((n + kStoreThreads - 1) / kStoreThreads));
    hipLaunchKernelGGL(k_scale_clear_kernel, all, dim3(kStoreThreads), 0, s, dst, n);
    hipLaunchKernelGGL(k_scale_kernel<true>, dim3(hkv * kHeadDim / kScaleDims, num_layers, parts), dim3(kScaleThreads),
                       0, s, k, kv_layer_stride, T, hkv, dst);
    hipLaunchKernelGGL(k_scale_finish_kernel, all, dim3(kStoreThreads), 0, s, dst, n);
  }
  return launch_status("nkv_store_chunk/k_scale");
}

}  // namespace

extern "C" int nkv_store_chunk(const nkv_store* st, int layer0, int num_layers, const uint16_t* k,
                               const uint16_t* v, int64_t kv_layer_stride, int T, int start_block,
                               int compute_k_scale, int write_sink, void* stream) {
  StoreArgs a;
  int rc = fill_store_args("nkv_store_chunk", st, layer0, num_layers, k, v, kv_layer_stride, T, start_block, &a);
  if (rc != NKV_OK) return rc;
  NKV_CHECK_ARG(k != nullptr && v != nullptr, "nkv_store_chunk: k and v must be non-NULL");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (st->kv_format == NKV_KV_INT8_CHANNEL && compute_k_scale) {
    rc = launch_k_scale(st, layer0, num_layers, k, kv_layer_stride, T, s);
    if (rc != NKV_OK) return rc;
  }
  a.sink_n = write_sink ? std::min(T, st->sink_tokens) : 0;
  launch_store<true, false>(st->kv_format, num_layers, a, s);
  return launch_status("nkv_store_chunk");
}

extern "C" int nkv_build_reps(const nkv_store* st, int layer0, int num_layers, const uint16_t* k,
                              int64_t kv_layer_stride, int T, int start_block, void* stream) {
  StoreArgs a;
  const int rc = fill_store_args("nkv_build_reps", st, layer0, num_layers, k, nullptr, kv_layer_stride, T, start_block,
                                 &a);
  if (rc != NKV_OK) return rc;
  NKV_CHECK_ARG(k != nullptr, "nkv_build_reps: k must be non-NULL");
  launch_store<false, true>(st->kv_format, num_layers, a, reinterpret_cast<hipStream_t>(stream));
  return launch_status("nkv_build_reps");
}

extern "C" int nkv_store_append(const nkv_store* st, int layer0, int num_layers, const uint16_t* k,
                                const uint16_t* v, int64_t kv_layer_stride, int T, int start_block,
                                int compute_k_scale, int write_sink, int rec_src_lo, int rec_n, int rec_slot,
                                void* stream) {
  StoreArgs a;
  int rc = fill_store_args("nkv_store_append", st, layer0, num_layers, k, v, kv_layer_stride, T, start_block, &a);
  if (rc != NKV_OK) return rc;
  NKV_CHECK_ARG(k != nullptr && v != nullptr, "nkv_store_append: k and v must be non-NULL");
  NKV_CHECK_ARG(rec_src_lo >= 0 && rec_n >= 0 && rec_n <= T && rec_src_lo <= T - rec_n && rec_n <= st->recent_tokens,
                "nkv_store_append: recent tokens [%d, %d) outside the chunk or more than the window (T=%d, R=%d)",
                rec_src_lo, rec_src_lo + rec_n, T, st->recent_tokens);
  NKV_CHECK_ARG(rec_slot >= 0 && rec_slot < st->recent_tokens, "nkv_store_append: rec_slot %d outside [0, %d)", rec_slot,
                st->recent_tokens);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (st->kv_format == NKV_KV_INT8_CHANNEL && compute_k_scale) {
    rc = launch_k_scale(st, layer0, num_layers, k, kv_layer_stride, T, s);
    if (rc != NKV_OK) return rc;
  }
  a.sink_n = write_sink ? std::min(T, st->sink_tokens) : 0;
  a.rec_lo = rec_src_lo;
  a.rec_n = rec_n;
  a.rec_slot = rec_slot;
  launch_store<true, true>(st->kv_format, num_layers, a, s);
  return launch_status("nkv_store_append");
}

extern "C" int nkv_history_bf16(const nkv_store* st, int layer0, int num_layers, const int32_t* ids,
                                int64_t ids_layer_stride, int n_hist, uint16_t* out_k, uint16_t* out_v,
                                int32_t* out_ids, void* stream) {
  const int rc = check_store(st, layer0, num_layers);
  if (rc != NKV_OK) return rc;
  NKV_CHECK_ARG(ids != nullptr && out_k != nullptr && out_v != nullptr && out_ids != nullptr,
                "nkv_history_bf16: ids and the outputs must be non-NULL");
  NKV_CHECK_ARG(n_hist >= 1 && n_hist <= 4096, "nkv_history_bf16: n_hist must be in [1, 4096] (got %d)", n_hist);
  NKV_CHECK_ARG(num_layers == 1 || ids_layer_stride >= n_hist, "nkv_history_bf16: ids_layer_stride too small");
  NKV_CHECK_SUPPORTED(st->kv_format != NKV_KV_BF16, "nkv_history_bf16: the history is bf16 already");
  const int hkv = st->num_kv_heads;
  const int64_t hist_ls = static_cast<int64_t>(hkv) * st->cap_blocks * kBlock * kHeadDim;
  const int64_t ts_ls = static_cast<int64_t>(hkv) * st->cap_blocks * kBlock;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(n_hist, hkv, num_layers), dim3(kStoreThreads), 0,
                       reinterpret_cast<hipStream_t>(stream), static_cast<const int8_t*>(st->hist_k) + layer0 * hist_ls,
                       static_cast<const int8_t*>(st->hist_v) + layer0 * hist_ls, hist_ls,
                       st->k_scale ? st->k_scale + static_cast<int64_t>(layer0) * hkv * kHeadDim : nullptr,
                       st->v_scale ? st->v_scale + static_cast<int64_t>(layer0) * hkv * st->cap_blocks : nullptr,
                       st->k_tscale ? st->k_tscale + layer0 * ts_ls : nullptr,
                       st->v_tscale ? st->v_tscale + layer0 * ts_ls : nullptr, hkv, st->cap_blocks, ids,
                       ids_layer_stride, n_hist, out_k, out_v, out_ids);
  };
  if (st->kv_format == NKV_KV_INT8_CHANNEL)
    go(history_bf16_kernel<NKV_KV_INT8_CHANNEL>);
  else
    go(history_bf16_kernel<NKV_KV_INT8_TOKEN>);
  return launch_status("nkv_history_bf16");
}

extern "C" int nkv_recent_update(const nkv_store* st, int layer0, int num_layers, const uint16_t* k,
                                 const uint16_t* v, int64_t kv_layer_stride, int src_lo, int n_src,
                                 int ring_start, int old_len, int carry, void* stream) {
  int rc = check_store(st, layer0, num_layers);
  if (rc != NKV_OK) return rc;
  const int R = st->recent_tokens;
  NKV_CHECK_ARG(ring_start >= 0 && ring_start < R, "nkv_recent_update: ring_start %d outside [0, %d)", ring_start, R);
  NKV_CHECK_ARG(carry >= 0 && old_len >= carry && old_len <= R,
                "nkv_recent_update: need 0 <= carry <= old_len <= R (carry=%d, old_len=%d)", carry, old_len);
  NKV_CHECK_ARG(n_src >= 0 && src_lo >= 0 && carry + n_src <= R,
                "nkv_recent_update: carry + n_src must be <= R (carry=%d, n_src=%d)", carry, n_src);
  NKV_CHECK_ARG(n_src == 0 || (k != nullptr && v != nullptr), "nkv_recent_update: k/v are NULL");
  const int64_t rec_ls = static_cast<int64_t>(st->num_kv_heads) * R * kHeadDim;
  const bool moves = old_len > carry && carry > 0;
  if (!moves && n_src == 0) return NKV_OK;
  const int nz = moves ? 1 : (n_src + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(recent_update_kernel, dim3(st->num_kv_heads, num_layers, nz), dim3(kStoreThreads), 0,
                     reinterpret_cast<hipStream_t>(stream), k, v, kv_layer_stride, src_lo, n_src, ring_start,
                     moves ? old_len : carry, carry, st->num_kv_heads, R,
                     static_cast<uint16_t*>(st->recent_k) + layer0 * rec_ls,
                     static_cast<uint16_t*>(st->recent_v) + layer0 * rec_ls, rec_ls);
  return launch_status("nkv_recent_update");
}

extern "C" int nkv_query_summaries(const uint16_t* q, int64_t q_layer_stride, int num_layers, int T,
                                   int num_heads, int head_dim, int nsegments, uint16_t* out,
                                   int64_t out_layer_stride, void* stream) {
  NKV_CHECK_ARG(q != nullptr && out != nullptr, "nkv_query_summaries: q and out must be non-NULL");
  NKV_CHECK_ARG(T >= 1 && nsegments >= 1 && num_layers >= 1 && num_heads >= 1,
                "nkv_query_summaries: T, nsegments, num_layers and num_heads must be >= 1");
  NKV_CHECK_SUPPORTED(head_dim == kHeadDim, "nkv_query_summaries: head_dim must be %d", kHeadDim);
  const int nseg = nsegments < T ? nsegments : T;
  const int nelem = num_heads * head_dim;
  if ((reinterpret_cast<uintptr_t>(q) & 15u) == 0 && q_layer_stride % 8 == 0) {
    const int nc = nelem / 8;
    auto go = [&](auto kern, int threads, int cl) {
      hipLaunchKernelGGL(kern, dim3((nc + cl - 1) / cl, nseg, num_layers), dim3(threads), 0,
                         reinterpret_cast<hipStream_t>(stream), q, q_layer_stride, T, nelem, nseg, out, out_layer_stride);
    };
    // fewer workgroups than CUs, with many rows each: narrower row pieces and
    // more threads a workgroup (us, <256, 16> / <1024, 8>, 32 heads: 128
    // workgroups, 4 layers x 4096 tokens 33.0 / 27.5; 256, 8 layers 45.2 /
    // 47.4; one layer of 2048 tokens 16.4 / 10.4, of 700 7.6 / 7.6)
    const int64_t wgs = static_cast<int64_t>((nc + 15) / 16) * nseg * num_layers;
    if (wgs < 256 && T / nseg >= 512)
      go(query_mean8_kernel<1024, 8>, 1024, 8);
    else
      go(query_mean8_kernel<kStoreThreads, 16>, kStoreThreads, 16);
  } else {
    hipLaunchKernelGGL(query_mean_kernel, dim3((nelem + kStoreThreads - 1) / kStoreThreads, nseg, num_layers),
                       dim3(kStoreThreads), 0, reinterpret_cast<hipStream_t>(stream), q, q_layer_stride, T,
                       nelem, nseg, out, out_layer_stride);
  }
  return launch_status("nkv_query_summaries");
}
