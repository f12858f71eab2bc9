// Top-K of one row of score keys by one wavefront, used by the selection
// kernels (nkv_select.hip) and by the attention of small decode steps
// (nkv_attend.hip), which selects for itself.
#pragma once

#include "nkv_common.h"

namespace nkv {
namespace select_detail {

constexpr uint32_t kNegInfKey = 0x007fffffu;  // score_key(-inf)

// 64-bit sort/selection entry: key in the high word, ~id in the low word, so
// that a larger entry means a larger score, and on equal scores a lower id.
__device__ __forceinline__ unsigned long long sel_entry(uint32_t key, int id) {
  return (static_cast<unsigned long long>(key) << 32) |
         static_cast<unsigned long long>(0xffffffffu - static_cast<uint32_t>(id));
}

// Same selection as topk_kernel (identical ids, values and order) for one row
// of at most 64 J blocks, computed by ONE wavefront with no workgroup barrier
// (pmask: 2 J words of LDS, sel: LDS for max(k, 64) rounded up to a power of
// two entries).  Returns the number of ids written: k_req, or the number of
// selectable blocks when that is smaller (at least 1).
// Lane l holds the keys of blocks 64 j + l (j < J) in registers.  The k-th
// largest key T is found by a bitwise search of at most 32 steps: T is the
// largest value with count(key >= T) >= k, built from the high bit down, each
// count being J ballots.  Collection is the same ascending-id ballot pass as
// topk_kernel; up to 64 selected entries are then placed by their rank among
// the selection, larger k sorted by a bitonic network over LDS.
//
// STEP (the decode step's selection): the scorer left the protected blocks'
// keys at 0 (every scored key is >= score_key(-inf) > 0), and the step's
// attention launch zeroes the keys afterwards, so the row needs neither the
// protected list nor the zeroing stores; key 0 is read as score_key(-inf),
// exactly the protected mask of the general form.
template <int J, bool STEP>
__device__ __forceinline__ int select_row_wave(
    uint32_t* __restrict__ sk, int nblocks, const int32_t* __restrict__ prot, int nprot,
    int k_req, int order, int32_t* __restrict__ ids, float* __restrict__ vals,
    float* __restrict__ scores, uint32_t* pmask, unsigned long long* sel, int lane) {
  const int nwords = (nblocks + 31) >> 5;

  // The key reads go out first (they do not depend on the protected set), so
  // their latency overlaps the protected-id reads.  Keys past nblocks are 0,
  // below every key score_key() produces.  Every read is issued (past nblocks
  // it re-reads the last key), so one wait covers them all.
  uint32_t key[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int i = kWave * j + lane;
    key[j] = sk[i < nblocks ? i : nblocks - 1];
  }

  int avail = 0;
  if constexpr (STEP) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int i = kWave * j + lane;
      const bool valid = i < nblocks;
      avail += __popcll(__ballot(valid && key[j] != 0u));
      key[j] = !valid ? 0u : (key[j] == 0u ? kNegInfKey : key[j]);
    }
  } else {
    for (int w = lane; w < nwords; w += kWave) pmask[w] = 0u;
    wave_lds_sync();
    for (int i = lane; i < nprot; i += kWave) {
      const int p = prot[i];
      if (p >= 0 && p < nblocks) atomicOr(&pmask[p >> 5], 1u << (p & 31));
    }
    wave_lds_sync();

    // blocks in range and not protected, counted with ballots
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int i = kWave * j + lane;
      const bool valid = i < nblocks;
      const bool prot_i = valid && ((pmask[i >> 5] >> (i & 31)) & 1u);
      if (valid) {
        sk[i] = 0u;  // leave the key buffer zeroed for the next scoring pass
        if (scores) scores[i] = key_score(key[j]);
        if (prot_i) key[j] = kNegInfKey;
      } else {
        key[j] = 0u;
      }
      avail += __popcll(__ballot(valid && !prot_i));
    }
  }
  const int k = min(k_req, max(1, avail));

  // ---- fast path: rank a short candidate list -----------------------------
  // L0 = the k-th largest of the 64 lane maxima (one ballot per search step)
  // bounds the k-th largest key from below: k lanes hold a key >= L0.  Every
  // valid key >= L0 is a candidate; when there are at most 64 of them they
  // go to LDS in ascending block order and each lane ranks one against all
  // (the entries are distinct: the id is part of each), which places the
  // selection directly.  Otherwise (ties, adversarial spreads) the bitwise
  // search below runs over all keys.  Same selection either way.
  if (k <= kWave) {
    uint32_t lmax = key[0];
#pragma unroll
    for (int j = 1; j < J; ++j) lmax = max(lmax, key[j]);   // keys past nblocks are 0
    uint32_t L0 = 0u;
    for (uint32_t m = 0x80000000u; m != 0u; m >>= 1) {
      const uint32_t cand = L0 | m;
      const int cnt = __popcll(__ballot(lmax >= cand));
      if (cnt >= k) L0 = cand;
      if (cnt == k) break;
    }
    unsigned long long bc[J];
#pragma unroll
    for (int j = 0; j < J; ++j) bc[j] = __ballot(kWave * j + lane < nblocks && key[j] >= L0);
    int C = 0;
#pragma unroll
    for (int j = 0; j < J; ++j) C += __popcll(bc[j]);
    if (C <= kWave) {
      const unsigned long long lt = (1ull << lane) - 1ull;
      int base = 0;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        if ((bc[j] >> lane) & 1ull) sel[base + __popcll(bc[j] & lt)] = sel_entry(key[j], kWave * j + lane);
        base += __popcll(bc[j]);
      }
      wave_lds_sync();
      // sel holds >= 64 entries, so the pair read at j = C - 1 stays inside it
      const unsigned long long e = sel[lane < C ? lane : 0];
      int rank = 0;
      const int cp = (C + 1) & ~1;
#pragma unroll 8
      for (int j = 0; j < cp; j += 2) {
        const unsigned long long a = sel[j], b = sel[j + 1];
        rank += (a > e) + ((j + 1 < C) & (b > e));
      }
      const bool chosen = lane < C && rank < k;
      int pos = rank;
      if (order != NKV_ORDER_SCORE_DESC) pos = __popcll(__ballot(chosen) & lt);   // ascending id
      if (chosen) {
        ids[pos] = static_cast<int32_t>(0xffffffffu - static_cast<uint32_t>(e & 0xffffffffull));
        if (vals) vals[pos] = key_score(static_cast<uint32_t>(e >> 32));
      }
      return k;
    }
  }

  // ---- k-th largest key: largest T with count(key >= T) >= k ------------
  // Once count(key >= T) == k the k keys >= T are the selection itself (every
  // key equal to the k-th largest is among them), so the search stops there:
  // the collection below then takes exactly those keys, as it would with the
  // fully resolved T.
  // T and the candidate stay scalar (one vector-to-scalar hand-off per
  // ballot, none back), and the J ballot counts are summed as a tree.
  uint32_t T = 0u;
  for (uint32_t m = 0x80000000u; m != 0u; m >>= 1) {
    const uint32_t cand = T | m;
    // all J compares issue before the first count reads one, so only the
    // first count waits for a compare result
    unsigned long long b[J];
#pragma unroll
    for (int j = 0; j < J; ++j) b[j] = __ballot(key[j] >= cand);
    __builtin_amdgcn_sched_barrier(0);
    int c[J];
#pragma unroll
    for (int j = 0; j < J; ++j) c[j] = __popcll(b[j]);
#pragma unroll
    for (int w = 1; w < J; w <<= 1)
#pragma unroll
      for (int j = 0; j + w < J; j += 2 * w) c[j] += c[j + w];
    const int cnt = c[0];
    if (cnt >= k) T = cand;
    if (cnt == k) break;
  }
  int above = 0;
#pragma unroll
  for (int j = 0; j < J; ++j) above += __popcll(__ballot(key[j] > T));

  // ---- collect in ascending block order ----------------------------------
  const unsigned long long lt = (1ull << lane) - 1ull;
  uint32_t base = 0u;
  uint32_t need = static_cast<uint32_t>(k - above);
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int i = kWave * j + lane;
    const bool gt = key[j] > T;
    const bool eq = key[j] == T && i < nblocks;
    const unsigned long long meq = __ballot(eq);
    const uint32_t rank = __popcll(meq & lt);
    const bool take = gt || (eq && rank < need);
    const unsigned long long mt = __ballot(take);
    if (take) sel[base + __popcll(mt & lt)] = sel_entry(key[j], i);
    base += __popcll(mt);
    const uint32_t neq = __popcll(meq);
    need -= (neq < need ? neq : need);
  }
  wave_lds_sync();

  if (order == NKV_ORDER_SCORE_DESC && k > 1 && k <= kWave) {
    // Rank sort: the entries are distinct (the id is part of each), so the
    // position of entry e in the descending order is the number of entries
    // larger than e.  Lane l < k ranks sel[l] against all k entries, read as
    // LDS broadcasts two at a time (sel holds at least 64 entries, so the
    // pair read at j = k - 1 stays inside it; its second entry is ignored).
    const unsigned long long e = sel[lane < k ? lane : 0];
    int rank = 0;
    const int kp = (k + 1) & ~1;
#pragma unroll 8
    for (int j = 0; j < kp; j += 2) {
      const unsigned long long a = sel[j], b = sel[j + 1];
      rank += (a > e) + ((j + 1 < k) & (b > e));
    }
    if (lane < k) {
      ids[rank] = static_cast<int32_t>(0xffffffffu - static_cast<uint32_t>(e & 0xffffffffull));
      if (vals) vals[rank] = key_score(static_cast<uint32_t>(e >> 32));
    }
    return k;
  }
  if (order == NKV_ORDER_SCORE_DESC && k > 1) {
    int n2 = 1;
    while (n2 < k) n2 <<= 1;
    for (int i = k + lane; i < n2; i += kWave) sel[i] = 0ull;
    wave_lds_sync();
    for (int size = 2; size <= n2; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        for (int i = lane; i < (n2 >> 1); i += kWave) {
          const int lo = 2 * i - (i & (stride - 1));
          const int hi = lo + stride;
          const bool desc = (lo & size) == 0;
          const unsigned long long a = sel[lo], b = sel[hi];
          if (desc ? (a < b) : (a > b)) {
            sel[lo] = b;
            sel[hi] = a;
          }
        }
        wave_lds_sync();
      }
    }
  }
  for (int i = lane; i < k; i += kWave) {
    const unsigned long long e = sel[i];
    ids[i] = static_cast<int32_t>(0xffffffffu - static_cast<uint32_t>(e & 0xffffffffull));
    if (vals) vals[i] = key_score(static_cast<uint32_t>(e >> 32));
  }
  return k;
}

}  // namespace select_detail
}  // namespace nkv
