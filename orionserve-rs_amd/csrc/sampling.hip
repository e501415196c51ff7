// Device-side DefaultSampler (crates/orion-runtime/src/sampling.rs:266-293):
// repetition penalty, then greedy argmax or temperature -> top-k -> top-p ->
// softmax -> draw, over rows of logits already in HBM, so only one token per
// row crosses to the host instead of the [rows, vocab] f32 logits.
//
// One 1024-thread workgroup per row.  The row is walked in tiles of
// 1024 x 8 elements: thread t holds elements [8t, 8t + 8) of each tile (two
// 16-byte accesses, so a wave moves 2 KiB contiguously).  Rows of up to 32768
// entries are kept in LDS.  What bounds it is the arithmetic and the barriers of
// the passes, not the 8 bytes an entry moves: 32 rows of 32000 with mixed
// settings took 237 us with 8-bit radix digits (the exponents of a row's logits
// fill a handful of 256 buckets, so most of a wave's LDS atomics met on one
// address), serial suffix sums and every probability recomputed in every pass.
// The same results take 82 us with 11-bit digits, prefix sums over the
// buckets, and one exponential and one division per entry and softmax.  (The
// row in registers, 32 entries a thread, took 81 us: 14,000 unrolled
// instructions and spills.)
// Order-sensitive quantities (the draw's cumulative sum, the tie ranks of
// top-p) are formed in index order inside a thread's 8 elements and by a
// fixed-tree prefix across threads and tiles: deterministic, and equal to the
// reference's sequential f32 sums up to rounding.
//
// The uniform `r` of each draw comes from the caller (the reference draws it
// from a per-request ChaCha8Rng, sampling.rs:209-210); everything after it is
// computed here.
#include "common.hpp"
#include "kernels.hpp"


namespace orion {

namespace {

constexpr int kT = 1024;  // threads per row
constexpr int kWavesPerRow = kT / 64;
constexpr float kMasked = -1.0e30f;  // sampling.rs:36

// Order-preserving uint key of a float (larger float -> larger key); NaN maps
// below every number, so it never wins a selection.
__device__ inline uint32_t fkey(float f) {
  if (f != f) return 0u;
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ inline float key_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

struct Scratch {
  float f[kWavesPerRow];
  uint32_t u[kWavesPerRow];
  int64_t i[kWavesPerRow];
};

// Block reductions in a fixed order (lanes by butterfly, then waves 0..15).
__device__ float block_sum(float v, Scratch& s) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.f[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
  for (int w = 0; w < kWavesPerRow; ++w) t += s.f[w];
  return t;
}
__device__ float block_max(float v, Scratch& s) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.f[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = s.f[0];
  for (int w = 1; w < kWavesPerRow; ++w) t = fmaxf(t, s.f[w]);
  return t;
}
__device__ uint32_t block_count(uint32_t v, Scratch& s) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.u[threadIdx.x >> 6] = v;
  __syncthreads();
  uint32_t t = 0;
  for (int w = 0; w < kWavesPerRow; ++w) t += s.u[w];
  return t;
}
__device__ int64_t block_min_i64(int64_t v, Scratch& s) {
  for (int o = 32; o > 0; o >>= 1) v = min(v, (int64_t)__shfl_xor(v, o));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.i[threadIdx.x >> 6] = v;
  __syncthreads();
  int64_t t = s.i[0];
  for (int w = 1; w < kWavesPerRow; ++w) t = min(t, s.i[w]);
  return t;
}
__device__ int64_t block_max_i64(int64_t v, Scratch& s) {
  for (int o = 32; o > 0; o >>= 1) v = max(v, (int64_t)__shfl_xor(v, o));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s.i[threadIdx.x >> 6] = v;
  __syncthreads();
  int64_t t = s.i[0];
  for (int w = 1; w < kWavesPerRow; ++w) t = max(t, s.i[w]);
  return t;
}

// Exclusive prefix of per-thread values in thread order, by a fixed tree
// (inclusive lane scan by shuffles, then the wave totals in wave order):
// deterministic.  `wave_tot` is a 16-entry shared array of the value type.
template <typename V>
__device__ V block_exclusive_prefix(V v, V* wave_tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  V inc = v;
  for (int o = 1; o < 64; o <<= 1) {
    const V n = __shfl_up(inc, o);
    if (lane >= o) inc += n;
  }
  __syncthreads();
  if (lane == 63) wave_tot[wave] = inc;
  __syncthreads();
  V base = V(0);
  for (int w = 0; w < wave; ++w) base += wave_tot[w];
  return base + inc - v;
}

constexpr int kE = 8;            // contiguous elements per thread per tile
constexpr int kTile = kT * kE;   // elements per tile
constexpr int kLdsRow = 32768;   // rows up to this many entries are held in LDS

// Radix digits of the selects: 11, 11 and 10 bits from the top.
constexpr int kDigits = 3;
constexpr int kBuckets = 2048;
__device__ inline int digit_shift(int d) { return d == 0 ? 21 : d == 1 ? 10 : 0; }
__device__ inline uint32_t digit_mask(int d) { return d == 2 ? 1023u : 2047u; }
__device__ inline uint32_t above_mask(int d) {  // the bits of the digits before d
  return d == 0 ? 0u : d == 1 ? 0xFFE00000u : 0xFFFFFC00u;
}

}  // namespace

// OWN: the row (up to kLdsRow entries) in LDS, where it becomes exponentials
// and probabilities; else it stays in memory, each pass reading it and the
// filters writing it there.
template <bool OWN>
__global__ void __launch_bounds__(kT)
    sample_kernel(float* __restrict__ logits, int64_t vocab64,
                  const SampleParams* __restrict__ params, const int64_t* __restrict__ prev_off,
                  const uint32_t* __restrict__ prev_tok, const float* __restrict__ uniform,
                  int32_t* __restrict__ out) {
#pragma clang fp contract(off)
  __shared__ Scratch s;
  __shared__ float own_row[OWN ? kLdsRow : 1];
  __shared__ uint32_t seen[(OWN ? kLdsRow : kSampleMaxVocab) / 32];
  __shared__ unsigned long long bucket[kBuckets];
  __shared__ unsigned long long wave_u64[kWavesPerRow];
  __shared__ unsigned long long sel_above;
  __shared__ uint32_t sel_key, sel_rank;
  __shared__ int sel_found;
  const int64_t row = blockIdx.x;
  const int vocab = (int)vocab64;
  float* gx = logits + row * vocab64;
  const SampleParams sp = params[row];
  const int tid = threadIdx.x;
  const int ntiles = (vocab + kTile - 1) / kTile;
  auto base = [&](int t) { return t * kTile + tid * kE; };
  auto valid = [&](int t, int e) { return base(t) + e < vocab; };
  // (rows in memory are 4-byte aligned: two 16-byte accesses of that alignment)
  auto load8 = [&](const float* from, int t, float (&v)[kE]) {
    const int b = base(t);
    if (b + kE <= vocab) {
      __builtin_memcpy(v, from + b, kE * sizeof(float));
    } else {
#pragma unroll
      for (int e = 0; e < kE; ++e) v[e] = b + e < vocab ? from[b + e] : 0.f;
    }
  };
  auto store8 = [&](float* to, int t, const float (&v)[kE]) {
    const int b = base(t);
    if (b + kE <= vocab) {
      __builtin_memcpy(to + b, v, kE * sizeof(float));
    } else {
#pragma unroll
      for (int e = 0; e < kE; ++e)
        if (b + e < vocab) to[b + e] = v[e];
    }
  };
  float* row_at = OWN ? own_row : gx;
  // f(tile, its 8 elements) over the row; `update` keeps what f changes, `own`
  // only in LDS
  auto pass = [&](auto f, bool keep) {
    for (int t = 0; t < ntiles; ++t) {
      float v[kE];
      load8(row_at, t, v);
      f(t, v);
      if (keep) store8(row_at, t, v);
    }
  };
  auto tiles = [&](auto f) { pass(f, false); };
  auto update = [&](auto f) { pass(f, true); };
  auto own = [&](auto f) { pass(f, OWN); };
  // (each thread moves, and only ever reads, its own elements)
  auto copy_row = [&](const float* from, float* to) {
    if constexpr (OWN)
      for (int t = 0; t < ntiles; ++t) {
        float v[kE];
        load8(from, t, v);
        store8(to, t, v);
      }
  };
  copy_row(gx, own_row);

  // ---- repetition penalty (sampling.rs:46-60): once per distinct token, from
  // a bitmap of the previous ones (a thread's 8 elements are one byte of it) ----
  const bool greedy = sp.temperature == 0.0f;
  if (sp.repetition_penalty != 1.0f) {
    for (int w = tid; w < (vocab + 31) / 32; w += kT) seen[w] = 0u;
    __syncthreads();
    for (int64_t j = prev_off[row] + tid; j < prev_off[row + 1]; j += kT) {
      const uint32_t t = prev_tok[j];
      if ((int64_t)t < vocab64) atomicOr(&seen[t >> 5], 1u << (t & 31));
    }
    __syncthreads();
    update([&](int t, float (&v)[kE]) {
      const int b = base(t);
      if (b >= vocab) return;
      const uint32_t bits = (seen[b >> 5] >> (b & 31)) & 255u;
      if (!bits) return;
#pragma unroll
      for (int e = 0; e < kE; ++e) {
        if (!(bits >> e & 1u)) continue;
        v[e] = v[e] > 0.0f ? v[e] / sp.repetition_penalty : v[e] * sp.repetition_penalty;
        if (OWN && greedy && valid(t, e)) gx[b + e] = v[e];  // (else written back whole)
      }
    });
  }

  // ---- greedy (SamplingParams::mode, temperature 0): argmax, strict '>' in
  // index order, lowest index on ties, NaN never wins (sampling.rs:196-207) ----
  if (greedy) {
    float best = -INFINITY;
    int64_t bi = INT64_MAX;
    tiles([&](int t, float (&v)[kE]) {
#pragma unroll
      for (int e = 0; e < kE; ++e)
        if (valid(t, e) && v[e] > best) {
          best = v[e];
          bi = base(t) + e;
        }
    });
    const float bmax = block_max(best, s);
    const int64_t win = block_min_i64((best == bmax && bi != INT64_MAX) ? bi : INT64_MAX, s);
    if (tid == 0) out[row] = win == INT64_MAX ? -1 : (int32_t)win;
    return;
  }

  // ---- temperature (sampling.rs:67-75) ----
  if (sp.temperature != 1.0f) {
    const float inv = 1.0f / sp.temperature;
    update([&](int t, float (&v)[kE]) {
#pragma unroll
      for (int e = 0; e < kE; ++e) v[e] = v[e] * inv;
    });
  }

  // One digit of a select over the buckets, largest first: the bucket whose
  // predecessors hold less than `want` and that reaches it, with what they
  // hold.  `none` (thread 0's bucket of the last, the lowest) when no bucket
  // does.  Thread t owns buckets 2047 - 2t and 2046 - 2t.
  auto pick = [&](unsigned long long above0, unsigned long long want, auto found, auto none) {
    const int hi = kBuckets - 1 - 2 * tid, lo = hi - 1;
    const unsigned long long a = bucket[hi], b = bucket[lo];
    const unsigned long long above =
        above0 + block_exclusive_prefix<unsigned long long>(a + b, wave_u64);
    if (above < want && above + a >= want)
      found(hi, above);
    else if (above + a < want && above + a + b >= want)
      found(lo, above + a);
    else if (lo == 0 && above + a + b < want)
      none(above + a);
  };
  auto clear_buckets = [&]() {
    bucket[tid] = 0ull;
    bucket[tid + kT] = 0ull;
  };

  // ---- top-k (sampling.rs:82-99): the k-th largest value by a radix select
  // on order-preserving keys; strictly smaller logits are masked ----
  if (sp.top_k > 0 && sp.top_k < vocab) {
    if (tid == 0) {
      sel_key = 0u;
      sel_rank = (uint32_t)sp.top_k;  // rank among the remaining, 1-based
    }
    for (int d = 0; d < kDigits; ++d) {
      clear_buckets();
      __syncthreads();
      const uint32_t pre = sel_key, rank = sel_rank;
      const uint32_t above = above_mask(d), mask = digit_mask(d);
      const int shift = digit_shift(d);
      tiles([&](int t, float (&v)[kE]) {
#pragma unroll
        for (int e = 0; e < kE; ++e) {
          const uint32_t k = fkey(v[e]);
          if (valid(t, e) && (k & above) == pre)
            atomicAdd(reinterpret_cast<uint32_t*>(&bucket[(k >> shift) & mask]), 1u);
        }
      });
      __syncthreads();
      auto take = [&](int b, unsigned long long higher) {
        sel_key = pre | ((uint32_t)b << shift);
        sel_rank = rank - (uint32_t)higher;
      };
      pick(0ull, rank, take, [&](unsigned long long higher) { take(0, higher); });
      __syncthreads();
    }
    const float thr = key_float(sel_key);
    update([&](int t, float (&v)[kE]) {
#pragma unroll
      for (int e = 0; e < kE; ++e)
        if (v[e] < thr) v[e] = kMasked;
    });
    __syncthreads();
  }

  // softmax (sampling.rs:160-190) of the current row: its max and sum.  In
  // LDS the row becomes its exponentials (the values are in memory by then);
  // in memory they are recomputed when a probability is needed.
  float sm_max = 0.f, sm_sum = 1.f;
  bool sm_uniform = true;
  const float sm_u = 1.0f / (float)vocab64;
  auto exponential = [&](float v) { return v <= kMasked ? 0.0f : expf(v - sm_max); };
  auto softmax_row = [&]() {
    float mloc = -INFINITY;
    tiles([&](int t, float (&v)[kE]) {
#pragma unroll
      for (int e = 0; e < kE; ++e) mloc = valid(t, e) && v[e] > mloc ? v[e] : mloc;
    });
    sm_max = block_max(mloc, s);
    sm_uniform = !(sm_max == sm_max) || isinf(sm_max) || sm_max <= kMasked;
    float part = 0.f;
    if (!sm_uniform) {
      own([&](int t, float (&v)[kE]) {
#pragma unroll
        for (int e = 0; e < kE; ++e) {
          v[e] = valid(t, e) ? exponential(v[e]) : 0.0f;
          part += v[e];
        }
      });
    }
    sm_sum = block_sum(part, s);
    if (!sm_uniform && !(sm_sum > 0.0f)) sm_uniform = true;
  };
  copy_row(own_row, gx);

  // ---- top-p (sampling.rs:108-144): keep the most probable candidates until
  // their mass reaches p, the crossing one included.  The crossing
  // probability K is found by a radix select on probability keys
  // (descending), the bucket masses summed exactly in 2^-40 fixed point with
  // integer atomics (order-independent, so deterministic); then tokens above
  // K are kept, plus the first tied ones (index order) the cumulative sum
  // needs. ----
  if (sp.top_p < 1.0f) {
    softmax_row();
    // the candidates' probabilities, 0 for what is no candidate
    auto candidate = [&](float v) {
      return !(v > kMasked) ? 0.0f : sm_uniform ? sm_u : exponential(v) / sm_sum;
    };
    if constexpr (OWN) {
      if (sm_uniform) copy_row(gx, own_row);
      update([&](int t, float (&v)[kE]) {
#pragma unroll
        for (int e = 0; e < kE; ++e) v[e] = sm_uniform ? candidate(v[e]) : v[e] / sm_sum;
      });
    }
    auto candidates = [&](auto f) {
      tiles([&](int t, float (&v)[kE]) {
#pragma unroll
        for (int e = 0; e < kE; ++e)
          v[e] = !valid(t, e) ? 0.0f : OWN ? v[e] : candidate(v[e]);
        f(t, v);
      });
    };
    constexpr double kFix = 1099511627776.0;  // 2^40
    // (at least one unit: the first candidate always reaches a positive p)
    const unsigned long long p_fix =
        max((unsigned long long)((double)sp.top_p * kFix), 1ull);
    if (tid == 0) {
      sel_above = 0ull;
      sel_key = 0u;
      sel_found = 1;
    }
    for (int d = 0; d < kDigits; ++d) {
      clear_buckets();
      __syncthreads();
      const uint32_t pre = sel_key;
      const unsigned long long above0 = sel_above;
      const uint32_t above = above_mask(d), mask = digit_mask(d);
      const int shift = digit_shift(d);
      candidates([&](int, float (&pv)[kE]) {
#pragma unroll
        for (int e = 0; e < kE; ++e) {
          const uint32_t k = __float_as_uint(pv[e]);
          if (pv[e] > 0.0f && (k & above) == pre)
            atomicAdd(&bucket[(k >> shift) & mask], (unsigned long long)((double)pv[e] * kFix));
        }
      });
      __syncthreads();
      // no bucket reaches p: at the first digit the whole candidate mass is
      // below it and every candidate stays (cutoff = len)
      pick(above0, p_fix,
           [&](int b, unsigned long long higher) {
             sel_key = pre | ((uint32_t)b << shift);
             sel_above = higher;
           },
           [&](unsigned long long higher) {
             if (d == 0) sel_found = 0;
             sel_key = pre;
             sel_above = higher;
           });
      __syncthreads();
      if (!sel_found) break;
    }
    if (sel_found) {
      const float K = __uint_as_float(sel_key);
      const float above = (float)((double)sel_above / kFix);
      uint32_t ties_loc = 0;
      candidates([&](int, float (&pv)[kE]) {
#pragma unroll
        for (int e = 0; e < kE; ++e) ties_loc += (pv[e] > 0.0f && pv[e] == K) ? 1u : 0u;
      });
      const uint32_t ties = block_count(ties_loc, s);
      // tied tokens the cumulative sum takes before reaching p (at least one)
      uint32_t need = 0;
      float cum = above;
      while (need < ties && cum < sp.top_p) {
        cum += K;
        ++need;
      }
      // tie ranks in index order, where not every tied token stays: a prefix
      // over threads per tile, carried across tiles
      uint32_t carry = 0;
      candidates([&](int t, float (&pv)[kE]) {
        uint32_t rank = 0;
        if (need < ties) {  // uniform over the workgroup
          uint32_t mine = 0;
#pragma unroll
          for (int e = 0; e < kE; ++e) mine += (pv[e] > 0.0f && pv[e] == K) ? 1u : 0u;
          rank = carry + block_exclusive_prefix(mine, s.u);
          carry += block_count(mine, s);
        }
#pragma unroll
        for (int e = 0; e < kE; ++e) {
          if (!(pv[e] > 0.0f)) continue;
          bool keep = pv[e] > K;
          if (pv[e] == K) keep = rank++ < need;
          if (!keep) gx[base(t) + e] = kMasked;
        }
      });
    }
    copy_row(gx, own_row);
  }

  // ---- final softmax and the draw (sample_from, sampling.rs:208-223): the
  // first index whose cumulative probability exceeds r; past the end, the
  // last index with a non-zero probability.  (The filtered row is in memory:
  // the reference's &mut logits.) ----
  softmax_row();
  const float r = uniform[row];
  int64_t first = INT64_MAX, last_nz = -1;
  float carry = 0.f;  // cumulative probability before the tile
  tiles([&](int t, float (&v)[kE]) {
    if (first != INT64_MAX || t * kTile >= vocab) return;  // uniform over the workgroup
    float mine = 0.f;
    float pv[kE];
#pragma unroll
    for (int e = 0; e < kE; ++e) {
      const float ev = OWN ? v[e] : exponential(v[e]);
      pv[e] = !valid(t, e) ? 0.0f : sm_uniform ? sm_u : ev / sm_sum;
      mine += pv[e];
    }
    float cum = carry + block_exclusive_prefix(mine, s.f);
    int64_t hit = INT64_MAX;
#pragma unroll
    for (int e = 0; e < kE; ++e) {
      if (!valid(t, e)) continue;
      cum += pv[e];
      if (hit == INT64_MAX && r < cum) hit = base(t) + e;
      if (pv[e] > 0.0f) last_nz = base(t) + e;
    }
    first = block_min_i64(hit, s);  // cumulative sums only grow: the first tile with a hit
    carry += block_sum(mine, s);
  });
  if (first == INT64_MAX) {
    const int64_t last = block_max_i64(last_nz, s);
    if (tid == 0) out[row] = (int32_t)(last >= 0 ? last : vocab - 1);
  } else if (tid == 0) {
    out[row] = (int32_t)first;
  }
}

hipError_t launch_sample(hipStream_t st, float* logits, int64_t rows, int64_t vocab,
                         const SampleParams* params, const int64_t* prev_off,
                         const uint32_t* prev_tok, const float* uniform, int32_t* out) {
  if (rows == 0) return hipSuccess;
  if (vocab <= 0 || vocab > kSampleMaxVocab || rows > INT32_MAX) return hipErrorInvalidValue;
#define ORION_SAMPLE(OWN)                                                                      \
  hipLaunchKernelGGL(sample_kernel<OWN>, dim3((unsigned)rows), dim3(kT), 0, st, logits, vocab, \
                     params, prev_off, prev_tok, uniform, out)
  if (vocab <= kLdsRow)
    ORION_SAMPLE(true);
  else
    ORION_SAMPLE(false);
#undef ORION_SAMPLE
  return hipGetLastError();
}

}  // namespace orion
