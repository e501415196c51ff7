// Projection GEMMs of a decode-shaped forward (up to 64 rows) on the packed
// weights: out[M,N] = x[M,K] . W[N,K]^T, one launch each.
//
// Bound by the weight stream.  A workgroup owns 16*NT output columns over the
// whole of K; its KW waves cut K into KW contiguous ranges, each wave streams
// its range's MFMA B fragments (one contiguous KiB per 16 columns and 32 k)
// straight into registers, U k-steps ahead of the MFMAs, and the waves' partial
// tiles are summed in LDS in a fixed order.  So no partial tile leaves the CU
// and no reduce launch follows.  The split over workgroups this replaces
// (slices of 256 k, partials in memory, a reduce launch per GEMM) wrote and
// read back 16*MT rows of partials per slice: 102 MB at 45 rows x 37888
// columns x 3584 (271 MB of weights), 150 + 16 us against 61 us here (4.5 TB/s).
//
// What it pays instead is x: every workgroup reads all of it from L2, at about
// 75 KB/us per CU.  Hence
//  * the columns per workgroup (rows_shape): as few workgroups as there are
//    CUs, so each CU reads x once (32 rows x 32000 columns x 2048, repeated: 26
//    us with 250 workgroups of 128 columns, 33 us with 500 of 64, 42 us before;
//    27.8 us in a step, 4.7 TB/s);
//  * activations in fragment order past 8 rows (kFrag): the producer writes
//    them split into hi/lo bf16 in the order the lanes read, so a load is one
//    contiguous KiB and no wave splits (32 rows x 2048 x 2048, repeated: 10.4 us
//    from f32 rows, 7.6 us; 9.5 us in a step); up to 8 rows the f32 rows are
//    fewer bytes than 16 padded ones, and stay;
//  * a K split over workgroups where x is far more than a CU's share of W
//    (rows_shape): partials of few splits and a reduce launch.
// Weights are read once: their loads are nontemporal, which keeps x in L2
// (28672 columns x 4096, 32 rows, repeated: 51 -> 44 us).
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace orion {

namespace {

__device__ inline bf16x8 frag_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ inline uint4 load_stream16(const uint16_t* p) {
  typedef unsigned int v4u __attribute__((ext_vector_type(4)));
  const v4u v = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(p));
  return uint4{v.x, v.y, v.z, v.w};
}

// One finished element of an output tile, 16 consecutive lanes holding 16
// consecutive columns of one row (all 16 call this together).
__device__ inline void rows_epilogue(const RowsGemm& g, int row, int col, float v, float pre) {
  const int c = col & 15;
  const bool live = row < (int)g.M && col < (int)g.N;
  if (g.ep == Epilogue::kSwiGLU) {  // columns [0, 8) of a tile gate, [8, 16) up
    const float u = __shfl_xor(v, 8);
    if (c >= 8 || !live) return;
    const float act = v / (1.0f + __expf(-v)) * u;
    const int oc = (col & ~15) / 2 + c;
    if (g.out_frag)
      store_frag(g.out_frag, act_tiles(g.M), row, oc, act);
    else
      g.out[(int64_t)row * (g.N >> 1) + oc] = act;
  } else if (g.ep == Epilogue::kAccumulate) {
    const float nv = pre + v;
    if (live) {
      g.out[(int64_t)row * g.N + col] = nv;
      if (g.out_frag) store_frag(g.out_frag, act_tiles(g.M), row, col, nv * g.next_weight[col]);
    }
    if (g.sumsq_out) {  // f64 sum of squares of the tile's 16 columns
      double q = live ? (double)nv * (double)nv : 0.0;
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) q += __shfl_xor(q, o);
      if (c == 0 && live) g.sumsq_out[(int64_t)row * ((g.N + 15) >> 4) + (col >> 4)] = q;
    }
  } else if (live) {
    const int oc = packed_column(col, g.pair_dim, g.pair_cols);
    g.out[(int64_t)row * g.N + oc] = g.bias ? v + g.bias[oc] : v;
  }
}

// QKV with RoPE and the cache write: the 16 columns of a Q or K tile are 8 of
// the head's first half and the 8 they rotate with (packed_column), a V tile
// 16 consecutive ones.  The same f32 expressions as rope_cache_kernel.
__device__ inline void rope_epilogue(const RowsGemm& g, int row, int col, float v,
                                     const RowSlot& slot) {
#pragma clang fp contract(off)
  const RopeOut& r = g.rope;
  const int D = (int)g.pair_dim, half = D >> 1;
  const int oc = packed_column(col, g.pair_dim, g.pair_cols);
  if (g.bias && col < (int)g.N) v = v + g.bias[oc];
  const float w = __shfl_xor(v, 8);  // the rotate-half partner (Q and K tiles)
  if (row >= (int)g.M || col >= (int)g.N) return;
  const int unit = oc / D, i = oc - unit * D;
  if (unit >= r.hq + r.hkv) {
    store_kv1(r.kv, r.kv_bf16, slot.kv + r.v_off + (int64_t)(unit - r.hq - r.hkv) * r.head + i, v);
    return;
  }
  const int j = i < half ? i : i - half;
  const float cs = r.cos[(int64_t)slot.pos * half + j], sn = r.sin[(int64_t)slot.pos * half + j];
  const float y = i < half ? v * cs - w * sn : w * sn + v * cs;
  if (unit < r.hq)
    r.q_out[((int64_t)row * r.hq + unit) * D + i] = y;
  else
    store_kv1(r.kv, r.kv_bf16, slot.kv + (int64_t)(unit - r.hq) * r.head + i, y);
}

// Waves per workgroup: 16 (128 registers each) where the tile leaves room for
// two k-steps in flight, else 8; and k-steps in flight per wave.
constexpr int rows_step_regs(int MT, int NT, bool frag) { return MT * 8 + NT * 4 + (frag ? 0 : 8); }
constexpr int rows_waves(int MT, int NT, bool frag) {
  return MT * NT * 4 + 2 * rows_step_regs(MT, NT, frag) <= 84 ? 16 : 8;
}
constexpr int rows_ahead(int MT, int NT, bool frag) {
  const int budget = (rows_waves(MT, NT, frag) == 16 ? 92 : 200) - MT * NT * 4;
  const int u = budget / rows_step_regs(MT, NT, frag);
  return u < 1 ? 1 : u > 6 ? 6 : u;
}
// Threads that sum one row's norm slots.
constexpr int rows_norm_threads(int MT, int KW) {
  const int t = 64 * KW / (MT * 16);
  return t >= 32 ? 32 : t >= 16 ? 16 : 8;
}

}  // namespace

// FRAG: x arrives in fragment order, its norm weight already multiplied in;
// otherwise as f32 rows.  The row's norm scale multiplies the finished sums.
template <int MT, int NT, bool FRAG>
__global__ void __launch_bounds__(64 * rows_waves(MT, NT, FRAG)) gemm_rows_kernel(RowsGemm g) {
  constexpr int KW = rows_waves(MT, NT, FRAG), HW = KW / 2, U = rows_ahead(MT, NT, FRAG);
  constexpr int TPR = rows_norm_threads(MT, KW);
  __shared__ float4 red[HW][MT * NT][64];
  __shared__ float nscale[MT * 16];
  __shared__ RowSlot slots[MT * 16];
  const int M = (int)g.M, N = (int)g.N, K = (int)g.K;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, grp = lane >> 4;
  const int ksteps = K >> 5, ctiles = (N + 15) >> 4;
  const int part = blockIdx.y * KW + wave, parts = gridDim.y * KW;
  const int ks0 = (int)((int64_t)part * ksteps / parts);
  const int n = (int)((int64_t)(part + 1) * ksteps / parts) - ks0;
  const int t0 = blockIdx.x * NT;

  // the norm slots go out first: they are waited for first
  constexpr int kSlots = 8;
  double sq[kSlots];
  const int nrow = tid / TPR, nj = tid % TPR;
  const double* sp = nullptr;
  if (g.norm_sumsq) {
    sp = g.norm_sumsq + (int64_t)min(nrow, M - 1) * g.norm_slots;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int s = nj + i * TPR;
      const double v = sp[min(s, g.norm_slots - 1)];
      sq[i] = s < g.norm_slots ? v : 0.0;
    }
  }

  const uint16_t* wp[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    wp[nt] = g.w + ((int64_t)min(t0 + nt, ctiles - 1) * ksteps + ks0) * 512 + lane * 8;
  const float* xp[MT];
  const uint4* xf = reinterpret_cast<const uint4*>(g.x) + (int64_t)ks0 * (MT * 128) + lane;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xp[mt] = g.x + (int64_t)min(mt * 16 + l16, M - 1) * K + ks0 * 32 + grp * 8;
  const float* nwp = g.norm_weight ? g.norm_weight + ks0 * 32 + grp * 8 : nullptr;

  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint4 b[U][NT], a[U][MT][2];
  float4 nw[U][2];
  auto load = [&](int u, int s) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if constexpr (FRAG) {
        a[u][mt][0] = xf[(int64_t)s * (MT * 128) + mt * 128];
        a[u][mt][1] = xf[(int64_t)s * (MT * 128) + mt * 128 + 64];
      } else {
        a[u][mt][0] = *reinterpret_cast<const uint4*>(xp[mt] + s * 32);
        a[u][mt][1] = *reinterpret_cast<const uint4*>(xp[mt] + s * 32 + 4);
      }
    }
    if constexpr (!FRAG) {
      if (nwp) {
        nw[u][0] = *reinterpret_cast<const float4*>(nwp + s * 32);
        nw[u][1] = *reinterpret_cast<const float4*>(nwp + s * 32 + 4);
      } else {
        nw[u][0] = nw[u][1] = make_float4(1.f, 1.f, 1.f, 1.f);
      }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) b[u][nt] = load_stream16(wp[nt] + (int64_t)s * 512);
  };
  auto compute = [&](int u) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      bf16x8 hi, lo;
      if constexpr (FRAG) {
        hi = frag_bf16x8(a[u][mt][0]);
        lo = frag_bf16x8(a[u][mt][1]);
      } else {
        float v[8], wv[8];
        __builtin_memcpy(v, &a[u][mt][0], 16);
        __builtin_memcpy(v + 4, &a[u][mt][1], 16);
        __builtin_memcpy(wv, &nw[u][0], 32);
        uint4 h, l;
        split2_rne(v[0] * wv[0], v[1] * wv[1], h.x, l.x);
        split2_rne(v[2] * wv[2], v[3] * wv[3], h.y, l.y);
        split2_rne(v[4] * wv[4], v[5] * wv[5], h.z, l.z);
        split2_rne(v[6] * wv[6], v[7] * wv[7], h.w, l.w);
        hi = frag_bf16x8(h);
        lo = frag_bf16x8(l);
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const bf16x8 wb = frag_bf16x8(b[u][nt]);
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, wb, acc[mt][nt], 0, 0, 0);
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, wb, acc[mt][nt], 0, 0, 0);
      }
    }
  };
  if (n > 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, min(u, n - 1));
  }
  __builtin_amdgcn_sched_barrier(0);
  // scale = 1 / sqrt(mean(x^2) + eps), from the f64 sums as rmsnorm_kernel does
  if (g.norm_sumsq) {
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) t += sq[i];
    for (int s = nj + kSlots * TPR; s < g.norm_slots; s += TPR) t += sp[s];
#pragma unroll
    for (int o = TPR / 2; o > 0; o >>= 1) t += __shfl_xor(t, o);
    if (nj == 0 && nrow < MT * 16)
      nscale[nrow] = (float)(1.0 / sqrt(t / (double)K + (double)g.norm_eps));
  }
  if (g.rope.q_out && tid < MT * 16) slots[tid] = row_slot(g.rope, min(tid, M - 1));
  if (n > 0) {
    int s = 0;
    for (; s + U < n; s += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        compute(u);
        load(u, min(s + U + u, n - 1));
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < n) compute(u);
  }

  // The residuals an accumulate adds to, in flight while the sums meet.
  constexpr int kIters = (MT * NT * 256 + 64 * KW - 1) / (64 * KW);
  constexpr bool kPreload = kIters <= 4;
  float pre[kPreload ? kIters : 1];
  const bool residual = g.ep == Epilogue::kAccumulate && !g.partial;
  auto element = [&](int idx, int& row, int& col) {
    const int tile = idx >> 8, mt = tile / NT;
    row = mt * 16 + ((idx >> 4) & 15);
    col = (t0 + tile - mt * NT) * 16 + (idx & 15);
  };
  if constexpr (kPreload) {
#pragma unroll
    for (int j = 0; j < kIters; ++j) {
      int row, col;
      element(tid + j * 64 * KW, row, col);
      pre[j] = residual && row < M && col < N ? g.out[(int64_t)row * N + col] : 0.f;
    }
  }
  // The waves' sums: the upper half through LDS into the lower half's, which
  // the epilogue adds in wave order.
  if (wave >= HW) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        red[wave - HW][mt * NT + nt][lane] = __builtin_bit_cast(float4, acc[mt][nt]);
  }
  __syncthreads();
  if (wave < HW) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        f32x4* p = reinterpret_cast<f32x4*>(&red[wave][mt * NT + nt][lane]);
        *p = acc[mt][nt] + *p;
      }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kIters; ++j) {
    const int idx = tid + j * 64 * KW;
    if (idx >= MT * NT * 256) break;  // (whole waves)
    int row, col;
    element(idx, row, col);
    const int tile = idx >> 8, r16 = (idx >> 4) & 15;
    const bool live = row < M && col < N;
    float res = 0.f;
    if constexpr (kPreload)
      res = pre[j];
    else if (residual && live)
      res = g.out[(int64_t)row * N + col];
    float v = 0.f;
#pragma unroll
    for (int h = 0; h < HW; ++h)
      v += reinterpret_cast<const float*>(&red[h][tile][(r16 >> 2) * 16 + (idx & 15)])[r16 & 3];
    if (g.norm_sumsq) v *= nscale[row];
    if (g.partial) {
      if (live) g.partial[((int64_t)blockIdx.y * M + row) * N + col] = v;
    } else if (g.rope.q_out) {
      rope_epilogue(g, row, col, v, slots[row]);
    } else {
      rows_epilogue(g, row, col, v, res);
    }
  }
}

// Sums the K splits of gemm_rows_kernel in split order and applies the
// epilogue; 16 consecutive threads per 16 columns of a row.
template <int S>
__global__ void __launch_bounds__(256) gemm_rows_reduce_kernel(RowsGemm g) {
  const int N = (int)g.N, npad = (N + 15) & ~15;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= g.M * npad) return;  // whole 16-lane groups exit together
  const int row = (int)(idx / npad), col = (int)(idx - (int64_t)row * npad);
  const int64_t at = (int64_t)row * N + min(col, N - 1);
  const float pre = g.ep == Epilogue::kAccumulate ? g.out[at] : 0.f;
  float t[S];
#pragma unroll
  for (int s = 0; s < S; ++s) t[s] = g.partial[(int64_t)s * g.M * N + at];
  float v = 0.f;
#pragma unroll
  for (int s = 0; s < S; ++s) v += t[s];
  rows_epilogue(g, row, col, v, pre);
}

namespace {

// Column tiles and K splits of an M x N x K call.
struct RowsShape {
  int nt, splits, grid;
};

constexpr int kRowsCus = 256;
// column tiles a workgroup may own (instantiated below)
constexpr int kRowsNt[] = {1, 2, 3, 4, 6, 8, 10};

// The fewest tiles per workgroup that put splits * tiles on the CUs in whole
// rounds (one round wherever the widest workgroup allows it).
RowsShape rows_split(int64_t tiles, int64_t splits, int64_t M) {
  const int64_t widest = M > 48 ? 8 : 10;  // (four row tiles x 10: more LDS than a CU has)
  const int64_t items = tiles * splits;
  const int64_t rounds = (items + kRowsCus * widest - 1) / (kRowsCus * widest);
  const int64_t want = (items + kRowsCus * rounds - 1) / (kRowsCus * rounds);
  RowsShape s{(int)widest, (int)splits, 0};
  for (int nt : kRowsNt)
    if (nt >= want) {
      s.nt = nt;
      break;
    }
  s.grid = (int)((tiles + s.nt - 1) / s.nt);
  return s;
}

// K splits, for the residual GEMMs (the norm and pair epilogues need whole
// sums): the count with the least of W per workgroup / 22 KB/us + x per
// workgroup / 80 KB/us + 4 + S / 4 us for the partials and the reduce launch,
// fitted to 1 .. 64 rows of 2048 x 2048, 2048 x 5632, 4096 x 4096, 4096 x
// 14336, 3584 x 3584 and 3584 x 18944, where it picks the fastest of 1, 2, 4
// and 8 or one within 1.5 us of it.  For instance 32 rows x 2048 x 5632: 18.0
// us whole, 11.5 in 4; 45 x 3584 x 18944: 66 whole, 35 in 8; 6 x 4096 x 4096:
// 9.2 whole, 12.2 in 2.
RowsShape rows_shape(int64_t M, int64_t N, int64_t K, Epilogue ep, bool frag) {
  const int64_t tiles = (N + 15) / 16;
  RowsShape best = rows_split(tiles, 1, M);
  if (ep != Epilogue::kAccumulate) return best;
  const double x_kb = frag ? act_tiles(M) * 16 * K / 256.0 : M * K / 256.0;
  double best_us = 0;
  for (int splits : {1, 2, 4, 8}) {
    if (K / 32 < 32 * splits && splits > 1) break;  // at least 2 k-steps a wave
    const RowsShape s = rows_split(tiles, splits, M);
    if (splits > 1 && (int64_t)s.grid * splits > kRowsCus) continue;
    const double us = s.nt * (K / 32.0) / splits / 22 + x_kb / splits / 80 +
                      (splits > 1 ? 4 + splits * 0.25 : 0);
    if (splits == 1 || us < best_us) {
      best = s;
      best_us = us;
    }
  }
  return best;
}

template <int MT, bool FRAG>
hipError_t launch_mt(hipStream_t st, const RowsGemm& g, const RowsShape& s) {
  const dim3 grid((unsigned)s.grid, (unsigned)s.splits);
#define ORION_ROWS(NT)                                                                      \
  case NT:                                                                                  \
    hipLaunchKernelGGL((gemm_rows_kernel<MT, NT, FRAG>), grid,                               \
                       dim3(64 * rows_waves(MT, NT, FRAG)), 0, st, g);                      \
    break;
  switch (s.nt) {
    ORION_ROWS(1)
    ORION_ROWS(2)
    ORION_ROWS(3)
    ORION_ROWS(4)
    ORION_ROWS(6)
    ORION_ROWS(8)
    default:
      if constexpr (MT < 4) {
        switch (s.nt) { ORION_ROWS(10) }
      } else {
        return hipErrorInvalidValue;
      }
  }
#undef ORION_ROWS
  return hipGetLastError();
}

}  // namespace

size_t rows_scratch_bytes(const RowsGemm& g) {
  const RowsShape s = rows_shape(g.M, g.N, g.K, g.ep, g.x_frag);
  return s.splits > 1 ? (size_t)s.splits * (size_t)(g.M * g.N) * sizeof(float) : 0;
}

hipError_t launch_gemm_rows(hipStream_t st, const RowsGemm& call, float* scratch,
                            size_t scratch_bytes) {
  RowsGemm g = call;
  if (g.M < 1 || g.M > kRowsMax || g.K % 32 || g.K < 32 || g.N < 1 || g.N > INT32_MAX - 256 ||
      g.K > INT32_MAX || !g.w || !g.x)
    return hipErrorInvalidValue;
  if (g.ep == Epilogue::kSwiGLU && g.N % 16) return hipErrorInvalidValue;
  if (g.norm_sumsq && g.norm_slots < 1) return hipErrorInvalidValue;
  if (g.out_frag && g.ep == Epilogue::kAccumulate && !g.next_weight) return hipErrorInvalidValue;
  if (g.rope.q_out && (g.ep != Epilogue::kStore || g.pair_dim < 16)) return hipErrorInvalidValue;
  const RowsShape s = rows_shape(g.M, g.N, g.K, g.ep, g.x_frag);
  g.partial = nullptr;
  if (s.splits > 1) {
    if (scratch_bytes < rows_scratch_bytes(g)) return hipErrorInvalidValue;
    g.partial = scratch;
  }
  hipError_t e;
  switch ((g.M + 15) / 16) {
    case 1: e = g.x_frag ? launch_mt<1, true>(st, g, s) : launch_mt<1, false>(st, g, s); break;
    case 2: e = g.x_frag ? launch_mt<2, true>(st, g, s) : launch_mt<2, false>(st, g, s); break;
    case 3: e = g.x_frag ? launch_mt<3, true>(st, g, s) : launch_mt<3, false>(st, g, s); break;
    default: e = g.x_frag ? launch_mt<4, true>(st, g, s) : launch_mt<4, false>(st, g, s); break;
  }
  if (e != hipSuccess || s.splits == 1) return e;
  const int64_t threads = g.M * ((g.N + 15) & ~(int64_t)15);
  const dim3 grid((unsigned)((threads + 255) / 256));
  switch (s.splits) {
    case 2: hipLaunchKernelGGL(gemm_rows_reduce_kernel<2>, grid, dim3(256), 0, st, g); break;
    case 4: hipLaunchKernelGGL(gemm_rows_reduce_kernel<4>, grid, dim3(256), 0, st, g); break;
    default: hipLaunchKernelGGL(gemm_rows_reduce_kernel<8>, grid, dim3(256), 0, st, g); break;
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Packed weights
// ---------------------------------------------------------------------------

// One thread per 16-byte unit: unit (column tile, k-step, lane), lane l holding
// columns l % 16 and k 8 * (l / 16) .. + 8 of the fragment.  Columns past N are
// zero.
__global__ void __launch_bounds__(256)
    pack_weights_kernel(const uint16_t* __restrict__ w, int N, int K, int pair_dim, int pair_cols,
                        int64_t units, uint4* __restrict__ out) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;
  const int lane = (int)(u & 63), ksteps = K >> 5;
  const int64_t f = u >> 6;
  const int col = (int)(f / ksteps) * 16 + (lane & 15);
  const int k = (int)(f % ksteps) * 32 + (lane >> 4) * 8;
  uint4 v = uint4{0u, 0u, 0u, 0u};
  if (col < N)
    v = *reinterpret_cast<const uint4*>(
        w + (int64_t)packed_column(col, pair_dim, pair_cols) * K + k);
  out[u] = v;
}

// The inverse.
__global__ void __launch_bounds__(256)
    unpack_weights_kernel(const uint4* __restrict__ in, int N, int K, int pair_dim, int pair_cols,
                          int64_t units, uint16_t* __restrict__ w) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;
  const int lane = (int)(u & 63), ksteps = K >> 5;
  const int64_t f = u >> 6;
  const int col = (int)(f / ksteps) * 16 + (lane & 15);
  const int k = (int)(f % ksteps) * 32 + (lane >> 4) * 8;
  if (col < N)
    *reinterpret_cast<uint4*>(w + (int64_t)packed_column(col, pair_dim, pair_cols) * K + k) =
        in[u];
}

size_t packed_weight_bytes(int64_t N, int64_t K) {
  if (K % 32 != 0 || K <= 0 || N <= 0) return 0;
  return (size_t)((N + 15) / 16) * (size_t)(K / 32) * 1024;
}

hipError_t launch_pack_weights(hipStream_t st, const uint16_t* w, int64_t N, int64_t K,
                               int64_t pair_dim, int64_t pair_cols, uint16_t* out) {
  if (K % 32 != 0 || K <= 0 || N <= 0 || N > INT32_MAX - 16 || K > INT32_MAX)
    return hipErrorInvalidValue;
  const int64_t units = (int64_t)packed_weight_bytes(N, K) / 16;
  hipLaunchKernelGGL(pack_weights_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, st,
                     w, (int)N, (int)K, (int)pair_dim, (int)pair_cols, units,
                     reinterpret_cast<uint4*>(out));
  return hipGetLastError();
}

hipError_t launch_unpack_weights(hipStream_t st, const uint16_t* packed, int64_t N, int64_t K,
                                 int64_t pair_dim, int64_t pair_cols, uint16_t* w) {
  if (K % 32 != 0 || K <= 0 || N <= 0 || N > INT32_MAX - 16 || K > INT32_MAX)
    return hipErrorInvalidValue;
  const int64_t units = (int64_t)packed_weight_bytes(N, K) / 16;
  hipLaunchKernelGGL(unpack_weights_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0,
                     st, reinterpret_cast<const uint4*>(packed), (int)N, (int)K, (int)pair_dim,
                     (int)pair_cols, units, w);
  return hipGetLastError();
}

}  // namespace orion
