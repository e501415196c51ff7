// Projection GEMMs on bf16 MFMA for gfx950: out[M,N] = x[M,K] . W[N,K]^T.
//
// Restates the reference's `linear` (crates/orion-models/src/tensor.rs:96-130):
// W keeps the HF layout [out_features, in_features] (row-major, K contiguous),
// which is exactly the MFMA B-operand layout: a lane loads 8 consecutive k of
// one output column with one 16-byte load, straight from HBM into registers.
//
// Activations arrive in f32.  Each 8-element A fragment is split on the fly
// into hi = the top 16 bits of x and lo = the top 16 bits of (x - hi) and both
// are multiplied against the bf16 weight (two MFMAs, f32 accumulation), so the
// product carries ~16 mantissa bits of x instead of 8.  Weights are exact
// (bf16 checkpoints widen exactly in the reference loader), so the only
// departure from the reference's f32 arithmetic is summation order plus a
// ~2^-16 relative term per product.
//
// The epilogue fuses the bias add, the residual accumulate
// (transformer.rs:328-332, :345) or SwiGLU (tensor.rs:175-189) on gate/up rows
// interleaved in groups of 8.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

namespace orion {

__device__ inline bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// x -> (hi, lo) bf16 fragments by truncation (x = hi + lo to ~2^-16 relative).
__device__ inline void split8(const float (&a)[8], bf16x8& hi, bf16x8& lo) {
  uint4 hv, lv;
  split2_trunc(a[0], a[1], hv.x, lv.x);
  split2_trunc(a[2], a[3], hv.y, lv.y);
  split2_trunc(a[4], a[5], hv.z, lv.z);
  split2_trunc(a[6], a[7], hv.w, lv.w);
  hi = as_bf16x8(hv);
  lo = as_bf16x8(lv);
}

// Decode-shaped (small M) weight-streaming GEMM.  Workgroup = KW waves on one
// 16*NT-column tile of up to 16*MT rows; the waves split K into KW contiguous
// ranges and each walks its range UNR k-steps (32 k each) at a time, so UNR
// weight loads per column tile are in flight before the MFMAs consume them.
// Each x fragment (loaded from L2) feeds NT column tiles.  The KW partial
// tiles are summed through LDS in wave order (deterministic) and the epilogue
// is applied once.  Weights are read from HBM exactly once per 16*MT rows.
template <int MT, int NT, int KW, int UNR>
__global__ void __launch_bounds__(64 * KW)
    gemm_skinny_kernel(const float* __restrict__ x, const uint16_t* __restrict__ w,
                       const float* __restrict__ bias, int M, int N, int K, int ep,
                       float* __restrict__ out) {
  constexpr int BN = 16 * NT;
  constexpr int BM = 16 * MT;
  __shared__ float red[KW][BM][BN + 1];

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * BM;
  const int n0 = blockIdx.x * BN;
  const int mt_count = min(MT, (M - m0 + 15) >> 4);
  const int ksteps = K >> 5;
  const int ks0 = wave * ksteps / KW;
  const int ks1 = (wave + 1) * ksteps / KW;
  const int lr = lane & 15;
  const int lk = (lane >> 4) * 8;

  const uint16_t* wrow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = min(n0 + nt * 16 + lr, N - 1);
    wrow[nt] = w + (int64_t)n * K + lk;
  }
  const float* xrow[MT];
  bool xvalid[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + mt * 16 + lr;
    xvalid[mt] = m < M;
    xrow[mt] = x + (int64_t)min(m, M - 1) * K + lk;
  }

  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int ks = ks0; ks < ks1; ks += UNR) {
    // Fragments for UNR k-steps (indices clamped into the range; the
    // products of a clamped step are skipped below).
    bf16x8 b[UNR][NT];
    float4 a0[UNR][MT], a1[UNR][MT];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int k = min(ks + u, ks1 - 1) << 5;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        b[u][nt] = as_bf16x8(*reinterpret_cast<const uint4*>(wrow[nt] + k));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if (mt < mt_count && xvalid[mt]) {
          a0[u][mt] = *reinterpret_cast<const float4*>(xrow[mt] + k);
          a1[u][mt] = *reinterpret_cast<const float4*>(xrow[mt] + k + 4);
        } else {
          a0[u][mt] = make_float4(0.f, 0.f, 0.f, 0.f);
          a1[u][mt] = a0[u][mt];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      if (ks + u < ks1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          if (mt < mt_count) {
            const float a[8] = {a0[u][mt].x, a0[u][mt].y, a0[u][mt].z, a0[u][mt].w,
                                a1[u][mt].x, a1[u][mt].y, a1[u][mt].z, a1[u][mt].w};
            bf16x8 ahi, alo;
            split8(a, ahi, alo);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
              acc[mt][nt] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahi, b[u][nt], acc[mt][nt], 0, 0, 0);
              acc[mt][nt] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(alo, b[u][nt], acc[mt][nt], 0, 0, 0);
            }
          }
        }
      }
    }
  }

  // C fragment layout: lane holds rows 4*(lane/16) + i, column lane % 16.
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (mt < mt_count) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          red[wave][mt * 16 + (lane >> 4) * 4 + i][nt * 16 + lr] = acc[mt][nt][i];
    }
  }
  __syncthreads();

  const int rows = min(BM, M - m0);
  if (ep == (int)Epilogue::kSwiGLU) {
    // Tile columns nt*16 + [0,8) are gate rows, nt*16 + [8,16) the matching up rows.
    const int half_n = N >> 1;
    for (int idx = threadIdx.x; idx < rows * NT * 8; idx += 64 * KW) {
      const int r = idx / (NT * 8);
      const int cc = idx - r * (NT * 8);
      const int nt = cc >> 3, j = cc & 7;
      const int gcol = n0 + nt * 16 + j;
      if (gcol >= N) continue;
      float g = 0.f, u = 0.f;
#pragma unroll
      for (int wv = 0; wv < KW; ++wv) {
        g += red[wv][r][nt * 16 + j];
        u += red[wv][r][nt * 16 + 8 + j];
      }
      const float act = g / (1.0f + __expf(-g)) * u;
      out[(int64_t)(m0 + r) * half_n + (n0 >> 1) + nt * 8 + j] = act;
    }
  } else {
    for (int idx = threadIdx.x; idx < rows * BN; idx += 64 * KW) {
      const int r = idx / BN;
      const int cc = idx - r * BN;
      const int col = n0 + cc;
      if (col >= N) continue;
      float v = 0.f;
#pragma unroll
      for (int wv = 0; wv < KW; ++wv) v += red[wv][r][cc];
      float* op = out + (int64_t)(m0 + r) * N + col;
      if (ep == (int)Epilogue::kAccumulate)
        *op += v;
      else
        *op = bias ? v + bias[col] : v;
    }
  }
}

// Prefill-shaped (large M) GEMM: 128 x 128 output tile per 256-thread
// workgroup (2 x 2 waves of 64 x 64), k-steps of 32.  The f32 activation tile
// (128 x 32) and the bf16 weight tile (128 x 32) are copied HBM -> LDS with
// global_load_lds (no staging registers), double-buffered so the next
// k-step's copy is in flight while this one computes.  Each wave splits its A
// fragments into hi/lo bf16 on the fly (as the skinny kernel does) and issues
// 4 x 4 x 2 MFMAs per k-step; B fragments are reused by the 4 row tiles and A
// fragments by the 4 column tiles.  LDS rows are XOR-swizzled in 16-byte
// chunks (conflict-free 16-byte fragment reads; the DMA writes stay linear).
namespace {
constexpr int kTN = 128, kTK = 32;
// A tile row r: 8 chunks of 4 floats; chunk c stored at c ^ swz_a(r).
__device__ inline int swz_a(int r) {
  return ((r >> 2) & 1) | (((r >> 1) & 1) << 1) | (((r >> 3) & 1) << 2);
}
// B tile row n: 4 chunks of 8 bf16; chunk c stored at c ^ swz_b(n).
__device__ inline int swz_b(int n) { return (n >> 2) & 3; }
}  // namespace

// W is either row-major [N, K] or in packed order (launch_pack_weights): there
// a 16-column x 32-k MFMA B fragment is one contiguous KiB, lane l's 16 bytes
// at l * 16, so each of the tile's fragments per k-step is copied to LDS
// verbatim and read back with one conflict-free ds_read_b128 per lane.
struct PackedGeom {
  bool packed = false;
  int pair_dim = 0, pair_cols = 0;  // packed_column
};

// The QKV tile of a wave with RoPE and the cache write (a prefill-shaped
// forward's): columns 2j and 2j + 1 of 16 hold 16 columns of a head's first half
// and the 16 they rotate with, 8 and 8 of each (packed_column), so one exchange
// within 16 lanes leaves a lane both of a pair and every store 16 consecutive
// elements.  The same f32 expressions as rope_cache_kernel.  As a kernel of its
// own RoPE re-read the f32 QKV matrix, 60 us at 17631 rows of 2560 columns, and
// storing that matrix from this column order took 22 us more; the GEMM with both
// takes 353 us.
template <int MTW, int NTW>
__device__ inline void rope_tiles(const RopeOut& r, const f32x4 (&acc)[MTW][NTW],
                                  const RowSlot* slots, int row0, int col0, int M, int N, int D,
                                  const float* __restrict__ bias) {
#pragma clang fp contract(off)
  const int l16 = threadIdx.x & 15, grp = (threadIdx.x & 63) >> 4;
  const int half = D >> 1;
  const float* __restrict__ cos_t = r.cos;
  const float* __restrict__ sin_t = r.sin;
#pragma unroll
  for (int nt = 0; nt < NTW; nt += 2) {
    const int c = col0 + 16 * nt;  // 32 columns of one head (D is a multiple of 32)
    if (c >= N) continue;
    const int unit = c / D, at = c - unit * D;
    if (unit >= r.hq + r.hkv) {  // V: as it is
      const int64_t to = r.v_off + (int64_t)(unit - r.hq - r.hkv) * r.head + at + l16;
      const float b0 = bias ? bias[c + l16] : 0.f, b1 = bias ? bias[c + 16 + l16] : 0.f;
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int rl = mt * 16 + 4 * grp + i;
          float v0 = acc[mt][nt][i], v1 = acc[mt][nt + 1][i];
          if (bias) v0 = v0 + b0, v1 = v1 + b1;
          if (row0 + rl < M) {
            store_kv1(r.kv, r.kv_bf16, slots[rl].kv + to, v0);
            store_kv1(r.kv, r.kv_bf16, slots[rl].kv + to + 16, v1);
          }
        }
      continue;
    }
    const int j = (at >> 1) + l16;  // of the first half
    const bool q = unit < r.hq;
    const int64_t k_to = (int64_t)(unit - r.hq) * r.head + j;
    const float b0 = bias ? bias[unit * D + j] : 0.f, b1 = bias ? bias[unit * D + half + j] : 0.f;
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) {
      float cs[4], sn[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t a = (int64_t)slots[mt * 16 + 4 * grp + i].pos * half + j;
        cs[i] = cos_t[a];
        sn[i] = sin_t[a];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rl = mt * 16 + 4 * grp + i;
        const float even = acc[mt][nt][i], odd = acc[mt][nt + 1][i];
        const float got = dpp<kDppRor8>(l16 < 8 ? odd : even);
        float x0 = l16 < 8 ? even : got, x1 = l16 < 8 ? got : odd;
        if (bias) x0 = x0 + b0, x1 = x1 + b1;
        const float y0 = x0 * cs[i] - x1 * sn[i], y1 = x0 * sn[i] + x1 * cs[i];
        if (row0 + rl >= M) continue;
        if (q) {
          float* to = r.q_out + ((int64_t)(row0 + rl) * r.hq + unit) * D + j;
          to[0] = y0;
          to[half] = y1;
        } else {
          store_kv1(r.kv, r.kv_bf16, slots[rl].kv + k_to, y0);
          store_kv1(r.kv, r.kv_bf16, slots[rl].kv + k_to + half, y1);
        }
      }
    }
  }
}

// HILO: x carried as a truncated hi + lo bf16 pair (two MFMAs, ~16 bits of
// x per product); otherwise rounded to bf16 (nearest even, one MFMA).
// XS (with HILO): x is already in that split layout (GemmFuse::x_hilo), so a
// fragment's two 16-byte LDS chunks are its hi and lo bf16x8 as they are.
// NTW: 16-column tiles per wave (4: 128-column workgroup tiles; 8: 256).
// out_hilo: the SwiGLU epilogue writes its output in the split layout.
// MTW: 16-row tiles per wave (TM = 32 MTW workgroup rows).  ST: k-step tiles in
// LDS (see the loop).  ROPE: the QKV GEMM, whose epilogue is rope's.
template <bool HILO, int NTW, bool XS = false, int MTW = 4, int ST = 2, bool ROPE = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NTW == 8 ? 2 : 1)))
    gemm_tiled_kernel(const float* __restrict__ x, const uint16_t* __restrict__ w,
                      const float* __restrict__ bias, int M, int N, int K, int ep,
                      float* __restrict__ out, PackedGeom pk, int gm, int kspan,
                      float* __restrict__ partial, bool out_hilo, RopeOut rope) {
  static_assert(HILO || !XS, "a pre-split x needs the hi/lo MFMAs");
  constexpr int TM = 32 * MTW;   // workgroup rows
  constexpr int TN = 32 * NTW;   // workgroup columns
  constexpr int BJ = NTW / 2;    // B copies (1 KiB each) per wave per k-step
  __shared__ __attribute__((aligned(1024))) float As[ST][TM * kTK];
  __shared__ __attribute__((aligned(1024))) uint16_t Bs[ST][TN * kTK];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int l16 = lane & 15, grp = lane >> 4;
  // Tile order.  gm == 0: the 2D grid is (n tile, m tile).  gm > 0: a 1D grid
  // of 8 * ceil(tiles / 8) workgroups in XCD-aware grouped order: workgroup b
  // runs on XCD b % 8 (round-robin dispatch), each XCD takes a contiguous
  // eighth of the tiles and walks it in groups of gm m tiles, n outer, so the
  // tiles in flight on one XCD share A and B slabs in its L2.
  int mt_i = blockIdx.y, nt_i = blockIdx.x;
  if (gm > 0) {
    const int gx = (N + TN - 1) / TN, gy = (M + TM - 1) / TM, total = gx * gy;
    const int b = blockIdx.x;
    const int per = (total + 7) / 8;
    const int t = (b & 7) * per + (b >> 3);
    if (t >= total) return;  // padding workgroups (before any barrier)
    const int g = t / (gm * gx), within = t - g * gm * gx;
    const int gm_eff = min(gm, gy - g * gm);
    mt_i = g * gm + within % gm_eff;
    nt_i = within / gm_eff;
  }
  const int m0 = mt_i * TM, n0 = nt_i * TN;

  // ---- DMA addressing: A = MTW wave instructions (8 rows x 128 B each),
  // B = BJ wave instructions (16 rows x 64 B each). ----
  const float* a_src[MTW];
  const uint16_t* b_src[BJ];
#pragma unroll
  for (int j = 0; j < MTW; ++j) {
    const int r = (wave * MTW + j) * 8 + (lane >> 3);
    const int c = (lane & 7) ^ swz_a(r);
    a_src[j] = x + (int64_t)min(m0 + r, M - 1) * K + c * 4;
  }
  // Packed W: fragment f = wave * BJ + j holds columns n0 + 16 f .. + 16
  // (clamped to the last column tile; columns past it are past N anyway), its
  // k-steps 512 elements apart.
  const bool packed = pk.packed;
#pragma unroll
  for (int j = 0; j < BJ; ++j) {
    if (packed) {
      const int c16 = min(n0 / 16 + wave * BJ + j, (N + 15) / 16 - 1);
      b_src[j] = w + (int64_t)c16 * (K / kTK) * 512 + lane * 8;
    } else {
      const int r = (wave * BJ + j) * 16 + (lane >> 2);
      const int c = (lane & 3) ^ swz_b(r);
      b_src[j] = w + (int64_t)min(n0 + r, N - 1) * K + c * 8;
    }
  }
  const int b_step = packed ? 512 : kTK;
  const uint32_t as_base = (uint32_t)(uintptr_t)&As[0][0];
  const uint32_t bs_base = (uint32_t)(uintptr_t)&Bs[0][0];
  auto load_tile = [&](int ks, int buf) {
    const int k0 = ks * kTK;
#pragma unroll
    for (int j = 0; j < MTW; ++j)
      lds_load16(a_src[j] + k0, as_base + (uint32_t)(buf * TM * kTK * 4 + (wave * MTW + j) * 1024));
#pragma unroll
    for (int j = 0; j < BJ; ++j)
      lds_load16(b_src[j] + (int64_t)ks * b_step,
                 bs_base + (uint32_t)(buf * TN * kTK * 2 + (wave * BJ + j) * 1024));
  };

  // where each row's K and V go, and its position: read while the first tiles load
  __shared__ RowSlot slots[ROPE ? TM : 1];
  auto find_slots = [&] {
    if constexpr (ROPE)
      if (tid < TM) slots[tid] = row_slot(rope, min(m0 + tid, M - 1));
  };

  // ---- fragment read addresses (bytes, buffer 0) ----
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
  uint32_t a_rd0[MTW], a_rd1[MTW], b_rd[NTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    const int r = wm * 16 * MTW + mt * 16 + l16;
    a_rd0[mt] = as_base + (uint32_t)(r * kTK + (((2 * grp) ^ swz_a(r)) * 4)) * 4;
    a_rd1[mt] = as_base + (uint32_t)(r * kTK + (((2 * grp + 1) ^ swz_a(r)) * 4)) * 4;
  }
#pragma unroll
  for (int nt = 0; nt < NTW; ++nt) {
    const int n = wn * 16 * NTW + nt * 16 + l16;
    b_rd[nt] = packed ? bs_base + (uint32_t)((wn * NTW + nt) * 1024 + lane * 16)
                      : bs_base + (uint32_t)(n * kTK + ((grp ^ swz_b(n)) * 8)) * 2;
  }

  f32x4 acc[MTW][NTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // K split z = blockIdx.z covers k-steps [z * kspan, min(ksteps, (z + 1) * kspan))
  const int ks_begin = blockIdx.z * kspan;
  const int ksteps = min(K / kTK, ks_begin + kspan);
  // ST - 1 k-steps in flight.  A k-step's copies are this wave's MTW + BJ
  // newest but (ST - 2) k-steps'; the barrier makes every wave's visible, and
  // says that all have read the tile the next copies overwrite.
  if constexpr (ST > 2) {
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
      if (ks_begin + s < ksteps) load_tile(ks_begin + s, s);
    find_slots();
  } else {
    load_tile(ks_begin, 0);
    find_slots();
    wait_vmem_all();
    __syncthreads();
  }
  int buf = 0;
  auto compute = [&] {
    const uint32_t aoff = (uint32_t)(buf * TM * kTK * 4);
    const uint32_t boff = (uint32_t)(buf * TN * kTK * 2);
    bf16x8 bw[NTW];
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt)
      bw[nt] = __builtin_bit_cast(bf16x8, *(const lds_u32x4*)(uintptr_t)(b_rd[nt] + boff));
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) {
      const u32x4 lo4 = *(const lds_u32x4*)(uintptr_t)(a_rd0[mt] + aoff);
      const u32x4 hi4 = *(const lds_u32x4*)(uintptr_t)(a_rd1[mt] + aoff);
      const float a[8] = {__uint_as_float(lo4.x), __uint_as_float(lo4.y),
                          __uint_as_float(lo4.z), __uint_as_float(lo4.w),
                          __uint_as_float(hi4.x), __uint_as_float(hi4.y),
                          __uint_as_float(hi4.z), __uint_as_float(hi4.w)};
      bf16x8 ahi, alo;
      if constexpr (XS) {
        ahi = __builtin_bit_cast(bf16x8, lo4);
        alo = __builtin_bit_cast(bf16x8, hi4);
        (void)a;
      } else if constexpr (HILO) {
        split8(a, ahi, alo);
      } else {
        typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
        typedef float f32x8 __attribute__((ext_vector_type(8)));
        const f32x8 av = {a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7]};
        ahi = __builtin_bit_cast(bf16x8, __builtin_convertvector(av, bf16x8v));
        (void)alo;
      }
#pragma unroll
      for (int nt = 0; nt < NTW; ++nt) {
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahi, bw[nt], acc[mt][nt], 0, 0, 0);
        if constexpr (HILO)
          acc[mt][nt] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(alo, bw[nt], acc[mt][nt], 0, 0, 0);
      }
    }
  };
  if constexpr (NTW == 8) {
    // The last k-step apart: a copy in every round of the loop and no branch in
    // it.  With the stores below, f32 activations, us: 16384 columns x 2048, 400
    // rows 99 -> 81, 4096 rows 548 -> 490; 32000 x 2048, 4096 rows 1001 -> 905;
    // 37888 x 3584, 4096 rows 1902 -> 1795.  (128-column tiles at three workgroups
    // per CU lose 4 to 8 % by it past 1000 rows.)
    static_assert(ST == 2, "two k-steps in LDS");
    for (int ks = ks_begin; ks + 1 < ksteps; ++ks) {
      load_tile(ks + 1, buf ^ 1);
      compute();
      wait_vmem_all();
      __syncthreads();
      buf ^= 1;
    }
    compute();
  } else {
    for (int ks = ks_begin; ks < ksteps; ++ks) {
      if constexpr (ST > 2) {
        if (ks + ST - 2 < ksteps)
          wait_vmem<(ST - 2) * (MTW + BJ)>();
        else
          wait_vmem_all();
        __syncthreads();
        if (ks + ST - 1 < ksteps) load_tile(ks + ST - 1, buf ? buf - 1 : ST - 1);
      } else if (ks + 1 < ksteps) {
        load_tile(ks + 1, buf ^ 1);
      }
      compute();
      if constexpr (ST > 2) {
        buf = buf + 1 < ST ? buf + 1 : 0;
      } else {
        wait_vmem_all();
        __syncthreads();
        buf ^= 1;
      }
    }
  }

  // ---- epilogue: acc[mt][nt][i] = C[m0 + wm*16*MTW + mt*16 + 4*grp + i][n0 + wn*16*NTW + nt*16 + l16] ----
  if constexpr (ROPE) {
    rope_tiles<MTW, NTW>(rope, acc, slots + wm * 16 * MTW, m0 + wm * 16 * MTW, n0 + wn * 16 * NTW, M,
                         N, pk.pair_dim, bias);
    return;
  }
  if (partial) {  // one K split: raw sums, reduced by gemm_tiled_reduce_kernel
    float* pz = partial + (int64_t)blockIdx.z * M * N;
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      const int col = n0 + wn * 16 * NTW + nt * 16 + l16;
      const int oc = packed_column(col, pk.pair_dim, pk.pair_cols);
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = m0 + wm * 16 * MTW + mt * 16 + 4 * grp + i;
          if (row < M && col < N) pz[(int64_t)row * N + oc] = acc[mt][nt][i];
        }
    }
    return;
  }
  if (ep == (int)Epilogue::kStore) {
    if constexpr (NTW == 8) {
      // A row's columns one after another, and whole tiles without a test per
      // element: a lane of a 256-column tile stores 128 values.
      int oc[NTW];
      float b[NTW];
#pragma unroll
      for (int nt = 0; nt < NTW; ++nt) {
        const int col = n0 + wn * 16 * NTW + nt * 16 + l16;
        oc[nt] = packed_column(col, pk.pair_dim, pk.pair_cols);
        b[nt] = bias && col < N ? bias[oc[nt]] : 0.f;
      }
      const bool whole = m0 + TM <= M && n0 + TN <= N;
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = m0 + wm * 16 * MTW + mt * 16 + 4 * grp + i;
          float* to = out + (int64_t)row * N;
          if (whole) {
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt)
              to[oc[nt]] = bias ? acc[mt][nt][i] + b[nt] : acc[mt][nt][i];
          } else if (row < M) {
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt)
              if (n0 + wn * 16 * NTW + nt * 16 + l16 < N)
                to[oc[nt]] = bias ? acc[mt][nt][i] + b[nt] : acc[mt][nt][i];
          }
        }
    } else {
#pragma unroll
      for (int nt = 0; nt < NTW; ++nt) {
        const int col = n0 + wn * 16 * NTW + nt * 16 + l16;
        const int oc = packed_column(col, pk.pair_dim, pk.pair_cols);
        const float b = bias && col < N ? bias[oc] : 0.f;
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = m0 + wm * 16 * MTW + mt * 16 + 4 * grp + i;
            if (row < M && col < N) out[(int64_t)row * N + oc] = bias ? acc[mt][nt][i] + b : acc[mt][nt][i];
          }
      }
    }
    return;
  }
  if (ep == (int)Epilogue::kAccumulate) {
    // Residual add, one 16-row tile at a time: all of its residual values are
    // loaded before any sum is stored.  Written as `out[i] += v` per element,
    // every load would wait for the stores before it (loads and stores to one
    // array keep their order), one memory round trip per element: at config
    // 4's prefill O and down shapes that epilogue cost 76 and 84 us per
    // launch.  (Loading the whole tile at once, or before the k-loop, takes
    // the kernel past the registers of three workgroups per CU.)
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) {
      float res[NTW][4];
#pragma unroll
      for (int nt = 0; nt < NTW; ++nt) {
        const int col = n0 + wn * 16 * NTW + nt * 16 + l16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = m0 + wm * 16 * MTW + mt * 16 + 4 * grp + i;
          res[nt][i] = (row < M && col < N) ? out[(int64_t)row * N + col] : 0.f;
        }
      }
#pragma unroll
      for (int nt = 0; nt < NTW; ++nt) {
        const int col = n0 + wn * 16 * NTW + nt * 16 + l16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = m0 + wm * 16 * MTW + mt * 16 + 4 * grp + i;
          if (row < M && col < N) out[(int64_t)row * N + col] = res[nt][i] + acc[mt][nt][i];
        }
      }
    }
    return;
  }
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      const int col = n0 + wn * 16 * NTW + nt * 16 + l16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + wm * 16 * MTW + mt * 16 + 4 * grp + i;
        const float v = acc[mt][nt][i];
        // kSwiGLU: tile columns [0, 8) are gate rows of W, [8, 16) the matching
        // up rows.
        const float u = __shfl_xor(v, 8);
        if (l16 < 8 && row < M && col < N) {
          const float act = v / (1.0f + __expf(-v)) * u;
          const int c8 = (n0 + wn * 16 * NTW + nt * 16) >> 1;  // a multiple of 8
          if (out_hilo) {
            uint16_t h, lo;
            split1_trunc(act, h, lo);
            uint16_t* o16 = reinterpret_cast<uint16_t*>(out) + (int64_t)row * N + c8 * 2;
            o16[l16] = h;
            o16[8 + l16] = lo;
          } else {
            out[(int64_t)row * (N >> 1) + c8 + l16] = act;
          }
        }
      }
    }
  }
}

// Sums the K splits of gemm_tiled_kernel in split order, then the store (+
// bias) or accumulate epilogue.
__global__ void __launch_bounds__(256)
    gemm_tiled_reduce_kernel(const float* __restrict__ partial, int splits, int64_t M, int64_t N,
                             const float* __restrict__ bias, int ep, float* __restrict__ out) {
  const int64_t total = M * N;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * 256) {
    float v = 0.f;
    for (int z = 0; z < splits; ++z) v += partial[z * total + i];
    if (ep == (int)Epilogue::kAccumulate)
      out[i] += v;
    else
      out[i] = bias ? v + bias[i % N] : v;
  }
}

// Few rows (M <= 64) of a row-major W, split over K across workgroups: the
// op-level entry points (a forward's decode GEMMs read packed weights,
// gemm_rows.hip).  Workgroup (256 threads) = 4 waves x NT column tiles of 16 =
// 64*NT output columns, over one K slice of KSTEPS k-steps (32 k each).
//   1. Every wave issues all of its slice's weight loads at once
//      (KSTEPS x NT 16-byte loads per lane straight into MFMA B fragments),
//      so a wave keeps KSTEPS*NT KiB in flight.
//   2. Meanwhile the workgroup stages the activation slice x[0:M, slice] in
//      LDS once, already split into hi/lo bf16 A fragments (lane-major), so
//      the 4 waves share one read of x instead of one read per 16 columns.
//   3. MFMAs; with one K slice the epilogue is applied directly.  With
//      several, each workgroup writes its partial tile to the scratch and a
//      second kernel sums the slices in slice order (deterministic) and
//      applies the epilogue.
template <int MT, int NT, int KSTEPS>
__global__ void __launch_bounds__(256)
    gemm_gemv_kernel(const float* __restrict__ x, const uint16_t* __restrict__ w,
                     const float* __restrict__ bias, int M, int N, int K, int ep,
                     float* __restrict__ out, float* __restrict__ partial) {
  constexpr int BN = 64 * NT;
  __shared__ __attribute__((aligned(16))) uint4 xs[2][MT * KSTEPS * 64];  // [hi|lo][frag][lane]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, grp = lane >> 4;
  const int n0 = blockIdx.x * BN;
  const int kslices = gridDim.y;
  const int k0 = blockIdx.y * KSTEPS * 32;
  const int nsteps = min(KSTEPS, (K - k0) >> 5);

  // Load order: the activation slice first, the weights last, so staging the
  // activations waits only for the L2-resident inputs while the weight stream
  // is still arriving (a wave's loads complete in issue order).
  // 1. activation slice fragments: fragment f = (mt, step), lane l holds row
  //    mt*16 + l%16, k = step*32 + (l/16)*8 .. +8.
  constexpr int FR = MT * KSTEPS * 64 / 256;  // fragments per thread
  static_assert(MT * KSTEPS * 64 % 256 == 0, "fragments must split evenly over the workgroup");
  // Every load below is unconditional (clamped address, value selected
  // afterwards), so the waits can count them in issue order.
  float4 xa[FR][2];
#pragma unroll
  for (int j = 0; j < FR; ++j) {
    const int idx = tid + j * 256;
    const int fl = idx & 63, f = idx >> 6;
    const int mt = f / KSTEPS, s2 = f - mt * KSTEPS;
    const int row = mt * 16 + (fl & 15);
    const int kk = k0 + min(s2, nsteps - 1) * 32 + (fl >> 4) * 8;
    const float* xp = x + (int64_t)min(row, M - 1) * K + kk;
    xa[j][0] = *reinterpret_cast<const float4*>(xp);
    xa[j][1] = *reinterpret_cast<const float4*>(xp + 4);
  }

  // 2. weight loads (clamped column and k-step: unconditional loads)
  //    in k-step order, so the MFMAs of step s wait only for its loads; lane
  //    (l16, grp) reads W[col][k .. k+8) of its column
  bf16x8 bw[KSTEPS][NT];
  const uint16_t* wrow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    wrow[nt] = w + (int64_t)min(n0 + (wave * NT + nt) * 16 + l16, N - 1) * K + k0 + grp * 8;
#pragma unroll
  for (int s2 = 0; s2 < KSTEPS; ++s2)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      bw[s2][nt] = __builtin_bit_cast(
          bf16x8, *reinterpret_cast<const uint4*>(wrow[nt] + min(s2, nsteps - 1) * 32));
  // nothing that waits for a load may be scheduled above this point
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int j = 0; j < FR; ++j) {
    const int idx = tid + j * 256;
    const int fl = idx & 63, f = idx >> 6;
    const int row = (f / KSTEPS) * 16 + (fl & 15);
    const bool live = row < M && (f % KSTEPS) < nsteps;
    float a[8] = {xa[j][0].x, xa[j][0].y, xa[j][0].z, xa[j][0].w,
                  xa[j][1].x, xa[j][1].y, xa[j][1].z, xa[j][1].w};
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = live ? a[e] : 0.f;
    uint4 hv, lv;
    split2_trunc(a[0], a[1], hv.x, lv.x);
    split2_trunc(a[2], a[3], hv.y, lv.y);
    split2_trunc(a[4], a[5], hv.z, lv.z);
    split2_trunc(a[6], a[7], hv.w, lv.w);
    xs[0][idx] = hv;
    xs[1][idx] = lv;
  }
  __syncthreads();

  // 3. MFMAs
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s2 = 0; s2 < KSTEPS; ++s2) {
    if (s2 < nsteps) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const bf16x8 ahi = __builtin_bit_cast(bf16x8, xs[0][(mt * KSTEPS + s2) * 64 + lane]);
        const bf16x8 alo = __builtin_bit_cast(bf16x8, xs[1][(mt * KSTEPS + s2) * 64 + lane]);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahi, bw[s2][nt], acc[mt][nt], 0, 0, 0);
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(alo, bw[s2][nt], acc[mt][nt], 0, 0, 0);
        }
      }
    }
  }

  // C fragment: acc[mt][nt][i] = C[mt*16 + 4*grp + i][n0 + (wave*NT + nt)*16 + l16]
  auto epilogue = [&](int row, int tile_col0, float v) {
    const int col = tile_col0 + l16;
    if (ep == (int)Epilogue::kSwiGLU) {
      const float u = __shfl_xor(v, 8);
      if (l16 < 8 && row < M && col < N)
        out[(int64_t)row * (N >> 1) + (tile_col0 >> 1) + l16] = v / (1.0f + __expf(-v)) * u;
    } else if (row < M && col < N) {
      float* op = out + (int64_t)row * N + col;
      if (ep == (int)Epilogue::kAccumulate)
        *op += v;
      else
        *op = bias ? v + bias[col] : v;
    }
  };
  if (kslices == 1) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          epilogue(mt * 16 + 4 * grp + i, n0 + (wave * NT + nt) * 16, acc[mt][nt][i]);
    return;
  }
  // Partial tile of this K slice: partial[slice][tile][row][BN], rows < 16*MT.
  // gemm_gemv_reduce_kernel sums the slices in order; the kernel boundary
  // orders the two.
  const int64_t tile_elems = (int64_t)MT * 16 * BN;
  float* mine = partial + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * tile_elems;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        mine[(mt * 16 + 4 * grp + i) * BN + (wave * NT + nt) * 16 + l16] = acc[mt][nt][i];
}

// Sums the K-slice partials of gemm_gemv_kernel in slice order and applies
// the epilogue.  One thread per (row, 16-column tile lane); SwiGLU pairs lanes
// 8 apart within a 16-column tile.
template <int MT, int NT>
__global__ void __launch_bounds__(256)
    gemm_gemv_reduce_kernel(const float* __restrict__ partial, int kslices, int n_tiles,
                            const float* __restrict__ bias, int M, int N, int ep,
                            float* __restrict__ out) {
  constexpr int BN = 64 * NT;
  const int64_t tile_elems = (int64_t)MT * 16 * BN;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // over n_tiles * M * BN
  const int64_t per_tile = (int64_t)M * BN;
  if (idx >= (int64_t)n_tiles * per_tile) return;  // whole 16-lane groups exit together
  const int tile = (int)(idx / per_tile);
  const int rem = (int)(idx - tile * per_tile);
  const int row = rem / BN, c = rem - row * BN;
  const int col = tile * BN + c;
  // The residual (accumulate) or bias (store) first, then the slices 8 (or
  // 24) at a time with every load of a group in flight, added in slice order (a slice
  // past the end adds +0, which leaves the sum unchanged).
  float pre = 0.f;
  if (col < N && ep == (int)Epilogue::kAccumulate)
    pre = out[(int64_t)row * N + col];
  else if (col < N && bias && ep == (int)Epilogue::kStore)
    pre = bias[col];
  const float* pp = partial + (int64_t)tile * tile_elems + row * BN + c;
  const int64_t slice_stride = (int64_t)n_tiles * tile_elems;
  float v = 0.f;
  auto sum_slices = [&](auto group) {
    constexpr int NG = decltype(group)::value;
    for (int ks0 = 0; ks0 < kslices; ks0 += NG) {
      float t[NG];
#pragma unroll
      for (int j = 0; j < NG; ++j)
        t[j] = ks0 + j < kslices ? pp[(ks0 + j) * slice_stride] : 0.f;
#pragma unroll
      for (int j = 0; j < NG; ++j) v += t[j];
    }
  };
  // up to 24 slices (config 4's down projection has 22) in one round of loads
  if (kslices > 8)
    sum_slices(std::integral_constant<int, 24>{});
  else
    sum_slices(std::integral_constant<int, 8>{});
  if (ep == (int)Epilogue::kSwiGLU) {
    const float u = __shfl_xor(v, 8);
    if ((c & 15) < 8 && col < N)
      out[(int64_t)row * (N >> 1) + ((col & ~15) >> 1) + (c & 7)] = v / (1.0f + __expf(-v)) * u;
  } else if (col < N) {
    out[(int64_t)row * N + col] =
        ep == (int)Epilogue::kAccumulate ? pre + v : bias ? v + pre : v;
  }
}

template <int MT, int NT, int UNR>
static void launch_skinny(int KW, dim3 grid, hipStream_t st, const float* x, const uint16_t* w,
                          const float* bias, int M, int N, int K, int ep, float* out) {
  switch (KW) {
    case 16:
      hipLaunchKernelGGL((gemm_skinny_kernel<MT, NT, 16, UNR>), grid, dim3(1024), 0, st, x, w,
                         bias, M, N, K, ep, out);
      break;
    case 8:
      hipLaunchKernelGGL((gemm_skinny_kernel<MT, NT, 8, UNR>), grid, dim3(512), 0, st, x, w,
                         bias, M, N, K, ep, out);
      break;
    case 4:
      hipLaunchKernelGGL((gemm_skinny_kernel<MT, NT, 4, UNR>), grid, dim3(256), 0, st, x, w,
                         bias, M, N, K, ep, out);
      break;
    default:
      hipLaunchKernelGGL((gemm_skinny_kernel<MT, NT, 1, UNR>), grid, dim3(64), 0, st, x, w,
                         bias, M, N, K, ep, out);
      break;
  }
}

namespace {
// Split-K GEMM geometry for few rows: NT x 64 columns per workgroup (BN) and
// KS k-steps of 32 per K slice; the slices are summed by
// gemm_gemv_reduce_kernel.  Few column tiles want narrow tiles (more
// workgroups).  Chosen per shape from M = 32 measurements:
//   N <= 4096, K <= 4096  NT 1, KS 8
//   N > 4096              NT 2, KS 8
//   K > 4096              NT 1, KS 8 (2048 x 5632: 704 workgroups at 3 per CU;
//     NT 2, KS 16 had 176 at one per CU, 0.6 us slower)
// ORION_GEMV_NT / ORION_GEMV_KS override every shape (measurement knobs; NT in
// {1, 2, 4}, KS in {4, 8, 16}).
int gemv_knob(const char* name, int a, int b, int c) {
  const char* e = getenv(name);
  const int v = e ? atoi(e) : 0;
  return (v == a || v == b || v == c) ? v : 0;
}
struct GemvShape {
  int mt, nt, ks, n_tiles, kslices;
  size_t ws_bytes;
};
GemvShape gemv_shape(int64_t M, int64_t N, int64_t K) {
  static const int knob_nt = gemv_knob("ORION_GEMV_NT", 1, 2, 4);
  static const int knob_ks = gemv_knob("ORION_GEMV_KS", 4, 8, 16);
  GemvShape g;
  g.mt = (int)((M + 15) / 16);
  g.nt = K <= 4096 && N > 4096 ? 2 : 1;
  g.ks = 8;
  if (knob_nt) g.nt = knob_nt;
  if (knob_ks) g.ks = knob_ks;
  g.n_tiles = (int)((N + 64 * g.nt - 1) / (64 * g.nt));
  g.kslices = (int)((K + g.ks * 32 - 1) / (g.ks * 32));
  g.ws_bytes = g.kslices > 1 ? (size_t)g.kslices * g.n_tiles * g.mt * 16 * 64 * g.nt * 4 : 0;
  return g;
}
template <int MT, int NT, int KS>
void launch_gemv_t(const GemvShape& g, hipStream_t st, const float* x, const uint16_t* w,
                   const float* bias, int M, int N, int K, int ep, float* out,
                   const GemmScratch* sc) {
  hipLaunchKernelGGL((gemm_gemv_kernel<MT, NT, KS>),
                     dim3((unsigned)g.n_tiles, (unsigned)g.kslices), dim3(256), 0, st, x, w, bias,
                     M, N, K, ep, out, sc ? sc->ws : nullptr);
  if (g.kslices > 1) {
    const int64_t threads = (int64_t)g.n_tiles * M * 64 * NT;
    hipLaunchKernelGGL((gemm_gemv_reduce_kernel<MT, NT>),
                       dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, sc->ws,
                       g.kslices, g.n_tiles, bias, M, N, ep, out);
  }
}
template <int MT, int NT>
void launch_gemv_nt(const GemvShape& g, hipStream_t st, const float* x, const uint16_t* w,
                    const float* bias, int M, int N, int K, int ep, float* out,
                    const GemmScratch* sc) {
  if (g.ks == 4)
    launch_gemv_t<MT, NT, 4>(g, st, x, w, bias, M, N, K, ep, out, sc);
  else if (g.ks == 16)
    launch_gemv_t<MT, NT, 16>(g, st, x, w, bias, M, N, K, ep, out, sc);
  else
    launch_gemv_t<MT, NT, 8>(g, st, x, w, bias, M, N, K, ep, out, sc);
}
template <int MT>
void launch_gemv(const GemvShape& g, hipStream_t st, const float* x, const uint16_t* w,
                 const float* bias, int M, int N, int K, int ep, float* out,
                 const GemmScratch* sc) {
  if (g.nt == 1)
    launch_gemv_nt<MT, 1>(g, st, x, w, bias, M, N, K, ep, out, sc);
  else if (g.nt == 4)
    launch_gemv_nt<MT, 4>(g, st, x, w, bias, M, N, K, ep, out, sc);
  else
    launch_gemv_nt<MT, 2>(g, st, x, w, bias, M, N, K, ep, out, sc);
}
}  // namespace

// K splits of the LDS-tiled GEMM.  A call with fewer output tiles than CUs
// leaves CUs idle, so its K is split until the tiles x splits reach
// kTiledFill workgroups, up to 8 splits of at least 16 k-steps each; the
// splits' raw sums go to the scratch and gemm_tiled_reduce_kernel adds them.
// (Measured on config 5: the 16-tile LM head went 108 -> 28 us with 4
// splits; splitting the 504-tile O and down projections saved about what
// their 31 us reduce launches cost, so they stay whole.)  Not for the SwiGLU
// epilogue (its column pairs sit in one tile).  ORION_GEMM_TILED_SPLIT=n
// forces n (measurement knob, read per call).
// A long K (>= 256 k-steps) with fewer tiles than the resident slots (3
// workgroups x 256 CUs) is also split, into up to 2 x slots workgroups of at
// least 64 k-steps: config 5's down projection (K 18944, 504 tiles) went
// 664-697 -> 585 us + a 37 us reduce with 3 splits, while shorter-K calls
// with the same tile count (QKV, O) gained nothing.  These long-K splits are
// preferred, not required: a caller whose scratch cannot hold them (the
// no-allocation entry point) runs the required count.
namespace {
constexpr int64_t kTiledFill = 256;
constexpr int64_t kTiledSlots = 768;
constexpr int64_t kTM = 128;  // rows of a tile, for the counts below
int tiled_ksplits(int64_t M, int64_t N, int64_t K, bool preferred = true) {
  const int64_t tiles = ((N + kTN - 1) / kTN) * ((M + kTM - 1) / kTM);
  const int64_t ksteps = K / kTK;
  if (const char* e = getenv("ORION_GEMM_TILED_SPLIT")) {
    const int64_t f = atoll(e);
    return (int)std::max<int64_t>(1, std::min<int64_t>(f, std::max<int64_t>(1, ksteps / 4)));
  }
  int s = 1;
  while (s < 8 && tiles * s < kTiledFill && ksteps / (2 * s) >= 16) s *= 2;
  if (preferred && tiles < kTiledSlots && ksteps >= 256) {
    int64_t p = std::min<int64_t>(8, 2 * kTiledSlots / tiles);
    while (p > 1 && ksteps / p < 64) --p;
    s = std::max<int>(s, (int)p);
  }
  return s;
}

// Workgroup tiles of the LDS-tiled GEMM: 32 mtw rows x 32 ntw columns, st
// k-steps in LDS, `per_cu` workgroups resident (LDS and registers; the form with
// RoPE also holds its rows' slots, tiled_resident).  Up to
// kShapeRows rows the grid is a few workgroups per CU, and what a GEMM takes is
// its k-steps in a row times what one costs: `alone` us where the CU holds one
// workgroup (latency; with two k-steps in LDS one copy is in flight, and it
// is waited for) or `each` us per resident one where they fill the matrix cores;
// [0] for activations that arrive split, [1] for f32 ones, which the kernel splits.
// Fitted to every shape in 1 to 8 splits on 16 N x K of layers and heads (520 x
// 1056 to 37888 x 3584, 65 to 1024 rows), weights not in a cache, as a forward
// finds them; 14 others (704 x 2080 to 128256 x 4096) were kept to check it.
// There the estimate is within 10 % of 92 in 100 of the times that matter (up to
// 1.25 x the fastest), and what it chooses is 1.3 % slower than the fastest on
// average, at most 9 % in 95 of 100.
struct TiledShape {
  int ntw, mtw, st, per_cu;
  float alone[2], each[2];
};
constexpr TiledShape kTiledShapes[] = {
    {4, 4, 2, 3, {0.686f, 0.715f}, {0.431f, 0.512f}},
    {4, 4, 3, 2, {0.509f, 0.707f}, {0.423f, 0.538f}},
    {4, 3, 2, 4, {0.728f, 0.623f}, {0.317f, 0.397f}},
    {4, 3, 3, 2, {0.428f, 0.589f}, {0.332f, 0.445f}},
    {4, 2, 4, 2, {0.293f, 0.398f}, {0.247f, 0.305f}},
    {4, 5, 3, 1, {0.620f, 0.895f}, {0.675f, 0.962f}},
    {8, 4, 2, 2, {0.910f, 1.092f}, {0.782f, 0.885f}},
};
// the shape that batches past kShapeRows rows take, by their columns
constexpr const TiledShape& kTiledUsual = kTiledShapes[0];
constexpr const TiledShape& kTiledWide = kTiledShapes[6];
constexpr int64_t kShapeRows = 1024;
constexpr int kCus = 256;
constexpr int kLdsBytes = 160 * 1024;

// Workgroups of shape t that a CU holds.
constexpr int tiled_resident(const TiledShape& t, bool rope) {
  const int lds = t.st * (32 * t.mtw * kTK * 4 + 32 * t.ntw * kTK * 2) +
                  (rope ? 32 * t.mtw * (int)sizeof(RowSlot) : 0);
  return std::min(t.per_cu, kLdsBytes / lds);
}
constexpr bool lds_holds_per_cu() {
  for (const TiledShape& t : kTiledShapes)
    if (tiled_resident(t, false) != t.per_cu) return false;
  return true;
}
static_assert(lds_holds_per_cu(), "the table's workgroups per CU fit its LDS");
// 96 rows x 2 k-steps fill the LDS exactly; with the slots one less fits
static_assert(tiled_resident(kTiledShapes[2], true) == 3, "four without the slots");

// Microseconds of a GEMM on shape t in `splits` K splits: rounds of resident
// workgroups (the last of them counts less the fewer CUs have it: the others
// leave it their share of the L2 and of memory), the launch, and the sums' round
// trip at 3.9 TB/s.
float tiled_cost(const TiledShape& t, int64_t M, int64_t N, int64_t K, int splits, bool f32_x,
                 bool rope) {
  const int per_cu = tiled_resident(t, rope);
  const float alone = t.alone[f32_x], each = t.each[f32_x];
  const int64_t wgs = ((M + 32 * t.mtw - 1) / (32 * t.mtw)) * ((N + 32 * t.ntw - 1) / (32 * t.ntw)) * splits;
  const int64_t per = (wgs + kCus - 1) / kCus, whole = (per - 1) / per_cu;
  const float idle = (float)(per * kCus - wgs) / kCus, last = (float)(per - whole * per_cu) - 0.3f * idle;
  const float kspan = (float)((K / kTK + splits - 1) / splits);
  const float us = ((float)whole * std::max(alone, per_cu * each) + std::max(alone, last * each)) * kspan +
                   0.41f * (float)(whole + 1) + 7.1f;
  return us + (splits > 1 ? (splits + 1) * (float)(M * N) * 4e-6f / 3.9f : 0.f);
}

struct TiledPlan {
  TiledShape shape;
  int splits;
  float us;  // (up to kShapeRows rows)
};
// `splits` > 0: with that many.  Otherwise 1, 2, 4 or 8 of at least 16 k-steps
// where the call can take several.  f32_x: x does not arrive split.  `rope`: the
// QKV GEMM with RoPE, one split.
TiledPlan tiled_plan(int64_t M, int64_t N, int64_t K, Epilogue ep, int splits, bool f32_x,
                     bool rope = false) {
  // 128 x 256 workgroup tiles (64 x 128 per wave, 2 workgroups per CU) for
  // wide outputs: per MFMA a third less LDS traffic (copies + fragment
  // reads) than 128 x 128 tiles at 3 per CU.  Measured at config 4's prefill
  // shapes: gate/up (N 11264) 649-673 -> 692-700 TFLOP/s; QKV (2560) even,
  // down (2048) -3 %, O (2048) -13 % (too few tiles for 2 per CU).
  // ORION_GEMM_WIDE=0/1 forces the choice (measurement knob, read per call).
  const char* wide_env = getenv("ORION_GEMM_WIDE");
  const bool can_split = ep != Epilogue::kSwiGLU;
  const TiledShape& usual = (wide_env ? wide_env[0] == '1' : N >= 8192) ? kTiledWide : kTiledUsual;
  const int usual_splits = !can_split ? 1 : splits ? splits : tiled_ksplits(M, N, K);
  TiledPlan best{usual, usual_splits, 0.f};
  if (wide_env || M > kShapeRows) return best;
  if (can_split && !splits && getenv("ORION_GEMM_TILED_SPLIT")) splits = usual_splits;
  // Up to kShapeRows rows the usual shape stays unless another is estimated 5 %
  // faster, about what the estimate is off by: of the 1425 calls above 10 are then
  // more than 3 % slower than on the usual shape (without the margin 36), and all
  // take 0.82 of its time on average.
  best.us = tiled_cost(usual, M, N, K, usual_splits, f32_x, rope);
  float least = 0.95f * best.us;
  for (const TiledShape& t : kTiledShapes)
    for (int s = 1; s <= 8; s *= 2) {
      const int n = !can_split ? 1 : splits ? splits : s;
      if (n > 1 && !splits && K / kTK / n < 16) break;
      const float us = tiled_cost(t, M, N, K, n, f32_x, rope);
      if (us < least) {
        best = {t, n, us};
        least = us;
      }
      if (n != s) break;
    }
  return best;
}
}  // namespace

bool gemm_takes_rope(int64_t M, int64_t N, int64_t K, int64_t head_dim) {
  if (head_dim % 32 != 0) return false;
  const TiledPlan best = tiled_plan(M, N, K, Epilogue::kStore, 0, false);
  if (best.splits == 1 || M > kShapeRows || getenv("ORION_GEMM_TILED_SPLIT")) return best.splits == 1;
  // unsplit, with an epilogue that takes longer, and without RoPE's launch: a read
  // and a write of the matrix (over 65 to 1024 rows of 2560 x 2048 to 10240 x
  // 8192, 0.3 % slower on average than always taking the faster of the two)
  const float saved = 1.f + (float)(M * N) * 8e-6f / 6.f;
  return tiled_plan(M, N, K, Epilogue::kStore, 1, false, true).us < best.us + saved;
}

void gemm_scratch_need(int64_t M, int64_t N, int64_t K, size_t* ws_bytes, bool packed,
                       bool preferred) {
  *ws_bytes = 0;
  if (M < 1 || K % 32 != 0) return;
  if (M > 64) {
    const int s = preferred ? tiled_plan(M, N, K, Epilogue::kStore, 0, !packed).splits
                            : tiled_ksplits(M, N, K, false);
    if (s > 1) *ws_bytes = (size_t)s * (size_t)M * (size_t)N * sizeof(float);
    return;
  }
  *ws_bytes = gemv_shape(M, N, K).ws_bytes;
}

hipError_t launch_gemm(hipStream_t st, const float* x, const uint16_t* w, const float* bias,
                       int64_t M, int64_t N, int64_t K, Epilogue ep, float* out,
                       const GemmScratch* scratch, const GemmFuse* fuse) {
  const GemmFuse f = fuse ? *fuse : GemmFuse{};
  if (M == 0 || N == 0) return hipSuccess;
  if (K % 32 != 0 || K == 0) return hipErrorInvalidValue;
  if (ep == Epilogue::kSwiGLU && N % 16 != 0) return hipErrorInvalidValue;
  // ORION_GEMM_TILED_MIN_M: smallest M that takes the LDS-tiled kernel.
  static const int64_t tiled_min_m = [] {
    const char* e = getenv("ORION_GEMM_TILED_MIN_M");
    return e ? (int64_t)atoll(e) : (int64_t)256;
  }();
  // split-layout activations exist only for the LDS-tiled kernel
  if ((f.x_hilo || f.out_hilo) && (M <= 64 || (M < tiled_min_m && !f.w_packed)))
    return hipErrorInvalidValue;
  // Few rows: split-K weight streaming (needs the scratch when K spans
  // several slices).
  if (M <= 64 && !f.w_packed && N <= INT32_MAX && K <= INT32_MAX) {
    const GemvShape g = gemv_shape(M, N, K);
    const bool fits = g.kslices == 1 || (scratch && scratch->ws_bytes >= g.ws_bytes);
    if (fits && g.kslices <= 65535) {
      const int m = (int)M, n = (int)N, k = (int)K, e = (int)ep;
      switch (g.mt) {
        case 1: launch_gemv<1>(g, st, x, w, bias, m, n, k, e, out, scratch); break;
        case 2: launch_gemv<2>(g, st, x, w, bias, m, n, k, e, out, scratch); break;
        case 3: launch_gemv<3>(g, st, x, w, bias, m, n, k, e, out, scratch); break;
        default: launch_gemv<4>(g, st, x, w, bias, m, n, k, e, out, scratch); break;
      }
      return hipGetLastError();
    }
  }
  // The LDS-tiled kernel takes every larger M, and every M > 64 when only the
  // packed copy exists (the skinny kernel reads row-major W).
  if (M >= tiled_min_m || f.w_packed) {
    if (M > (int64_t)65535 * kTM || N > INT32_MAX || K > INT32_MAX) return hipErrorInvalidValue;
    PackedGeom pk;
    pk.packed = f.w_packed != nullptr;
    if (pk.packed) {
      if (f.pair_dim && ep != Epilogue::kStore) return hipErrorInvalidValue;
      pk.pair_dim = (int)f.pair_dim;
      pk.pair_cols = (int)f.pair_cols;
    }
    // Shape and K splits (tiled_plan), when the scratch holds their sums
    const size_t avail = scratch ? scratch->ws_bytes : 0;
    auto fits = [&](int s) {
      return s == 1 || (size_t)s * (size_t)M * (size_t)N * sizeof(float) <= avail;
    };
    // (a forward's K splits are those of split activations, whichever kernel
    // splits them: its sums are the same)
    const bool f32_x = !f.x_hilo;
    const int want = f.rope || f.unsplit ? 1 : f32_x && pk.packed ? tiled_plan(M, N, K, ep, 0, false).splits : 0;
    TiledPlan plan = tiled_plan(M, N, K, ep, want, f32_x, f.rope != nullptr);
    if (!fits(plan.splits)) plan = tiled_plan(M, N, K, ep, tiled_ksplits(M, N, K, false), f32_x);
    if (!fits(plan.splits)) plan = tiled_plan(M, N, K, ep, 1, f32_x);
    // ORION_GEMM_ACT=bf16 rounds the activations to bf16 (one MFMA per
    // fragment) instead of the hi/lo pair (measurement knob, read per call).
    const char* act = getenv("ORION_GEMM_ACT");
    const bool hilo = !(act && act[0] == 'b');
    if (f.x_hilo && !hilo) return hipErrorInvalidValue;
    if (f.rope && (!f.x_hilo || !pk.packed || ep != Epilogue::kStore || pk.pair_dim % 32 != 0 ||
                   pk.pair_dim < 32))
      return hipErrorInvalidValue;
    if (!hilo && plan.shape.ntw == 4) plan.shape = kTiledUsual;
    const int tn = 32 * plan.shape.ntw, tm = 32 * plan.shape.mtw;
    int splits = plan.splits;
    dim3 grid((unsigned)((N + tn - 1) / tn), (unsigned)((M + tm - 1) / tm));
    // XCD-aware grouped tile order with groups of 4 m tiles (measured at the
    // config-4 prefill shapes against the row-major grid: QKV 529 -> 563, O
    // 405 -> 443, down 513 -> 536 TFLOP/s, gate/up unchanged; groups of 8 and
    // 16 gained less).  ORION_GEMM_GM=g overrides the group (0: the 2D
    // row-major grid; measurement knob, read per call).
    int gm = 4;
    if (const char* e = getenv("ORION_GEMM_GM")) gm = std::max(0, atoi(e));
    if (gm > 0) {
      const int64_t total = (int64_t)grid.x * grid.y;
      grid = dim3((unsigned)(((total + 7) / 8) * 8), 1);
    }
    const int ksteps = (int)(K / kTK), kspan = (ksteps + splits - 1) / splits;
    // every split must start below K: with kspan rounded up, ceil(ksteps /
    // kspan) splits cover K (a forced count such as 16 splits of 66 k-steps
    // would otherwise leave splits 14 and 15 starting past the last row)
    splits = (ksteps + kspan - 1) / kspan;
    grid.z = (unsigned)splits;
    float* partial = splits > 1 ? scratch->ws : nullptr;
    auto launch = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, x, f.w_packed ? f.w_packed : w, bias,
                         (int)M, (int)N, (int)K, (int)ep, out, pk, gm, kspan, partial,
                         f.out_hilo && ep == Epilogue::kSwiGLU, f.rope ? *f.rope : RopeOut{});
      return hipGetLastError();
    };
    auto hilo_shape = [&](auto xs, auto rope) {
      constexpr bool X = decltype(xs)::value, R = decltype(rope)::value;
      const TiledShape& t = plan.shape;
      if (t.ntw == 8) return launch(gemm_tiled_kernel<true, 8, X, 4, 2, R>);
      switch (t.mtw * 10 + t.st) {
        case 24: return launch(gemm_tiled_kernel<true, 4, X, 2, 4, R>);
        case 32: return launch(gemm_tiled_kernel<true, 4, X, 3, 2, R>);
        case 33: return launch(gemm_tiled_kernel<true, 4, X, 3, 3, R>);
        case 43: return launch(gemm_tiled_kernel<true, 4, X, 4, 3, R>);
        case 53: return launch(gemm_tiled_kernel<true, 4, X, 5, 3, R>);
        default: return launch(gemm_tiled_kernel<true, 4, X, 4, 2, R>);
      }
    };
    using Yes = std::true_type;
    using No = std::false_type;
    const hipError_t err =
        !hilo ? (plan.shape.ntw == 8 ? launch(gemm_tiled_kernel<false, 8>)
                                     : launch(gemm_tiled_kernel<false, 4>))
        : f.rope   ? hilo_shape(Yes{}, Yes{})
        : f.x_hilo ? hilo_shape(Yes{}, No{})
                   : hilo_shape(No{}, No{});
    if (err != hipSuccess) return err;
    if (splits > 1) {
      const int64_t total = M * N;
      const unsigned blocks = (unsigned)std::min<int64_t>((total + 255) / 256, 8192);
      hipLaunchKernelGGL(gemm_tiled_reduce_kernel, dim3(blocks), dim3(256), 0, st, partial,
                         splits, M, N, bias, (int)ep, out);
    }
    return hipGetLastError();
  }
  // Rows per tile (MT x 16) and columns per tile (NT x 16): wide column tiles
  // only when there are many of them.  Waves per tile (KW, splitting K): as
  // many as it takes for each wave's whole k-range (<= UNR steps of 32) to be
  // in flight in one round, up to 16; the LDS reduction buffer
  // KW x 16MT x (16NT+1) floats stays <= 64 KiB.
  const int MT = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int NT = (MT <= 2 && N >= 8192) ? 4 : (N > 4096 ? 2 : 1);
  constexpr int UNR = 4;
  const int64_t ksteps = K / 32;
  const int kw_cap = (MT * NT <= 4) ? 16 : 8;
  int KW = 1;
  while (KW < kw_cap && (ksteps + KW - 1) / KW > UNR) KW <<= 1;
  if (KW == 2) KW = 4;
  const int BN = 16 * NT, BM = 16 * MT;
  dim3 grid((unsigned)((N + BN - 1) / BN), (unsigned)((M + BM - 1) / BM));
  const int m = (int)M, n = (int)N, k = (int)K, e = (int)ep;
  if (MT == 1) {
    if (NT == 4) launch_skinny<1, 4, UNR>(KW, grid, st, x, w, bias, m, n, k, e, out);
    else if (NT == 2) launch_skinny<1, 2, UNR>(KW, grid, st, x, w, bias, m, n, k, e, out);
    else launch_skinny<1, 1, UNR>(KW, grid, st, x, w, bias, m, n, k, e, out);
  } else if (MT == 2) {
    if (NT == 4) launch_skinny<2, 4, UNR>(KW, grid, st, x, w, bias, m, n, k, e, out);
    else if (NT == 2) launch_skinny<2, 2, UNR>(KW, grid, st, x, w, bias, m, n, k, e, out);
    else launch_skinny<2, 1, UNR>(KW, grid, st, x, w, bias, m, n, k, e, out);
  } else {
    if (NT == 2) launch_skinny<4, 2, UNR>(KW, grid, st, x, w, bias, m, n, k, e, out);
    else launch_skinny<4, 1, UNR>(KW, grid, st, x, w, bias, m, n, k, e, out);
  }
  return hipGetLastError();
}

}  // namespace orion
