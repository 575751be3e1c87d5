// f32 GEMV  y[n] = sum_k A[k][n] * x[k],  A is K x N row-major (trueno-gpu/src/kernels/gemv.rs: GemvKernel
// "gemv_warp_reduce" :21-166, CoalescedGemvKernel "gemv_coalesced" :188-398; both compute this product, in
// different summation orders).  Bound by HBM: 4 K N bytes of A read once.
//
// A lane owns four neighbouring columns, so a wave reads 1 KB of a row of A with one 128-bit load per lane, and
// the 8 waves of a workgroup take every eighth row of the workgroup's part of K (eight rows in flight per
// wave).  x[k] is the same for the whole wave: it comes through the scalar cache.  The waves' sums meet in LDS
// in wave order.  K is cut in parts over the grid so that a workgroup per CU exists and no more (up to two for matrices of
// more than 32768 columns, whose tiles alone do not divide well among the CUs): one in flight per CU reads
// whole lines at 6.3 TB/s, two at 5.0 (K x N; 4096 x 11008, 180 MB: 36.3 -> 28.7 us; 4096 x 4096 18.3 -> 15.3, 5000 x 3000
// 20.0 -> 16.0, 1000 x 14336 14.0 -> 12.2, 14336 x 4000 37.9 -> 36.2).  With several parts every part
// stores its partial y through to memory and the workgroup that arrives last at the column tile's counter adds
// the parts in part order and puts the counter back to zero - one launch, the same bits on every run.
//
// Columns that are no multiple of four, or buffers that do not begin at 16 bytes, take the same kernel with loads and stores at
// multiples of four bytes (kRagged; fewer than four columns: kNarrow, a lane with all of them).  A row then spans a line more and lines are
// shared between tiles, so these loads may stay in the caches.  Bound like the aligned form: 3778 x 3245 13.5 us beside
// 12.6 for 3597 x 3220, where a thread per column (k in order, a round trip to memory for every few rows) took 1278; 4853 x 1202
// 1131 -> 10.0, 577 x 595 118 -> 4.0.
#pragma once
#include "kquant_common.hip.h"

namespace gemv_f32 {

constexpr u32 kWaves = 8, kUnroll = 8, kTileCols = 256, kTailParts = 16;

enum Form { kAligned, kRagged, kNarrow };

struct __attribute__((packed, aligned(4))) Quad { f32x4 v; };      // four floats at any multiple of four bytes

// A lane's four columns of one row, read past the caches that a matrix read once would only sweep.
template <Form F>
__device__ __forceinline__ f32x4 load_quad(const float* p, u32 n_dim) {
  if constexpr (F == kAligned) return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
  if constexpr (F == kRagged) return reinterpret_cast<const Quad*>(p)->v;
  return f32x4{p[0], p[min(1u, n_dim - 1u)], p[n_dim - 1u], 0.0f};
}

template <Form F>
__device__ __forceinline__ void store_quad(float* p, f32x4 v, u32 n_dim) {
  if constexpr (F == kAligned) *reinterpret_cast<f32x4*>(p) = v;
  if constexpr (F == kRagged) reinterpret_cast<Quad*>(p)->v = v;
  if constexpr (F == kNarrow) {
    p[0] = v.x;
    if (n_dim > 1u) p[1] = v.y;
    if (n_dim > 2u) p[2] = v.z;
  }
}

template <Form F>
__device__ __forceinline__ void body(float* __restrict__ y, const float* __restrict__ a, const float* __restrict__ x,
                                          float* __restrict__ partial, u32* __restrict__ counters, u32 k_dim, u32 n_dim,
                                          u32 rows_per_part, u32 parts) {
  __shared__ f32x4 s_sum[kWaves][64];
  __shared__ u32 s_old;
  const u32 lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const u32 tile = blockIdx.x / parts, part = blockIdx.x - tile * parts;
  const u32 col = tile * kTileCols + 4u * lane;
  const bool col_ok = col < n_dim;
  // kAligned: a lane's four columns are all in or all out.  kRagged (n_dim >= 4): the last lane's columns move back so that
  // they end with the row; it and its neighbour then hold some columns twice, with the same bits.
  const u32 first = !col_ok || F == kNarrow ? 0u : F == kRagged ? min(col, n_dim - 4u) : col;
  const u32 k0 = part * rows_per_part, k1 = min(k_dim, k0 + rows_per_part);
  const float* ap = a + first;
  const u32 np = (n_dim + 3u) & ~3u;                       // columns of a part's results
  const __amdgpu_buffer_rsrc_t part_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      partial, 0, static_cast<int>(min(static_cast<size_t>(0x7FFFFFFF), static_cast<size_t>(parts) * np * 4u)), 0x00020000);
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  u32 k = k0 + wave;
  for (; k + (kUnroll - 1u) * kWaves < k1; k += kUnroll * kWaves) {
    f32x4 v[kUnroll];
    float xv[kUnroll];
#pragma unroll
    for (u32 u = 0; u < kUnroll; ++u) {
      v[u] = load_quad<F>(ap + static_cast<size_t>(k + u * kWaves) * n_dim, n_dim);
      xv[u] = x[k + u * kWaves];
    }
    f32x4 t = v[0] * xv[0];      // eight rows by themselves first: one rounding in eight at the size of the whole
#pragma unroll
    for (u32 u = 1; u < kUnroll; ++u) {
      t.x = fmaf(v[u].x, xv[u], t.x); t.y = fmaf(v[u].y, xv[u], t.y);
      t.z = fmaf(v[u].z, xv[u], t.z); t.w = fmaf(v[u].w, xv[u], t.w);
    }
    acc += t;
  }
  if (k < k1) {      // the last rows, together as well: one by one each would cost a round trip to memory
    f32x4 v[kUnroll];
    float xv[kUnroll];
#pragma unroll
    for (u32 u = 0; u < kUnroll; ++u) {
      const u32 row = min(k + u * kWaves, k1 - 1u);
      v[u] = load_quad<F>(ap + static_cast<size_t>(row) * n_dim, n_dim);
      xv[u] = x[row];
    }
    f32x4 t = v[0] * xv[0];
#pragma unroll
    for (u32 u = 1; u < kUnroll; ++u)
      if (k + u * kWaves < k1) {
        t.x = fmaf(v[u].x, xv[u], t.x); t.y = fmaf(v[u].y, xv[u], t.y);
        t.z = fmaf(v[u].z, xv[u], t.z); t.w = fmaf(v[u].w, xv[u], t.w);
      }
    acc += t;
  }
  s_sum[wave][lane] = acc;
  __syncthreads();
  if (wave != 0u) {
    if (parts == 1u) return;
  } else {
    for (u32 w = 1; w < kWaves; ++w) {
      const f32x4 o = s_sum[w][lane];
      acc.x += o.x; acc.y += o.y; acc.z += o.z; acc.w += o.w;
    }
    if (parts == 1u) {
      if (col_ok) store_quad<F>(y + first, acc, n_dim);
      return;
    }
    if (col_ok)      // across workgroups (and XCDs): one 16-byte buffer store at agent scope (sc1)
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(acc.x), __float_as_uint(acc.y), __float_as_uint(acc.z), __float_as_uint(acc.w)},
                                             part_rsrc, static_cast<int>((part * np + col) * 4u), 0, 16);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the coherent stores have been acknowledged
    if (lane == 0u) {
      const u32 old = __hip_atomic_fetch_add(counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (old == parts - 1u) __hip_atomic_store(counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_old = old;
    }
  }
  __syncthreads();
  if (s_old != parts - 1u) return;
  // The last workgroup to arrive adds the parts: sixteen of them a wave and round, all in flight, in part order, and then the waves' sums
  // in wave order.  (One wave for all took a round trip to memory for every
  // sixteen: 52 parts, 3968 x 1068, 11.2 us and 9.2 so.)
  f32x4 r = {0.0f, 0.0f, 0.0f, 0.0f};
  if (col_ok)
    for (u32 p0 = wave * kTailParts; p0 < parts; p0 += kWaves * kTailParts) {
      u32x4 got[kTailParts];
#pragma unroll
      for (u32 pp = 0; pp < kTailParts; ++pp)
        got[pp] = __builtin_amdgcn_raw_buffer_load_b128(part_rsrc, static_cast<int>((min(p0 + pp, parts - 1u) * np + col) * 4u), 0, 16);
#pragma unroll
      for (u32 pp = 0; pp < kTailParts; ++pp)
        if (p0 + pp < parts) {
          r.x += __uint_as_float(got[pp].x); r.y += __uint_as_float(got[pp].y);
          r.z += __uint_as_float(got[pp].z); r.w += __uint_as_float(got[pp].w);
        }
    }
  if (parts > kTailParts) {
    s_sum[wave][lane] = r;                                 // (wave 0 read the waves' sums before the last barrier)
    __syncthreads();
    if (wave == 0u)
      for (u32 w = 1; w < min(kWaves, (parts + kTailParts - 1u) / kTailParts); ++w) {
        const f32x4 o = s_sum[w][lane];
        r.x += o.x; r.y += o.y; r.z += o.z; r.w += o.w;
      }
  }
  if (wave == 0u && col_ok) store_quad<F>(y + first, r, n_dim);
}

// The named kernels' plain form: a thread per column, k in order (the summation order of the reference's gemv_coalesced).  The
// launcher takes it only for k = 0 and for rows of 2^31 columns and more.
__device__ __forceinline__ void generic_body(float* __restrict__ y, const float* __restrict__ a, const float* __restrict__ x,
                                             u32 k_dim, u32 n_dim) {
  const u32 col = blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= n_dim) return;
  float sum = 0.0f;
  for (u32 k = 0; k < k_dim; ++k) sum = fmaf(x[k], a[static_cast<size_t>(k) * n_dim + col], sum);
  y[col] = sum;
}

}  // namespace gemv_f32
