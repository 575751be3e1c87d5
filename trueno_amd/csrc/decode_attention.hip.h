// Single-query attention over a KV cache for autoregressive decoding (trueno-gpu/src/kernels/attention.rs:808-1095,
// IncrementalAttentionKernel, kernel name "incremental_attention"):
//   out[h][:] = sum_i softmax_i(scale * q[h] . k[kv(h)][i]) * v[kv(h)][i],  i < seq_len,  kv(h) = h * num_kv_heads / num_heads
//   q, out: [num_heads][head_dim];  k, v: [num_kv_heads][max_seq_len][head_dim];  f32.
// The reference walks the positions one by one in a single warp per head with an online softmax (Milakov &
// Gimelshein) and two elements per lane, which covers head_dim <= 64; this kernel computes the same function for
// head_dim up to 256.  Bound by HBM: K and V are read once, 8 * num_kv_heads * seq_len * head_dim bytes.
//
// A position's row of K (and of V) is read by head_dim/4 lanes with one 128-bit load each, so a wave takes
// 64 / (head_dim/4) positions at a time; each such lane group keeps its own running (max, sum, output) over the
// positions it sees.  The positions of a head are cut in chunks over the grid and a chunk over the 4 waves of a
// workgroup; groups, waves and chunks are merged with the usual rescaling, the chunks through memory by the
// workgroup that arrives last at the head's counter (in chunk order: the same bits on every run).  Exponentials
// are 2^x on scores pre-multiplied by log2(e), as in the reference (ex2.approx there, v_exp_f32 here).
#pragma once
#include "kquant_common.hip.h"
#include <type_traits>

namespace decode_attention {

constexpr u32 kWaves = 4;
constexpr float kLog2e = 1.4426950408889634f;

struct State {          // running softmax over some positions, in the 2^x domain
  float m, s;
  f32x4 o;
};

__device__ __forceinline__ void merge(State& a, float m, float s, const f32x4& o) {
  // one of the two factors is always 1: a single exponential, of (smaller maximum - larger maximum)
  const bool keep = a.m >= m;
  const float nm = keep ? a.m : m, other = keep ? m : a.m;
  const float e = other == nm ? 1.0f : __builtin_amdgcn_exp2f(other - nm);  // -inf - -inf never reaches exp2
  const float ca = keep ? 1.0f : e, cb = keep ? e : 1.0f;
  a.s = a.s * ca + s * cb;
  a.o.x = a.o.x * ca + o.x * cb; a.o.y = a.o.y * ca + o.y * cb;
  a.o.z = a.o.z * ca + o.z * cb; a.o.w = a.o.w * ca + o.w * cb;
  a.m = nm;
}

// Sum of v over each group of 2^lpp_log2 neighbouring lanes, in every lane of the group, without going through LDS
// (five dependent ds_bpermute per position cost more than the position's memory traffic): DPP within a row of 16
// lanes, row sums through SGPRs beyond that.
__device__ __forceinline__ float group_sum(float v, u32 lpp_log2, u32 lane) {
  if (lpp_log2 >= 1u) v += dpp_f32<0xB1>(v);    // quad_perm [1,0,3,2]
  if (lpp_log2 >= 2u) v += dpp_f32<0x4E>(v);    // quad_perm [2,3,0,1]
  if (lpp_log2 >= 3u) v += dpp_f32<0x141>(v);   // row_half_mirror
  if (lpp_log2 >= 4u) v += dpp_f32<0x140>(v);   // row_mirror: every lane of a row of 16 holds the row's sum
  if (lpp_log2 >= 5u) {
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    const float lo = r0 + r1, hi = r2 + r3;
    v = lpp_log2 >= 6u ? lo + hi : (lane < 32u ? lo : hi);
  }
  return v;
}

// lanes per position LPP = 2^lpp_log2 >= head_dim / 4
__device__ __forceinline__ void body(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                                     float* __restrict__ out, u32 seq_len, u32 head_dim, u32 num_heads, u32 num_kv_heads,
                                     u32 max_seq_len, float scale, u32 lpp_log2, u32 chunk, u32 chunks,
                                     float* __restrict__ partial, u32* __restrict__ counters) {
  __shared__ float s_m[kWaves][64], s_s[kWaves][64];
  __shared__ f32x4 s_o[kWaves][64];
  __shared__ u32 s_old;
  const u32 lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const u32 head = blockIdx.x / chunks, ci = blockIdx.x - head * chunks;
  const u32 kv_head = static_cast<u32>((static_cast<uint64_t>(head) * num_kv_heads) / num_heads);
  const u32 lpp = 1u << lpp_log2, ppw = 64u >> lpp_log2;           // lanes per position, positions per wave and step
  const u32 sub = lane & (lpp - 1u), grp = lane >> lpp_log2;
  const bool live = 4u * sub < head_dim;                             // head_dim % 4 == 0
  const size_t kv_base = static_cast<size_t>(kv_head) * max_seq_len * head_dim;
  const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  // the chunks' states cross workgroups (and XCDs): 16-byte buffer accesses at agent scope (sc1)
  const __amdgpu_buffer_rsrc_t part_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(partial, 0, static_cast<int>(min(static_cast<size_t>(0x7FFFFFFF), static_cast<size_t>(num_heads) * chunks * lpp * 32u)), 0x00020000);
  const f32x4 qv = live ? reinterpret_cast<const f32x4*>(q + static_cast<size_t>(head) * head_dim)[sub] : zero4;
  const float sl = scale * kLog2e;
  const u32 p0 = ci * chunk, p1 = min(seq_len, p0 + chunk);
  State st = {-INFINITY, 0.0f, zero4};
  constexpr u32 kAhead = 4;                     // positions per lane group whose rows are in flight together
  const u32 stride = kWaves * ppw;
  for (u32 p = p0 + wave * ppw + grp; p < p1; p += kAhead * stride) {
    f32x4 kk[kAhead], vv[kAhead];
#pragma unroll
    for (u32 a = 0; a < kAhead; ++a) {
      const u32 pa = min(p + a * stride, p1 - 1u);          // clamped: read, then ignored
      const size_t row = kv_base + static_cast<size_t>(pa) * head_dim;
      // (the cache is read once per call, a row in whole lines: the non-temporal hint is worth 3-11 % here)
      kk[a] = live ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(k + row) + sub) : zero4;
      vv[a] = live ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(v + row) + sub) : zero4;
    }
#pragma unroll
    for (u32 a = 0; a < kAhead; ++a) {
      float d = fmaf(qv.w, kk[a].w, fmaf(qv.z, kk[a].z, fmaf(qv.y, kk[a].y, qv.x * kk[a].x)));
      d = group_sum(d, lpp_log2, lane);
      if (p + a * stride < p1) merge(st, d * sl, 1.0f, vv[a]);
    }
  }
  // the lane groups of a wave, then the waves of the workgroup: lane `sub` of group 0 ends up with the chunk's state
  for (u32 off = lpp; off < 64u; off <<= 1) {
    const float m = __shfl_xor(st.m, off, 64), s = __shfl_xor(st.s, off, 64);
    f32x4 o;
    o.x = __shfl_xor(st.o.x, off, 64); o.y = __shfl_xor(st.o.y, off, 64);
    o.z = __shfl_xor(st.o.z, off, 64); o.w = __shfl_xor(st.o.w, off, 64);
    merge(st, m, s, o);
  }
  s_m[wave][lane] = st.m; s_s[wave][lane] = st.s; s_o[wave][lane] = st.o;
  __syncthreads();
  if (wave != 0u || lane >= lpp) {
    if (chunks == 1u) return;
  } else {
    for (u32 w = 1; w < kWaves; ++w) merge(st, s_m[w][lane], s_s[w][lane], s_o[w][lane]);
    float* dst = out + static_cast<size_t>(head) * head_dim + 4u * sub;
    if (chunks == 1u) {
      if (live) {
        const float inv = 1.0f / st.s;
        *reinterpret_cast<f32x4*>(dst) = f32x4{st.o.x * inv, st.o.y * inv, st.o.z * inv, st.o.w * inv};
      }
      return;
    }
    // [head][chunk][lpp lanes][m, s, -, -, o.xyzw] through to memory: two 16-byte stores at agent scope
    const u32 slot = static_cast<u32>(((static_cast<size_t>(head) * chunks + ci) * lpp + sub) * 32u);
    __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(st.m), __float_as_uint(st.s), 0u, 0u}, part_rsrc, static_cast<int>(slot), 0, 16);
    __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(st.o.x), __float_as_uint(st.o.y), __float_as_uint(st.o.z), __float_as_uint(st.o.w)},
                                           part_rsrc, static_cast<int>(slot + 16u), 0, 16);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (lane == 0u) {
      const u32 old = __hip_atomic_fetch_add(counters + head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (old == chunks - 1u) __hip_atomic_store(counters + head, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_old = old;
    }
  }
  __syncthreads();
  if (wave != 0u || lane >= lpp || s_old != chunks - 1u) return;
  State tot = {-INFINITY, 0.0f, zero4};
  constexpr u32 kRound = 16;                       // chunks whose states are in flight together; merged in chunk order
  for (u32 c0 = 0; c0 < chunks; c0 += kRound) {
    u32x4 ms[kRound], ov[kRound];
#pragma unroll
    for (u32 cc = 0; cc < kRound; ++cc) {
      const u32 c = min(c0 + cc, chunks - 1u);
      const u32 slot = static_cast<u32>(((static_cast<size_t>(head) * chunks + c) * lpp + sub) * 32u);
      ms[cc] = __builtin_amdgcn_raw_buffer_load_b128(part_rsrc, static_cast<int>(slot), 0, 16);
      ov[cc] = __builtin_amdgcn_raw_buffer_load_b128(part_rsrc, static_cast<int>(slot + 16u), 0, 16);
    }
#pragma unroll
    for (u32 cc = 0; cc < kRound; ++cc)
      if (c0 + cc < chunks)
        merge(tot, __uint_as_float(ms[cc].x), __uint_as_float(ms[cc].y),
              f32x4{__uint_as_float(ov[cc].x), __uint_as_float(ov[cc].y), __uint_as_float(ov[cc].z), __uint_as_float(ov[cc].w)});
  }
  if (live) {
    const float inv = 1.0f / tot.s;
    *reinterpret_cast<f32x4*>(out + static_cast<size_t>(head) * head_dim + 4u * sub) =
        f32x4{tot.o.x * inv, tot.o.y * inv, tot.o.z * inv, tot.o.w * inv};
  }
}

// ---- head dimensions 64, 128 and 256, the query heads of a KV head together (matrix cores, v_mfma_f32_16x16x4_f32) ----
// The kernel above reads the cache once per query head and spends about thirty vector instructions per two positions on the
// reduction over a position's lanes and the rescaling.  Here the query heads that share a KV head are the columns of
// a matrix product (f32 throughout; up to eight of them), so the cache is read once:
//   scores[16 positions][heads] = K tile . q,  lane l: K[position l%16][dims 16 j + 4 g + e], g = l/16, one 16-byte LDS read
//     for four products;
//   out[dims][heads] += V tile . p,  product v takes the positions 4 g + v: the score registers are its operand as they
//     lie, and V[position 4 g + v][dims 64 h + 4 (l%16) + e] is read in whole rows.
// A lane's running maximum and the factor of its sums belong to one head, l%16: nothing crosses lanes but the maximum of a
// tile (two swaps).
// Data movement: a wave's tile of 16 positions comes by copies into LDS, a KB of whole lines each and non-temporal (every line
// is read once; without the hint 128 query heads over 32 KV heads, 16384 positions: 97 us, with it 86).  K goes to registers
// as soon as it is there, and its place takes the next tile's K before the first product; V the same.  So every wave has one
// to two halves of a tile on their way while it computes, no register holds a load in flight, and two waves a SIMD fit
// (with K and V in registers they did not: 24 us where four waves took 18.7).
// Rounding: a score is added up in a tree over sums of four products, a tile's share of the output starts at zero (eight
// products in a row), waves and chunks meet in trees.  Against fp64, averages over 16 inputs, 64, 128 and 256 dims, heads alone and
// in pairs and fours: 0.94 .. 1.02 of the kernel's above with 64 and 256 positions (single inputs scatter by 10-20 %), 0.72 .. 0.95 with 1024 and 2048, 0.71 .. 0.84 with 8192.
// Bound: a launch's time is a fixed part and the bytes at the memory's own rate, 128 dims, caches out of the last level: 32 heads over 8 8-9 us + bytes / 6.8-7.05
// TB/s (4096 .. 32768 positions), 32 heads of their own 6.2-7.6 + bytes / 6.9-7.2.  The fixed part is the start (1 us before the first copies are out), the last tile
// and, with several chunks, their sum: the store of a chunk's state has to be acknowledged, the counter answers, the states come back.
// Measured (us, before -> now: before is the kernel above, or for 64 dims, several heads and from 4096 positions on one that
// kept K and V in registers, four waves a CU; 128 dims unless said): 32 heads over 8, 8192 positions 19.0 -> 17.1; 32 heads of their
// own, 2048 positions 16.65 -> 15.2, 1024 12.3 -> 10.7, 512 9.0 -> 8.2; four heads, 16000 positions 21.5 -> 16.9; 128 heads over 32,
// 16384 positions 84.0 -> 81.9 (6.6 TB/s); 256 dims, 64 heads over 16, 8000 positions 99.7 -> 52.
// Waves: eight; with 128 dims four where a workgroup has 512 positions or more, four tiles for a wave of eight, and a KV head at most eight workgroups
// (both sides at the runtime's kAttentionFourWaves: fewer streams at a time, but half the threads to join the chunks).  256 dims: four, an LDS tile is 32 KB.
constexpr u32 kTiledHeads = 8;
template <int DIM, int W> struct Tiled {
  static constexpr u32 HALF = 64u * DIM;               // bytes of a wave's tile: 16 positions of K, then of V
  static constexpr u32 LDS = W * 2u * HALF;
};

__device__ __forceinline__ float max_over_groups(float v) {      // over the four lanes l, l ^ 16, l ^ 32, l ^ 48
  const u32 b = __float_as_uint(v);
  const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(b, b, false, false));
  const float m = fmaxf(__uint_as_float(a.x), __uint_as_float(a.y));
  const u32 c = __float_as_uint(m);
  const u32x2 d = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(c, c, false, false));
  return fmaxf(__uint_as_float(d.x), __uint_as_float(d.y));
}
__device__ __forceinline__ float sum_over_groups(float v) {
  const u32 b = __float_as_uint(v);
  const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(b, b, false, false));
  const float m = __uint_as_float(a.x) + __uint_as_float(a.y);
  const u32 c = __float_as_uint(m);
  const u32x2 d = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(c, c, false, false));
  return __uint_as_float(d.x) + __uint_as_float(d.y);
}
// 2^(a - b) for a <= b, 1 where they are equal (two infinities as well)
__device__ __forceinline__ float factor(float a, float b) { return a == b ? 1.0f : __builtin_amdgcn_exp2f(a - b); }

// N states in registers (their o for the caller's four dims) as one; N a power of two
template <u32 N>
__device__ __forceinline__ State merge_tree(const float (&m)[N], const float (&s)[N], const f32x4 (&o)[N]) {
  float top = m[0];
#pragma unroll
  for (u32 i = 1; i < N; ++i) top = fmaxf(top, m[i]);
  float ss[N];
  f32x4 oo[N];
#pragma unroll
  for (u32 i = 0; i < N; ++i) {
    const float f = factor(m[i], top);
    ss[i] = s[i] * f;
    oo[i] = o[i] * f;
  }
#pragma unroll
  for (u32 w = N / 2; w >= 1; w /= 2)
#pragma unroll
    for (u32 i = 0; i < w; ++i) {
      ss[i] += ss[i + w];
      oo[i] += oo[i + w];
    }
  return State{top, ss[0], oo[0]};
}

// group = KV head * subs + sub: the query heads head0 .. head0 + heads - 1 of a KV head (per_kv of them, eight at a time)
template <int DIM, int W>     // W waves
__device__ __forceinline__ void tiled_body(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                                           float* __restrict__ out, u32 seq_len, u32 per_kv, u32 subs, u32 max_seq_len, float scale,
                                           u32 chunk, u32 chunks, u32 groups, float* __restrict__ partial, u32* __restrict__ counters,
                                           uint8_t* lds) {
  using T = Tiled<DIM, W>;
  constexpr u32 H = kTiledHeads, Q = DIM / 4, kRowBytes = 4u * DIM;      // Q: quads of a head's output
  constexpr int KJ = DIM / 16, VH = DIM / 64, COPIES = T::HALF / 1024u;
  __shared__ float s_m[W][H], s_s[W][H];
  __shared__ u32 s_old;
  const u32 lane = threadIdx.x & 63u, col = lane & 15u, g = lane >> 4;
  const u32 wave = static_cast<u32>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
  const u32 group = blockIdx.x / chunks, ci = blockIdx.x - group * chunks;
  const u32 kv_head = group / subs, sub = group - kv_head * subs;
  const u32 head0 = kv_head * per_kv + sub * H, heads = min(H, per_kv - sub * H);
  const u32 p0 = ci * chunk, len = min(seq_len, p0 + chunk) - p0;      // positions of this chunk (>= 1)
  u32x4 qv[KJ];      // in asm, like the waits: the compiler would wait for every copy behind them
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    const float* src = q + static_cast<size_t>(head0 + min(col, heads - 1u)) * DIM + 16 * j + 4u * g;
    asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(qv[j]) : "v"(src) : "memory");
  }
  // Copies into LDS, a KB of whole lines each.  Positions behind the chunk are outside the buffer: nothing is read for them
  // (what lies in their place has weight 0).
  const size_t kv_at = (static_cast<size_t>(kv_head) * max_seq_len + p0) * DIM;
  const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(k) + kv_at, 0, static_cast<int>(len * kRowBytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(v) + kv_at, 0, static_cast<int>(len * kRowBytes), 0x00020000);
  const u32 lds_k = static_cast<u32>(reinterpret_cast<size_t>((const __attribute__((address_space(3))) uint8_t*)lds)) + wave * (2u * T::HALF);
  const u32 lds_v = lds_k + T::HALF;
  // V lies in LDS as in memory.  K's unit u (16 bytes) of row r lies at u ^ r: the reads below take one unit of sixteen rows.
  constexpr u32 kRowsPerCopy = 1024u / kRowBytes;
  const u32 row_in = lane / Q, unit = lane - row_in * Q;
  u32 koff[COPIES];
#pragma unroll
  for (int i = 0; i < COPIES; ++i) koff[i] = row_in * kRowBytes + (unit ^ (i * kRowsPerCopy + row_in)) * 16u;
  // (the whole offset in the lane's register: a scalar part of it beyond the buffer's end would wrap the bounds check)
  auto copy = [&](__amdgpu_buffer_rsrc_t rsrc, u32 dst, u32 off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(uintptr_t)dst, 16, static_cast<int>(off), 0, 0, 2 /* nt */);
  };
  auto copy_k = [&](u32 p) {
#pragma unroll
    for (int i = 0; i < COPIES; ++i) copy(k_rsrc, lds_k + 1024u * i, koff[i] + (p * kRowBytes + 1024u * i));
  };
  auto copy_v = [&](u32 p) {
#pragma unroll
    for (int i = 0; i < COPIES; ++i) copy(v_rsrc, lds_v + 1024u * i, lane * 16u + (p * kRowBytes + 1024u * i));
  };
  u32 p = wave * 16u;      // of the chunk
  // (also by a wave that has no position: outside the buffer)
  copy_k(p);
  copy_v(p);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * COPIES) : "memory");
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    asm volatile("" : "+v"(qv[j])::"memory");
    if (col >= heads) qv[j] = u32x4{0u, 0u, 0u, 0u};
  }
  const u32 k_read = lds_k + col * kRowBytes + 16u * (g ^ (col & 3u)) + 64u * (col >> 2);      // unit 4 j + g: bits 6 and 7 ^ j, then 256 bytes on
  const u32 v_read = lds_v + 4u * g * kRowBytes + 16u * col;
  const float sl = scale * kLog2e;
  float m = -INFINITY, s = 0.0f;
  const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 o[VH][4];
#pragma unroll
  for (int h = 0; h < VH; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[h][e] = zero4;
  for (; p < len; p += W * 16u) {
    const bool more = p + W * 16u < len;
    u32x4 kk[KJ];
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COPIES) : "memory");      // K is there, V behind it
#pragma unroll
    for (int j = 0; j < KJ; ++j) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(kk[j]) : "v"(k_read ^ (64u * (j & 3))), "n"(256 * (j >> 2)) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < KJ; ++j) asm volatile("" : "+v"(kk[j])::"memory");
    if (more) copy_k(p + W * 16u);      // K is in registers: its place takes the next tile's
    f32x4 sc[KJ];
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      f32x4 part[4];
      const f32x4 kj = __builtin_bit_cast(f32x4, kk[j]), qj = __builtin_bit_cast(f32x4, qv[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) part[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kj[e], qj[e], zero4, 0, 0, 0);
      sc[j] = (part[0] + part[1]) + (part[2] + part[3]);
      __builtin_amdgcn_sched_barrier(0);      // (all the products first would take four times the registers)
    }
#pragma unroll
    for (int w = KJ / 2; w >= 1; w /= 2)
#pragma unroll
      for (int j = 0; j < w; ++j) sc[j] += sc[j + w];
    float x[4], top = -INFINITY;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      x[a] = sc[0][a] * sl;
      if (p + 4u * g + a < len) top = fmaxf(top, x[a]);      // (a NaN comes in again with its own weight)
    }
    const float nm = fmaxf(m, max_over_groups(top)), c = factor(m, nm);
    m = nm;
    float w[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) w[a] = p + 4u * g + a < len ? factor(x[a], nm) : 0.0f;
    s = fmaf(s, c, (w[0] + w[1]) + (w[2] + w[3]));
    u32x4 vv[4][VH];
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COPIES) : "memory");      // V is there, the next K behind it
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int h = 0; h < VH; ++h)
#pragma unroll
      for (int a = 0; a < 4; ++a) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(vv[a][h]) : "v"(v_read), "n"(a * kRowBytes + 256 * h) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int h = 0; h < VH; ++h)
#pragma unroll
      for (int a = 0; a < 4; ++a) asm volatile("" : "+v"(vv[a][h])::"memory");
    if (more) copy_v(p + W * 16u);
    if (p + 16u > len) {      // a last tile that is not full: what lies behind the positions may be anything, their weight is 0
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int h = 0; h < VH; ++h) vv[a][h] = p + 4u * g + a < len ? vv[a][h] : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int h = 0; h < VH; ++h) {
      f32x4 t[2][4];
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const f32x4 va = __builtin_bit_cast(f32x4, vv[a][h]);
#pragma unroll
        for (int e = 0; e < 4; ++e) t[a >> 1][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[e], w[a], (a & 1) ? t[a >> 1][e] : zero4, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int a = 0; a < 4; ++a) o[h][e][a] = fmaf(o[h][e][a], c, t[0][e][a] + t[1][e][a]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (a wave without positions: its copies)
  // The waves' states meet in LDS, each in its own wave's tile: [head][quad]
  f32x4* s_o = reinterpret_cast<f32x4*>(lds);
  constexpr u32 kWaveUnits = 2u * T::HALF / 16u;
  s = sum_over_groups(s);
  if (col < heads) {
    if (g == 0u) {
      s_m[wave][col] = m;
      s_s[wave][col] = s;
    }
    // register a of sum (h, e) is dim 64 h + 16 g + 4 a + e
#pragma unroll
    for (int h = 0; h < VH; ++h)
#pragma unroll
      for (int a = 0; a < 4; ++a) s_o[wave * kWaveUnits + col * Q + 16 * h + 4 * g + a] = f32x4{o[h][0][a], o[h][1][a], o[h][2][a], o[h][3][a]};
  }
  __syncthreads();
  // a thread per (head, quad of dims), or two: the waves in a tree (one without positions brings zeros under a maximum of
  // -infinity), then the chunks by the workgroup that arrives last
  constexpr u32 kThreads = 64u * W;
  const u32 pairs = heads * Q;
  // [group][chunk][head][quads, then {m, s}] through to memory: 16-byte buffer accesses at agent scope (sc1)
  constexpr u32 kHeadBytes = (Q + 1u) * 16u;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(partial, 0, static_cast<int>(groups * chunks * H * kHeadBytes), 0x00020000);
  auto slot = [&](u32 c, u32 hd) { return ((group * chunks + c) * H + hd) * kHeadBytes; };
  f32x4* dst = reinterpret_cast<f32x4*>(out + static_cast<size_t>(head0) * DIM);
  for (u32 i = threadIdx.x; i < pairs; i += kThreads) {
    const u32 hd = i / Q, quad = i - hd * Q;
    float wm[W], ws[W];
    f32x4 wo[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      wm[w] = s_m[w][hd];
      ws[w] = s_s[w][hd];
      wo[w] = s_o[w * kWaveUnits + i];
    }
    const State st = merge_tree<W>(wm, ws, wo);
    if (chunks == 1u) {
      const float inv = 1.0f / st.s;
      dst[i] = st.o * inv;
    } else {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, st.o), rsrc, static_cast<int>(slot(ci, hd) + quad * 16u), 0, 16);
      if (quad == 0u)
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(st.m), __float_as_uint(st.s), 0u, 0u}, rsrc, static_cast<int>(slot(ci, hd) + Q * 16u), 0, 16);
    }
  }
  if (chunks == 1u) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the coherent stores have been acknowledged
  __syncthreads();
  if (threadIdx.x == 0u) {
    const u32 old = __hip_atomic_fetch_add(counters + group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old == chunks - 1u) __hip_atomic_store(counters + group, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_old = old;
  }
  __syncthreads();
  if (s_old != chunks - 1u) return;
  // The last workgroup joins the chunks [c0, c1) of a pair, N of them in flight together and scaled once, as the waves' states are
  auto join = [&](u32 pair, u32 c0, u32 c1, auto n_c) {
    constexpr u32 N = decltype(n_c)::value;
    const u32 hd = pair / Q, quad = pair - hd * Q;
    State tot = {-INFINITY, 0.0f, zero4};
    for (; c0 < c1; c0 += N) {
      u32x4 ms[N], ov[N];
#pragma unroll
      for (u32 cc = 0; cc < N; ++cc) {
        const u32 at = slot(min(c0 + cc, c1 - 1u), hd);
        ms[cc] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(at + Q * 16u), 0, 16);
        ov[cc] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(at + quad * 16u), 0, 16);
      }
      float cm[N], cs[N];
      f32x4 co[N];
#pragma unroll
      for (u32 cc = 0; cc < N; ++cc) {
        const bool there = c0 + cc < c1;
        cm[cc] = there ? __uint_as_float(ms[cc].x) : -INFINITY;
        cs[cc] = there ? __uint_as_float(ms[cc].y) : 0.0f;
        co[cc] = there ? __builtin_bit_cast(f32x4, ov[cc]) : zero4;
      }
      const State r = merge_tree<N>(cm, cs, co);
      merge(tot, r.m, r.s, r.o);
    }
    return tot;
  };
  auto finish = [&](u32 pair, const State& tot) {
    const float inv = 1.0f / tot.s;
    dst[pair] = tot.o * inv;
  };
  // Up to sixteen chunks in one tree.  More: as many slices of the workgroup's threads as there are take runs of chunks, eight in flight, and the slices
  // meet in LDS.  (The way without slices in code of its own: through the other it took 0.3 us longer at every length - 32 heads over 8, 900
  // positions 8.1 and 7.8 us.  Slices of sixteen in flight: 8 heads over one, 6000 positions 13.5 us, of eight 12.0.)
  constexpr u32 kMostSlices = 16;
  u32 slices = 1u;
  while (chunks > 16u && slices < kMostSlices && 2u * slices * pairs <= kThreads && slices * 8u < chunks) slices *= 2u;
  if (slices == 1u) {
    for (u32 i = threadIdx.x; i < pairs; i += kThreads)
      finish(i, chunks <= 8u ? join(i, 0u, chunks, std::integral_constant<u32, 8>{}) : join(i, 0u, chunks, std::integral_constant<u32, 16>{}));
    return;
  }
  const u32 per_slice = (chunks + slices - 1u) / slices, slice = threadIdx.x / pairs;
  State tot = {-INFINITY, 0.0f, zero4};
  if (slice < slices) tot = join(threadIdx.x - slice * pairs, slice * per_slice, min(chunks, (slice + 1u) * per_slice), std::integral_constant<u32, 8>{});
  f32x2* s_ms = reinterpret_cast<f32x2*>(s_o + kThreads);
  s_o[threadIdx.x] = tot.o;
  s_ms[threadIdx.x] = f32x2{tot.m, tot.s};
  __syncthreads();
  if (threadIdx.x >= pairs) return;
  auto join_slices = [&](auto n_c) {
    constexpr u32 N = decltype(n_c)::value;
    float jm[N], js[N];
    f32x4 jo[N];
#pragma unroll
    for (u32 n = 0; n < N; ++n) {
      const f32x2 ms = s_ms[n * pairs + threadIdx.x];
      jm[n] = ms.x;
      js[n] = ms.y;
      jo[n] = s_o[n * pairs + threadIdx.x];
    }
    finish(threadIdx.x, merge_tree<N>(jm, js, jo));
  };
  if (slices == 2u) join_slices(std::integral_constant<u32, 2>{});
  else if (slices == 4u) join_slices(std::integral_constant<u32, 4>{});
  else if (slices == 8u) join_slices(std::integral_constant<u32, 8>{});
  else join_slices(std::integral_constant<u32, kMostSlices>{});
}

}  // namespace decode_attention
