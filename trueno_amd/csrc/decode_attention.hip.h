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

// ---- head dimensions 64 and 128, the query heads of a KV head together (matrix cores, v_mfma_f32_16x16x4_f32) ----
// The kernel above reads the cache once per query head and spends about thirty vector instructions per two positions on the
// reduction over a position's lanes and the rescaling.  Here the query heads that share a KV head are the columns of
// a matrix product (f32 throughout; up to eight of them), so the cache is read once:
//   scores[16 positions][heads] = K tile . q,  lane l: K[position l%16][dims 16 j + 4 g + e], g = l/16, a 16-byte load for
//     four products;
//   out[dims][heads] += V tile . p,  product v takes the positions 4 g + v: the score registers are its operand as they
//     lie, and V[position 4 g + v][dims 64 h + 4 (l%16) + e] is read in whole lines.
// A lane's running maximum and the factor of its sums belong to one head, l%16: nothing crosses lanes but the maximum of a
// tile (two swaps).  K of the next tile is asked for when the scores are made, V when the sums are.
// Rounding: a score is added up in a tree over sums of four products, a tile's share of the output starts at zero (eight
// products in a row), waves and chunks meet in trees.  Against fp64 the error is, on the average over 16 inputs, 0.94 .. 1.03 times
// the kernel's above up to 256 positions (no more: one input scatters by 5-10 %) and 0.98 .. 0.70 times from there to 8192.
// Bound by HBM with many positions; what is in flight is the next tile of every wave (16 KB at 128 dims).  Measured (us,
// the kernel above -> this one; 32 query heads x 128 unless said): 8 KV heads, 8192 positions 31.5 -> 18.7; 32 KV heads,
// 8192 positions 45.5 -> 43.3, 2048 positions 17.5 -> 17.3 (cold), 512 positions 10.0 -> 9.4 (cold); 64 heads x 64 over 16
// KV heads, 700 positions 9.4 -> 7.1.  With 128 dims workgroups of eight waves spill (24 us where four waves take 18.7),
// with 64 dims eight waves are faster than four (14.1 against 16.7 us, 32 KV heads, 4000 positions).  256 dims need 256
// registers for K, V, q and the sums alone: they spill, and stay with the kernel above (as do head counts that the number
// of KV heads does not divide).
constexpr u32 kTiledHeads = 8;
template <int DIM> struct Tiled { static constexpr u32 WAVES = DIM == 64 ? 8u : 4u; };

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
template <int N>
__device__ __forceinline__ State merge_tree(const float (&m)[N], const float (&s)[N], const f32x4 (&o)[N]) {
  float top = m[0];
#pragma unroll
  for (int i = 1; i < N; ++i) top = fmaxf(top, m[i]);
  float ss[N];
  f32x4 oo[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float f = factor(m[i], top);
    ss[i] = s[i] * f;
    oo[i] = o[i] * f;
  }
#pragma unroll
  for (int w = N / 2; w >= 1; w /= 2)
#pragma unroll
    for (int i = 0; i < w; ++i) {
      ss[i] += ss[i + w];
      oo[i] += oo[i + w];
    }
  return State{top, ss[0], oo[0]};
}

// group = KV head * subs + sub: the query heads head0 .. head0 + heads - 1 of a KV head (per_kv of them, eight at a time)
template <int DIM>
__device__ __forceinline__ void tiled_body(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                                           float* __restrict__ out, u32 seq_len, u32 per_kv, u32 subs, u32 max_seq_len, float scale,
                                           u32 chunk, u32 chunks, u32 groups, float* __restrict__ partial, u32* __restrict__ counters) {
  constexpr u32 W = Tiled<DIM>::WAVES, H = kTiledHeads, Q = DIM / 4;      // quads of a head's output
  constexpr int KJ = DIM / 16, VH = DIM / 64;
  __shared__ float s_m[W][H], s_s[W][H];
  __shared__ f32x4 s_o[W][H][Q];
  __shared__ u32 s_old;
  const u32 lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, col = lane & 15u, g = lane >> 4;
  const u32 group = blockIdx.x / chunks, ci = blockIdx.x - group * chunks;
  const u32 kv_head = group / subs, sub = group - kv_head * subs;
  const u32 head0 = kv_head * per_kv + sub * H, heads = min(H, per_kv - sub * H);
  const f32x4* kp = reinterpret_cast<const f32x4*>(k + static_cast<size_t>(kv_head) * max_seq_len * DIM) + g;
  const f32x4* vp = reinterpret_cast<const f32x4*>(v + static_cast<size_t>(kv_head) * max_seq_len * DIM) + col;
  f32x4 qv[KJ];
#pragma unroll
  for (int j = 0; j < KJ; ++j)
    qv[j] = col < heads ? reinterpret_cast<const f32x4*>(q + static_cast<size_t>(head0 + col) * DIM)[4 * j + g] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const float sl = scale * kLog2e;
  const u32 p0 = ci * chunk, p1 = min(seq_len, p0 + chunk);
  float m = -INFINITY, s = 0.0f;
  const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 o[VH][4];
#pragma unroll
  for (int h = 0; h < VH; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[h][e] = zero4;
  f32x4 kk[KJ], vv[4][VH];
  auto load_k = [&](u32 p) {      // (positions behind the chunk: its last one, which the cache holds; their weight is 0)
    const f32x4* row = kp + static_cast<size_t>(min(p + col, p1 - 1u)) * Q;
#pragma unroll
    for (int j = 0; j < KJ; ++j) kk[j] = row[4 * j];
  };
  auto load_v = [&](u32 p) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const f32x4* row = vp + static_cast<size_t>(min(p + 4u * g + a, p1 - 1u)) * Q;
#pragma unroll
      for (int h = 0; h < VH; ++h) vv[a][h] = __builtin_nontemporal_load(row + 16 * h);
    }
  };
  u32 p = p0 + wave * 16u;
  if (p < p1) {
    load_k(p);
    load_v(p);
  }
  for (; p < p1; p += W * 16u) {
    f32x4 sc[KJ];
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      f32x4 part[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) part[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j][e], qv[j][e], zero4, 0, 0, 0);
      sc[j] = (part[0] + part[1]) + (part[2] + part[3]);
      __builtin_amdgcn_sched_barrier(0);      // (all the products first would take four times the registers, and spill)
    }
#pragma unroll
    for (int w = KJ / 2; w >= 1; w /= 2)
#pragma unroll
      for (int j = 0; j < w; ++j) sc[j] += sc[j + w];
    const bool more = p + W * 16u < p1;
    if (more) load_k(p + W * 16u);
    float x[4], top = -INFINITY;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      x[a] = sc[0][a] * sl;
      if (p + 4u * g + a < p1) top = fmaxf(top, x[a]);      // (a NaN comes in again with its own weight)
    }
    const float nm = fmaxf(m, max_over_groups(top)), c = factor(m, nm);
    m = nm;
    float w[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) w[a] = p + 4u * g + a < p1 ? factor(x[a], nm) : 0.0f;
    if (p + 16u > p1) {      // a last tile that is not full: what stands in for the missing rows may be infinite, their weight is 0
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int h = 0; h < VH; ++h) vv[a][h] = p + 4u * g + a < p1 ? vv[a][h] : zero4;
    }
    s = fmaf(s, c, (w[0] + w[1]) + (w[2] + w[3]));
#pragma unroll
    for (int h = 0; h < VH; ++h) {
      f32x4 t[2][4];
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int e = 0; e < 4; ++e) t[a >> 1][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[a][h][e], w[a], (a & 1) ? t[a >> 1][e] : zero4, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int a = 0; a < 4; ++a) o[h][e][a] = fmaf(o[h][e][a], c, t[0][e][a] + t[1][e][a]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) load_v(p + W * 16u);
  }
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
      for (int a = 0; a < 4; ++a) s_o[wave][col][16 * h + 4 * g + a] = f32x4{o[h][0][a], o[h][1][a], o[h][2][a], o[h][3][a]};
  }
  __syncthreads();
  // a thread per (head, quad of dims): the waves in order, then the chunks in order by the workgroup that arrives last
  const u32 hd = threadIdx.x / Q, quad = threadIdx.x - hd * Q;
  const bool mine = hd < heads;
  State st = {-INFINITY, 0.0f, zero4};
  if (mine) {      // (a wave without positions brings nothing: zeros under a maximum of -infinity)
    float wm[W], ws[W];
    f32x4 wo[W];
#pragma unroll
    for (u32 w = 0; w < W; ++w) {
      wm[w] = s_m[w][hd];
      ws[w] = s_s[w][hd];
      wo[w] = s_o[w][hd][quad];
    }
    st = merge_tree<W>(wm, ws, wo);
  }
  f32x4* dst = reinterpret_cast<f32x4*>(out + static_cast<size_t>(head0 + hd) * DIM) + quad;
  if (chunks == 1u) {
    if (mine) {
      const float inv = 1.0f / st.s;
      *dst = f32x4{st.o.x * inv, st.o.y * inv, st.o.z * inv, st.o.w * inv};
    }
    return;
  }
  // [group][chunk][head][quads, then {m, s}] through to memory: 16-byte buffer accesses at agent scope (sc1)
  constexpr u32 kHeadBytes = (Q + 1u) * 16u;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(partial, 0, static_cast<int>(groups * chunks * H * kHeadBytes), 0x00020000);
  auto slot = [&](u32 c) { return ((group * chunks + c) * H + hd) * kHeadBytes; };
  if (mine) {
    __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(st.o.x), __float_as_uint(st.o.y), __float_as_uint(st.o.z), __float_as_uint(st.o.w)},
                                           rsrc, static_cast<int>(slot(ci) + quad * 16u), 0, 16);
    if (quad == 0u)
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(st.m), __float_as_uint(st.s), 0u, 0u}, rsrc, static_cast<int>(slot(ci) + Q * 16u), 0, 16);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the coherent stores have been acknowledged
  __syncthreads();
  if (threadIdx.x == 0u) {
    const u32 old = __hip_atomic_fetch_add(counters + group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old == chunks - 1u) __hip_atomic_store(counters + group, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_old = old;
  }
  __syncthreads();
  if (s_old != chunks - 1u || !mine) return;
  State tot = {-INFINITY, 0.0f, zero4};
  constexpr u32 kRound = 16;
  for (u32 c0 = 0; c0 < chunks; c0 += kRound) {
    u32x4 ms[kRound], ov[kRound];
#pragma unroll
    for (u32 cc = 0; cc < kRound; ++cc) {
      const u32 at = slot(min(c0 + cc, chunks - 1u));
      ms[cc] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(at + Q * 16u), 0, 16);
      ov[cc] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(at + quad * 16u), 0, 16);
    }
    float cm[kRound], cs[kRound];
    f32x4 co[kRound];
#pragma unroll
    for (u32 cc = 0; cc < kRound; ++cc) {
      const bool there = c0 + cc < chunks;
      cm[cc] = there ? __uint_as_float(ms[cc].x) : -INFINITY;
      cs[cc] = there ? __uint_as_float(ms[cc].y) : 0.0f;
      co[cc] = there ? f32x4{__uint_as_float(ov[cc].x), __uint_as_float(ov[cc].y), __uint_as_float(ov[cc].z), __uint_as_float(ov[cc].w)} : zero4;
    }
    const State r = merge_tree<kRound>(cm, cs, co);
    merge(tot, r.m, r.s, r.o);
  }
  const float inv = 1.0f / tot.s;
  *dst = f32x4{tot.o.x * inv, tot.o.y * inv, tot.o.z * inv, tot.o.w * inv};
}

}  // namespace decode_attention
