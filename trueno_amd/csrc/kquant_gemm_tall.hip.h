// Matrix-core k-quant GEMM for many tokens (gfx950, v_mfma_f32_32x32x16_f16):
//   C[m x n] = A[m x k] . dequant(W[n x k])^T,  c[row*n + col]      (trueno-gpu/src/kernels/quantize.rs:568-574)
// with the operands of kquant_gemm_f16.hip.h - weights as exact integers times a power of two in f16, activations as two
// f16 pieces of a run of 256 scaled by a power of two.  There a wave multiplies 32 rows of W with 16 tokens at a time and
// builds the weight operand anew for each 16: with many tokens the vector unit and the LDS (a page of token operands per
// matrix instruction) are what it waits for.  Here the activations are made into operands once, by a launch of their own
// (2048 x 4096: 11 us, 16 with the activations out of the caches), and a wave holds a tile of 32 rows x 64 tokens: a weight operand, which
// costs ten vector instructions (Q6_K thirty-two), feeds four matrix instructions (Q6_K six).
//   * What bounds it: beside other waves' vector instructions a matrix instruction takes half its cycles of a SIMD's issue and a vector
//     instruction four and a half (measured with one wave of each on a SIMD), so a super-block takes a wave the larger of M and M / 2 + 4.5 V cycles, M = 2304
//     (Q6_K 3072), V = 460 (Q5_K 610, Q6_K 860).  With 64 rows x 32 tokens, the same registers, V was 650 (1250 for Q6_K): us, that form -> this
//     one, Q6_K 4096 x 11008, 512 tokens 192 -> 163, 11008 x 4096, 1024 tokens 372 -> 309; Q5_K 11008 x 4096, 512 tokens 141 -> 135; Q4_K
//     14336 x 4096, 2048 tokens 538 -> 531.  The tokens' LDS reads double: 90 of 128 bytes a cycle.
//   * That accounts for four fifths of the cycles: Q4_K 14336 x 4096, 2048 tokens 722 k of 906 k (matrix cores busy 57 %), Q6_K 4096 x 11008, 512 tokens 232 k of
//     300 k; what the rest is has not been found.  The clock is not what it lacks: a library's f16 product of as many matrix operations runs at the same 1.7 GHz
//     and takes 642 k (72 %).
//   * A workgroup is four waves with a strip of 32 rows each against the same two operand tiles of 32 tokens, two workgroups a CU (70-80 KB of
//     LDS, 220-240 registers): their phases drift apart, so that one's sums and headers run under the other's products.
//   * Weights and token pages come by copies into LDS, pages in a ring of three chunks of four products (Q6_K two, its
//     weight tile is larger), the next super-block's weight tile as soon as the last of the current one is in registers.
//     Waits are counted by hand; every path issues the same number of copies (behind the end of a run the last
//     super-block's again).  A wave in its products goes first (up to 5 % against equal priorities).
//   * Rounding.  The hi pieces' sums are kept apart from the lo pieces' (alone they are whole numbers on a coarse grid and
//     hardly round), what is added to them is hi pieces as well, and the running sum over super-blocks is put by every few
//     (put_by).  Against fp64 the error is Q4_K 0.86 .. 1.02 (0.954 on the average), Q5_K 0.81 .. 1.02
//     (0.946), Q6_K 0.81 .. 0.94 (0.878) times the 16-token kernel's, over 70 shapes a format drawn from 33 .. 2048 tokens, 512 .. 32000 rows, 1024 .. 14336 columns that the rule gives this kernel.
#pragma once
#include "kquant_gemm_f16.hip.h"
#include <utility>

namespace gemm_tall {

using namespace gemm_f16;      // the LDS helpers, split_f16, pack_h2

constexpr u32 kTile = 32;                      // tokens of an operand tile
constexpr u32 kWaves = 4;                      // of a workgroup; a wave holds RT strips of 32 rows against TT operand tiles, RT TT = 2
constexpr u32 kPagesBytes = 32 * 1024;         // 16 products x (lo page, hi page) of 64 lanes x 16 bytes
constexpr u32 kAuxBytes = 2048;                // sums (1 KB), factors (128 bytes, padded)
constexpr u32 kOperandBytes = kPagesBytes + kAuxBytes;      // of a (token tile, super-block)
constexpr u32 kPageStride = 1024 + 16;         // LDS of the converter: pages apart by one slot more, so that a token's writes spread over the banks

// ---- the token operands of one (tile of 32 tokens, super-block), by one workgroup of 256 threads ----
//   pages 2 q (lo pieces) and 2 q + 1 (hi pieces), slot 32 g + token: eight f16, elements 32 j + 8 (u % 4) + perm of the token's run, u = q / 2,
//   j = 2 (2g + u / 4) + q % 2, perm = 0,2,1,3,4,6,5,7 - what the ANDs on a dword of nibbles leave in its 16-bit lanes
//   (a lo piece is 2^11 times what the hi piece leaves out: it keeps its eleven bits beside a value 2^24 times larger)
//   aux: slot 32 g + token: f16 hi pieces of 2^-5 * (sum of the scaled sub-block 4 g + e), e = 0, 2, 1, 3, then the lo pieces;
//        at 1024: f32 2^(E+14) per token (NaN where the run holds an infinity or a NaN)
__device__ __forceinline__ void convert_body(const float* __restrict__ a, uint8_t* __restrict__ ops, u32 m, u32 nsb) {
  __shared__ __attribute__((aligned(16))) uint8_t s_page[32 * kPageStride];
  __shared__ __attribute__((aligned(16))) uint8_t s_aux[kAuxBytes];
  const u32 lane = threadIdx.x & 63u, c = threadIdx.x & 31u;
  const u32 tile = blockIdx.x / nsb, sb = blockIdx.x - tile * nsb;
  f32x4 v[4][2];
#pragma unroll
  for (u32 i = 0; i < 4; ++i) {
    const u32 token = tile * kTile + 8u * i + (threadIdx.x >> 5);
    const f32x4* src = reinterpret_cast<const f32x4*>(a + (static_cast<size_t>(min(token, m - 1u)) * nsb + sb) * 256u + 8u * c);
    v[i][0] = src[0];
    v[i][1] = src[1];
  }
#pragma unroll
  for (u32 i = 0; i < 4; ++i) {
    const u32 token = 8u * i + (threadIdx.x >> 5);
    const bool live = tile * kTile + token < m;
    float x[8] = {v[i][0].x, v[i][0].y, v[i][0].z, v[i][0].w, v[i][1].x, v[i][1].y, v[i][1].z, v[i][1].w};
    u32 amax = 0u;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = live ? x[e] : 0.0f;
      amax = max(amax, __float_as_uint(x[e]) & 0x7FFFFFFFu);
    }
    amax = max(amax, static_cast<u32>(__builtin_amdgcn_update_dpp(0, static_cast<int>(amax), 0xB1, 0xF, 0xF, true)));
    amax = max(amax, static_cast<u32>(__builtin_amdgcn_update_dpp(0, static_cast<int>(amax), 0x4E, 0xF, 0xF, true)));
    amax = max(amax, static_cast<u32>(__builtin_amdgcn_update_dpp(0, static_cast<int>(amax), 0x141, 0xF, 0xF, true)));
    amax = max(amax, static_cast<u32>(__builtin_amdgcn_update_dpp(0, static_cast<int>(amax), 0x140, 0xF, 0xF, true)));
    const u32 r0 = static_cast<u32>(__builtin_amdgcn_readlane(static_cast<int>(amax), 0));
    const u32 r1 = static_cast<u32>(__builtin_amdgcn_readlane(static_cast<int>(amax), 16));
    const u32 r2 = static_cast<u32>(__builtin_amdgcn_readlane(static_cast<int>(amax), 32));
    const u32 r3 = static_cast<u32>(__builtin_amdgcn_readlane(static_cast<int>(amax), 48));
    amax = lane < 32u ? max(r0, r1) : max(r2, r3);
    u32 eb = amax >> 23;                      // biased exponent of the run's maximum
    const bool finite = eb != 255u;
    eb = eb < 14u ? 14u : eb;                 // keeps both powers of two normal
    const float down = __uint_as_float((268u - eb) << 23);        // 2^-E = 2^(141 - eb): the maximum comes to [2^14, 2^15)
    _Float16 hi[8], lo[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) split_f16(x[e] * down, hi[e], lo[e]);
    const u32 j = c >> 2, g = j >> 2, h = j & 1u, u = 4u * ((j & 3u) >> 1) + (c & 3u), q = 2u * u + h;
    const u32x4 ph = {pack_h2(hi[0], hi[2]), pack_h2(hi[1], hi[3]), pack_h2(hi[4], hi[6]), pack_h2(hi[5], hi[7])};
    const u32x4 pl = {pack_h2(lo[0], lo[2]), pack_h2(lo[1], lo[3]), pack_h2(lo[4], lo[6]), pack_h2(lo[5], lo[7])};
    *reinterpret_cast<u32x4*>(s_page + 2u * q * kPageStride + (32u * g + token) * 16u) = pl;
    *reinterpret_cast<u32x4*>(s_page + (2u * q + 1u) * kPageStride + (32u * g + token) * 16u) = ph;
    // the sub-block's sum out of the pieces (eleven significant bits each: thirty-two of similar size add up without rounding)
    const h16x2 ones = {static_cast<_Float16>(1.0f), static_cast<_Float16>(1.0f)};
    float sh = __builtin_amdgcn_fdot2(as_h16x2(ph.x), ones, 0.0f, false), sl = __builtin_amdgcn_fdot2(as_h16x2(pl.x), ones, 0.0f, false);
    sh = __builtin_amdgcn_fdot2(as_h16x2(ph.y), ones, sh, false); sl = __builtin_amdgcn_fdot2(as_h16x2(pl.y), ones, sl, false);
    sh = __builtin_amdgcn_fdot2(as_h16x2(ph.z), ones, sh, false); sl = __builtin_amdgcn_fdot2(as_h16x2(pl.z), ones, sl, false);
    sh = __builtin_amdgcn_fdot2(as_h16x2(ph.w), ones, sh, false); sl = __builtin_amdgcn_fdot2(as_h16x2(pl.w), ones, sl, false);
    sh += dpp_f32<0xB1>(sh); sl += dpp_f32<0xB1>(sl);
    sh += dpp_f32<0x4E>(sh); sl += dpp_f32<0x4E>(sl);      // the four threads of a sub-block hold its sums
    const float sj = fmaf(sl, 0.00048828125f, sh) * 0.03125f;
    if ((c & 3u) == 0u) {
      _Float16 s_hi, s_lo;
      split_f16(sj, s_hi, s_lo);
      _Float16* dst = reinterpret_cast<_Float16*>(s_aux + (32u * g + token) * 16u) + ((j & 1u) * 2u + ((j >> 1) & 1u));
      dst[0] = s_hi;
      dst[4] = s_lo;
    }
    if (c == 0u) *reinterpret_cast<u32*>(s_aux + 1024u + 4u * token) = finite ? (eb << 23) : 0x7FC00000u;
  }
  if (threadIdx.x < 56u) *reinterpret_cast<u32x4*>(s_aux + 1152u + 16u * threadIdx.x) = u32x4{0u, 0u, 0u, 0u};      // the padding
  __syncthreads();
  u32x4* out = reinterpret_cast<u32x4*>(ops + static_cast<size_t>(blockIdx.x) * kOperandBytes);
#pragma unroll
  for (u32 i = 0; i < 8; ++i) {
    const u32 at = 256u * i + threadIdx.x;
    out[at] = *reinterpret_cast<const u32x4*>(s_page + (at >> 6) * kPageStride + (at & 63u) * 16u);
  }
  if (threadIdx.x < kAuxBytes / 16u) out[2048u + threadIdx.x] = *reinterpret_cast<const u32x4*>(s_aux + 16u * threadIdx.x);
}

// ---- the product ----
__device__ __forceinline__ void buffer_dma16(__amdgpu_buffer_rsrc_t rsrc, u32 lds_addr, u32 voffset, u32 soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(uintptr_t)lds_addr, 16, static_cast<int>(voffset),
                                           static_cast<int>(soffset), 0, 0);
}
// the bytes 0 and 2 (1 and 3) of a word as f16 numbers
__device__ __forceinline__ h16x2 bytes_to_h2(u32 v) {
  const h16x2 k1024 = {static_cast<_Float16>(1024.0f), static_cast<_Float16>(1024.0f)};
  return as_h16x2((v & 0x00FF00FFu) | 0x64006400u) - k1024;
}
__device__ __forceinline__ h16x2 h2(float v) { return h16x2{static_cast<_Float16>(v), static_cast<_Float16>(v)}; }

// weight tile in LDS: STRIDE bytes a row (an odd number of 16-byte pieces), COPIES of 64 pieces for a wave's rows; STAGES chunks of tokens
template <int FMT, int RT> struct Layout {
  static constexpr u32 SB = FMT == FMT_Q4K ? 144u : 176u, STRIDE = SB, PIECES = SB / 16u, COPIES = (32u * RT * PIECES + 63u) / 64u, STAGES = RT == 1 ? 3u : 4u;
};

template <class F, int... I>
__device__ __forceinline__ void for_each_product(F& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }

// Which tile a workgroup takes.  A run of ids per XCD, and inside it blocks of eight groups of rows against all token
// tiles: the workgroups that run together on an XCD share both operands in its L2.
struct Place {
  u32 part, group, tile;
  bool valid;
  __device__ __forceinline__ Place(u32 id, u32 groups, u32 tiles, u32 kparts) {
    const u32 total = groups * tiles * kparts, per_xcd = (total + 7u) / 8u, lin0 = (id & 7u) * per_xcd + (id >> 3);
    valid = (id >> 3) < per_xcd && lin0 < total;
    part = lin0 / (groups * tiles);
    const u32 lin = lin0 - part * groups * tiles, blk = lin / (8u * tiles), rem = lin - blk * 8u * tiles, width = min(8u, groups - 8u * blk);
    tile = rem / width;
    group = 8u * blk + rem - tile * width;
  }
};

// lane l holds W row row (of strips 32 apart) and the tokens 8 (v / 4) + 4 g + v % 4 of a tile; sum i is strip i / TT, tile i % TT
template <int RT, int TT>
__device__ __forceinline__ void store_tiles(const f32x16 (&sum)[2], float* __restrict__ out, u32 m, u32 n, u32 row, u32 token0, u32 g) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (row + 32u * (i / TT) < n) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const u32 token = token0 + kTile * (i % TT) + 8u * (v >> 2) + 4u * g + (v & 3);
        if (token < m) out[static_cast<size_t>(token) * n + row + 32u * (i / TT)] = sum[i][v];
      }
    }
  }
}

// The running sums are put by; LOSSLESS: what the sum of both rounds away starts the next run, so that the length of a part costs no
// exactness (Q6_K 4096 x 11008 in one part instead of two: 4 % above the error of two without, 5 % below with it).  Q4_K, whose vector instructions weigh
// more beside its products, would lose 2 % of its time to it and does without.
template <bool LOSSLESS>
__device__ __forceinline__ void put_by(f32x16& stash, f32x16& tot) {
  __builtin_amdgcn_sched_barrier(0);      // (nothing else is alive here)
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const float s = stash[v] + tot[v], b = s - stash[v], rest = (stash[v] - (s - b)) + (tot[v] - b);
    tot[v] = LOSSLESS && rest == rest ? rest : 0.0f;      // (a sum that is infinite stays so: what it rounds away is no number)
    stash[v] = s;
  }
  __builtin_amdgcn_sched_barrier(0);
}

// the copies of both bodies: a chunk in LDS is [tile][product][lo, hi][64 lanes], 8 KB a tile, of which wave w brings product w
template <int TT>
struct TokenCopies {
  static constexpr u32 kChunk = TT * 8192u;
  static constexpr int kCopies = 2 * TT;      // of a wave's share of a chunk
  __amdgpu_buffer_rsrc_t rsrc;
  u32 lane16, wave, tile_bytes, ring, aux;
  // (a second tile that is not there: the first one again, its results are not stored)
  __device__ __forceinline__ TokenCopies(const uint8_t* ops, u32 tiles, u32 m, u32 nsb, u32 sb0, u32 ns, u32 lane, u32 wave_, u32 ring_, u32 aux_)
      : lane16(lane * 16u), wave(wave_), tile_bytes(TT == 2 && (TT * tiles + 1u) * kTile < m ? nsb * kOperandBytes : 0u), ring(ring_), aux(aux_) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(ops) + (static_cast<size_t>(tiles) * TT * nsb + sb0) * kOperandBytes, 0,
                                             static_cast<int>(tile_bytes + ns * kOperandBytes), 0x00020000);
  }
  __device__ __forceinline__ void chunk(u32 s, u32 c, u32 slot) const {
#pragma unroll
    for (u32 t = 0; t < TT; ++t) {
      const u32 src = s * kOperandBytes + t * tile_bytes + c * 8192u + wave * 2048u, dst = ring + slot * kChunk + t * 8192u + wave * 2048u;
      buffer_dma16(rsrc, dst, lane16, src);
      buffer_dma16(rsrc, dst + 1024u, lane16, src + 1024u);
    }
  }
  __device__ __forceinline__ void sums(u32 s, u32 buf) const {      // the tiles' aux, a KB a wave (one tile: by two waves and, for one count of copies, by the others as well)
    const u32 t = TT == 2 ? wave >> 1 : 0u;
    buffer_dma16(rsrc, aux + buf * (TT * kAuxBytes) + t * kAuxBytes + (wave & 1u) * 1024u, lane16, s * kOperandBytes + t * tile_bytes + kPagesBytes + (wave & 1u) * 1024u);
  }
};
// keeps an asm's outputs behind the wait in front of this
template <class T> __device__ __forceinline__ void landed(T& v) { asm volatile("" : "+v"(v)::"memory"); }

// dynamic LDS: the ring of chunks, two aux pages, a weight tile per wave (tall_lds_bytes of the runtime)
template <int FMT, int RT, int TT>
__device__ __forceinline__ void body(const uint8_t* __restrict__ ops, const uint8_t* __restrict__ w, float* __restrict__ c,
                                     u32 m, u32 n, u32 nsb, u32 ksb, u32 kparts, u32 groups, u32 pairs, u32 run, u32 lds_base) {
  static_assert(RT * TT == 2, "");
  using L = Layout<FMT, RT>;
  using Tokens = TokenCopies<TT>;
  constexpr u32 kWaveRows = 32u * RT;
  constexpr int S = static_cast<int>(L::STAGES), TD = Tokens::kCopies, WD = static_cast<int>(L::COPIES);
  const u32 lane = threadIdx.x & 63u;
  const u32 wave = static_cast<u32>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
  const Place at(blockIdx.x, groups, pairs, kparts);
  if (!at.valid) return;
  const u32 sb0 = at.part * ksb, ns = min(ksb, nsb - sb0);
  const u32 col = lane & 31u, g = lane >> 5;
  const u32 row0 = at.group * (kWaves * kWaveRows) + wave * kWaveRows;
  const size_t row_bytes = static_cast<size_t>(nsb) * L::SB;

  const u32 lds_ring = lds_base, lds_aux = lds_base + S * Tokens::kChunk;
  const u32 lds_w = lds_aux + 2u * TT * kAuxBytes + wave * (WD * 1024u);

  u32 woff[WD];
  const u32 row_first = min(row0, n - 1u);
#pragma unroll
  for (int t = 0; t < WD; ++t) {
    const u32 p = min(64u * t + lane, kWaveRows * L::PIECES - 1u), r = p / L::PIECES, cc = p - L::PIECES * r;
    woff[t] = (min(row0 + r, n - 1u) - row_first) * static_cast<u32>(row_bytes) + 16u * cc;
  }
  // copies into LDS by buffer instructions: the lane's offset stays in its register, what moves is scalar
  const u32 strip_bytes = (min(row0 + kWaveRows, max(n, row0 + 1u)) - row0) * static_cast<u32>(row_bytes) - sb0 * L::SB;
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(w) + static_cast<size_t>(row_first) * row_bytes + static_cast<size_t>(sb0) * L::SB, 0, static_cast<int>(strip_bytes), 0x00020000);
  auto issue_w = [&](u32 s) {
#pragma unroll
    for (int t = 0; t < WD; ++t) buffer_dma16(w_rsrc, lds_w + 1024u * t, woff[t], s * L::SB);
  };
  const Tokens tokens(ops, at.tile, m, nsb, sb0, ns, lane, wave, lds_ring, lds_aux);

  // where Q4_K keeps a lane's four scales and mins: for the last four sub-blocks the upper two bits lie apart
  [[maybe_unused]] const u32 sc_up = g ? 2u : 0u, sc_mask = g ? 0x30303030u : 0x3F3F3F3Fu, sc_rest = g ? 0x0F0F0F0Fu : 0u;
  f32x16 tot[2], stash[2];
  const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < 2; ++i) tot[i] = stash[i] = zero;

  // chunks 0 .. S-1 of the run, behind the first weight tile and aux pages
  issue_w(0);
  tokens.sums(0, 0);
#pragma unroll
  for (int i = 0; i < S; ++i) tokens.chunk(min(i / 4u, ns - 1u), i & 3, i);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  asm volatile("s_barrier" ::: "memory");
  u32 slot = 0;      // of the chunk being multiplied
  u32 left = run;    // super-blocks until the running sums are put by
  for (u32 s = 0; s < ns; ++s) {
    const u32 wt = lds_w + col * L::STRIDE;
    const u32 aux = lds_aux + (s & 1u) * (TT * kAuxBytes);
    // the weight tile has landed: behind its copies those of two chunks, the last of which may be on its way
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(TD) : "memory");
    u32x4 raw[2][RT], hdr[RT], tok[2][TT][2];
    [[maybe_unused]] u32x4 qh[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      lds_read128<0>(hdr[r], wt + 32u * r * L::STRIDE);
      lds_read128<16>(raw[0][r], wt + 32u * r * L::STRIDE + g * 64u);
      if constexpr (FMT == FMT_Q5K) lds_read128<144>(qh[r], wt + 32u * r * L::STRIDE + g * 16u);
    }
    auto read_tokens = [&](int buf, u32 sl, auto page_c) {
      constexpr int PAGE = decltype(page_c)::value;
      const u32 at = lds_ring + sl * Tokens::kChunk + lane * 16u;
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        lds_read128<PAGE * 2048>(tok[buf][t][0], at + 8192u * t);
        lds_read128<PAGE * 2048 + 1024>(tok[buf][t][1], at + 8192u * t);
      }
    };
    read_tokens(0, slot, std::integral_constant<int, 0>{});
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * TT) : "memory");
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      landed(hdr[r]);
      landed(raw[0][r]);
      if constexpr (FMT == FMT_Q5K) landed(qh[r]);
    }
    h16x2 scale[RT][2], addend[RT][2], mins[RT][2];      // sub-blocks 0 and 2 (low nibbles), 1 and 3 (high nibbles) of the lane's four
    float d[RT], nm[RT];
    constexpr float kCentre = FMT == FMT_Q4K ? 8.0f : 16.0f;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const u32x4 hd = hdr[r];
      u32 s4, m4;
      d[r] = half_bits_to_f32(hd.x);
      nm[r] = half_bits_to_f32(hd.x >> 16) * -0.001953125f;       // -dmin * 2^-9: the sums carry 2^-5, the products 2^-14
      if constexpr (FMT == FMT_Q4K) {      // get_scale_min_k4, quantize.rs:1306-1385
        s4 = ((hd.y >> sc_up) & sc_mask) | (hd.w & sc_rest);
        m4 = ((hd.z >> sc_up) & sc_mask) | ((hd.w >> 4) & sc_rest);
      } else {                             // eight contiguous 12-bit fields, scale in the low six bits (quantize.rs:1607-1635)
        const u32 lo = g ? ((hd.z >> 16) | (hd.w << 16)) : hd.y;
        const u32 hi = g ? (hd.w >> 16) : (hd.z & 0xFFFFu);
        const u32 f0 = lo & 0xFFFu, f1 = (lo >> 12) & 0xFFFu, f2 = ((lo >> 24) | (hi << 8)) & 0xFFFu, f3 = (hi >> 4) & 0xFFFu;
        s4 = (f0 & 63u) | ((f1 & 63u) << 8) | ((f2 & 63u) << 16) | ((f3 & 63u) << 24);
        m4 = (f0 >> 6) | ((f1 >> 6) << 8) | ((f2 >> 6) << 16) | ((f3 >> 6) << 24);
      }
      const h16x2 s02 = bytes_to_h2(s4), s13 = bytes_to_h2(s4 >> 8);
      scale[r][0] = s02 * h2(1024.0f);
      scale[r][1] = s13 * h2(64.0f);
      addend[r][0] = s02 * h2(-kCentre * 0.00006103515625f);
      addend[r][1] = s13 * h2(-kCentre * 0.00006103515625f);
      mins[r][0] = bytes_to_h2(m4);
      mins[r][1] = bytes_to_h2(m4 >> 8);
    }
    // weight operand of product q (0..15), out of the four dwords of its chunk
    auto build = [&](int r, int q, const u32x4& rw) -> h16x8 {
      const int u = q >> 1, h = q & 1;
      const u32 t0 = (u & 1) ? rw.z : rw.x, t1 = (u & 1) ? rw.w : rw.y;
      const _Float16 sv = scale[r][h][u >> 2], av = addend[r][h][u >> 2];
      const h16x2 sc = {sv, sv}, ad = {av, av};
      const u32 mask = h ? 0x00F000F0u : 0x000F000Fu;
      u32 f[4] = {0u, 0u, 0u, 0u};
      if constexpr (FMT == FMT_Q5K) {      // the fifth bits (kquant_gemm_f16.hip.h)
        const u32 word = u < 4 ? (h ? qh[r].y : qh[r].x) : (h ? qh[r].w : qh[r].z);
#pragma unroll
        for (int dd = 0; dd < 2; ++dd) {
          const u32 nb = (word >> (4 * ((2 * u + dd) & 7))) & 15u;
          f[2 * dd] = h ? (__umul24(nb, 0x400100u) & 0x01000100u) : (__umul24(nb, 0x40010u) & 0x00100010u);
          f[2 * dd + 1] = h ? (__umul24(nb, 0x200080u) & 0x01000100u) : (__umul24(nb, 0x20008u) & 0x00100010u);
        }
      }
      const u32x4 o = {__builtin_bit_cast(u32, pk_fma_h2((t0 & mask) | f[0], sc, ad)), __builtin_bit_cast(u32, pk_fma_h2(((t0 >> 8) & mask) | f[1], sc, ad)),
                       __builtin_bit_cast(u32, pk_fma_h2((t1 & mask) | f[2], sc, ad)), __builtin_bit_cast(u32, pk_fma_h2(((t1 >> 8) & mask) | f[3], sc, ad))};
      return __builtin_bit_cast(h16x8, o);
    };
    h16x8 frag[2][RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) frag[0][r] = build(r, 0, raw[0][r]);
    f32x16 acc[2], low[2];      // of the hi and of the lo pieces
    auto step = [&](auto i_c) {
      constexpr int I = decltype(i_c)::value, CH = I / 4, B = I & 1;
      if constexpr (I % 4 == 2 && CH < 3)      // the next chunk's weight dwords
#pragma unroll
        for (int r = 0; r < RT; ++r) lds_read128<16 + 16 * (CH + 1)>(raw[(CH + 1) & 1][r], wt + 32u * r * L::STRIDE + g * 64u);
      auto tokens_landed = [&]() {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          landed(tok[B][t][0]);
          landed(tok[B][t][1]);
        }
      };
      if constexpr (I % 4 == 3) {
        // everything of this chunk is in registers: on to the next one, as soon as every wave is there
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        tokens_landed();
        if constexpr (CH < 3)
#pragma unroll
          for (int r = 0; r < RT; ++r) landed(raw[(CH + 1) & 1][r]);
        constexpr int X = CH + 1;                            // chunk X has landed: S - 2 chunks behind it, and what went out with them
        constexpr bool W_BEHIND = X == 4 && S >= 3;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * TD + (W_BEHIND ? WD + 1 : 0)) : "memory");
        asm volatile("s_barrier" ::: "memory");
        if constexpr (X == 3) {      // the last of this weight tile is in registers: its place takes the next one
          issue_w(min(s + 1u, ns - 1u));
          tokens.sums(min(s + 1u, ns - 1u), (s + 1u) & 1u);
        }
        constexpr int NX = CH + S;                           // chunk CH + S takes this chunk's place
        tokens.chunk(min(s + NX / 4u, ns - 1u), NX & 3, slot);
        slot = slot + 1u == S ? 0u : slot + 1u;
      }
      if constexpr (I < 15) read_tokens(1 - B, slot, std::integral_constant<int, (I + 1) & 3>{});
      if constexpr (I % 4 != 3) {
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * TT) : "memory");
        tokens_landed();
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = i / TT, t = i % TT;
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h16x8, tok[B][t][1]), frag[B][r], I == 0 ? zero : acc[i], 0, 0, 0);
        low[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h16x8, tok[B][t][0]), frag[B][r], I == 0 ? zero : low[i], 0, 0, 0);
        if constexpr (I < 15)
          if (t == TT - 1) frag[1 - B][r] = build(r, I + 1, raw[((I + 1) / 4) & 1][r]);
      }
    };

    __builtin_amdgcn_s_setprio(1);
    for_each_product(step, std::make_integer_sequence<int, 16>{});
    __builtin_amdgcn_s_setprio(0);
    // what the centring took out, then the min term, then the super-block's share of the running sums
    {
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        u32x4 sx, f0, f1, f2, f3;
        const u32 at_t = aux + t * kAuxBytes;
        lds_read128<0>(sx, at_t + lane * 16u);
        lds_read128<1024>(f0, at_t + g * 16u);          // 2^(E+14) of the tokens 8 a + 4 g + {0..3}, a = 0..3
        lds_read128<1056>(f1, at_t + g * 16u);
        lds_read128<1088>(f2, at_t + g * 16u);
        lds_read128<1120>(f3, at_t + g * 16u);
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(sx), "+v"(f0), "+v"(f1), "+v"(f2), "+v"(f3)::"memory");
        const u32 fb[16] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w, f2.x, f2.y, f2.z, f2.w, f3.x, f3.y, f3.z, f3.w};
        const h16x8 sv = __builtin_bit_cast(h16x8, sx);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const int i = r * TT + t;
          // C s_j 2^-9 and m_j against the sums' hi pieces (slots 0..3 of a lane), then against their lo pieces (4..7)
          const u32 c0 = __builtin_bit_cast(u32, addend[r][0] * h2(-32.0f)), c1 = __builtin_bit_cast(u32, addend[r][1] * h2(-32.0f));
          const u32 m0 = __builtin_bit_cast(u32, mins[r][0]), m1 = __builtin_bit_cast(u32, mins[r][1]);
          const u32x4 ch = {c0, c1, 0u, 0u}, cl = {0u, 0u, c0, c1}, mh = {m0, m1, 0u, 0u}, ml = {0u, 0u, m0, m1};
          const float d_lo = d[r] * 0.00048828125f, nm_lo = nm[r] * 0.00048828125f;
          const f32x16 mch = __builtin_amdgcn_mfma_f32_32x32x16_f16(sv, __builtin_bit_cast(h16x8, mh), zero, 0, 0, 0);
          const f32x16 mcl = __builtin_amdgcn_mfma_f32_32x32x16_f16(sv, __builtin_bit_cast(h16x8, ml), zero, 0, 0, 0);
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sv, __builtin_bit_cast(h16x8, ch), acc[i], 0, 0, 0);
          low[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sv, __builtin_bit_cast(h16x8, cl), low[i], 0, 0, 0);
          // (what the lo pieces gave comes first: next to no rounding is added at the size of the whole)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            tot[i][v] = fmaf(__uint_as_float(fb[v]), fmaf(d[r], acc[i][v], fmaf(nm[r], mch[v], fmaf(nm_lo, mcl[v], d_lo * low[i][v]))), tot[i][v]);
          __builtin_amdgcn_sched_barrier(0);      // (both at once would spill)
        }
      }
    }
    if (--left == 0u) {      // runs of super-blocks are summed by themselves: fewer roundings at the size of the whole
      left = run;
#pragma unroll
      for (int i = 0; i < 2; ++i) put_by<FMT == FMT_Q5K>(stash[i], tot[i]);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the copies asked for ahead of the end land before the workgroup's LDS is another's
#pragma unroll
  for (int i = 0; i < 2; ++i) stash[i] += tot[i];
  store_tiles<RT, TT>(stash, c + static_cast<size_t>(at.part) * m * n, m, n, row0 + col, at.tile * (TT * kTile), g);
}

// Q6_K: w = (q - 32) sc needs 13 bits, f16 holds 11.  Centred digits q - 32 = 8 (2 q2 - 3) + (nib - 8) as in
// kquant_gemm_f16.hip.h, but three products a step instead of four: the large digit with the hi pieces in one sum (small
// whole numbers, so that its partial sums hardly round), and in a second one, a quarter of its size, the small digit with
// the hi pieces and the whole weight rounded to f16 with the lo pieces.  Rounding leaves out at most 1 of odd weights above
// 2048, 2^-11 of w, against pieces of at most 2^-11 of the value: 2^-22 of such a term, which the sums' rounding covers
// (error 0.82 .. 0.93 times the 16-token kernel's on activations in use; where all but one in 64 activations are zero and
// little is added up, 1.07 times).  The two digits apart against the lo pieces, a fourth product, would be exact and
// take 8-10 % longer (4096 x 11008, 512 tokens: 212 -> 230 us).  Blocks of 210 bytes lie in LDS 224 apart: thirteen pieces,
// then the block's last sixteen bytes (d at 222); nothing behind a block is read.
constexpr u32 kQ6Stride = 224u, kQ6Pieces = 14u;

__device__ __forceinline__ void q6k_body(const uint8_t* __restrict__ ops, const uint8_t* __restrict__ w, float* __restrict__ c,
                                         u32 m, u32 n, u32 nsb, u32 ksb, u32 kparts, u32 groups, u32 pairs, u32 run, u32 lds_base) {
  using Tokens = TokenCopies<2>;
  constexpr int kTiles = 2, TD = Tokens::kCopies, WD = 7;             // 32 rows x 14 pieces
  constexpr u32 kWaveRows = 32u;
  const u32 lane = threadIdx.x & 63u;
  const u32 wave = static_cast<u32>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
  const Place at(blockIdx.x, groups, pairs, kparts);
  if (!at.valid) return;
  const u32 sb0 = at.part * ksb, ns = min(ksb, nsb - sb0);
  const u32 col = lane & 31u, g = lane >> 5;
  const u32 row0 = at.group * (kWaves * kWaveRows) + wave * kWaveRows;
  const size_t row_bytes = static_cast<size_t>(nsb) * 210u;
  const u32 lds_ring = lds_base, lds_aux = lds_base + 2u * Tokens::kChunk;
  const u32 lds_w = lds_aux + 2u * kTiles * kAuxBytes + wave * (kWaveRows * kQ6Stride);

  u32 woff[WD];
  const u32 row_first = min(row0, n - 1u);
#pragma unroll
  for (int t = 0; t < WD; ++t) {
    const u32 p = 64u * t + lane, r = p / kQ6Pieces, cc = p - kQ6Pieces * r;
    woff[t] = (min(row0 + r, n - 1u) - row_first) * static_cast<u32>(row_bytes) + min(16u * cc, 194u);
  }
  const uint8_t* wbase = w + static_cast<size_t>(row_first) * row_bytes + static_cast<size_t>(sb0) * 210u;
  auto issue_w = [&](u32 s) {
    const uint8_t* src = wbase + static_cast<size_t>(s) * 210u;
#pragma unroll
    for (int t = 0; t < WD; ++t) dma16(src + woff[t], lds_w + 1024u * t);
  };
  const Tokens tokens(ops, at.tile, m, nsb, sb0, ns, lane, wave, lds_ring, lds_aux);
  const u32 lane16 = lane * 16u;

  f32x16 tot[kTiles], stash[kTiles];
  const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < kTiles; ++t) tot[t] = stash[t] = zero;
  issue_w(0);
  tokens.sums(0, 0);
  tokens.chunk(0, 0, 0);
  tokens.chunk(0, 1, 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  asm volatile("s_barrier" ::: "memory");
  u32 left = run;
  for (u32 s = 0; s < ns; ++s) {
    const u32 wt = lds_w + col * kQ6Stride;
    const u32 aux = lds_aux + (s & 1u) * (kTiles * kAuxBytes);
    // the weight tile has landed: only the copies of a chunk are behind its own
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(TD) : "memory");
    u32x4 ql[2][2], qh[2], tok[2][kTiles][2];      // [set of this or the next chunk]
    u32x2 scv;
    u32 dv;
    auto read_raw = [&](auto c_c) {      // of chunk c
      constexpr int C = decltype(c_c)::value, SET = C & 1;
      lds_read128<16 * SET>(ql[SET][0], wt + g * 64u);
      lds_read128<32 + 16 * SET>(ql[SET][1], wt + g * 64u);
      lds_read128<128 + 16 * SET>(qh[SET], wt + g * 32u);
    };
    auto read_tokens = [&](int buf, u32 sl, auto page_c) {
      constexpr int PAGE = decltype(page_c)::value;
      const u32 at = lds_ring + sl * Tokens::kChunk + lane16;
      lds_read128<PAGE * 2048>(tok[buf][0][0], at);
      lds_read128<PAGE * 2048 + 1024>(tok[buf][0][1], at);
      lds_read128<PAGE * 2048 + 8192>(tok[buf][1][0], at);
      lds_read128<PAGE * 2048 + 8192 + 1024>(tok[buf][1][1], at);
    };
    lds_read64<192>(scv, wt + g * 8u);
    asm volatile("ds_read_u16 %0, %1 offset:222" : "=&v"(dv) : "v"(wt) : "memory");
    read_raw(std::integral_constant<int, 0>{});
    read_raw(std::integral_constant<int, 1>{});      // (chunks 2 and 3 are the high nibbles of the same words)
    read_tokens(0, 0u, std::integral_constant<int, 0>{});
    asm volatile("s_waitcnt lgkmcnt(%8)" : "+v"(scv), "+v"(dv), "+v"(ql[0][0]), "+v"(ql[0][1]), "+v"(qh[0]), "+v"(ql[1][0]), "+v"(ql[1][1]), "+v"(qh[1]) : "n"(2 * kTiles) : "memory");
    const float d = half_bits_to_f32(dv);
    h16x2 scale[4];      // chunk c: sc of its products with H = 0 and 1
    {
      const u32 x = scv.x ^ 0x80808080u, y = scv.y ^ 0x80808080u;
      scale[0] = as_h16x2((x & 0x00FF00FFu) | 0x64006400u) - h2(1152.0f);
      scale[1] = as_h16x2(((x >> 8) & 0x00FF00FFu) | 0x64006400u) - h2(1152.0f);
      scale[2] = as_h16x2((y & 0x00FF00FFu) | 0x64006400u) - h2(1152.0f);
      scale[3] = as_h16x2(((y >> 8) & 0x00FF00FFu) | 0x64006400u) - h2(1152.0f);
    }
    // (2 q2 - 3) sc 2^-20, (nib - 8) sc 2^-12, the whole weight rounded to f16 2^-23 (2^-11 of the former's scale: lo pieces
    // carry 2^11; what is below 2^-14 is a whole multiple of 2^-24 and exact as a subnormal)
    h16x8 wq, wn, wa;
    auto build = [&](int q) {      // product q = 4 c + 2 i + H
      const int cc = q >> 2, i = (q >> 1) & 1, H = q & 1, hi_nib = cc >> 1, gq = 2 * hi_nib + H, set = cc & 1;
      const u32 t0 = i ? ql[set][H].z : ql[set][H].x, t1 = i ? ql[set][H].w : ql[set][H].y, c0 = i ? qh[set].z : qh[set].x, c1 = i ? qh[set].w : qh[set].y;
      // nibbles to bits 4..7 of their 16-bit lanes, fields to bits 4..5: bytes 0 and 2 first, then 1 and 3
      auto up = [](u32 v, int by) { return by >= 0 ? v << by : v >> -by; };
      const u32 a[4] = {hi_nib ? t0 : t0 << 4, hi_nib ? t0 >> 8 : t0 >> 4, hi_nib ? t1 : t1 << 4, hi_nib ? t1 >> 8 : t1 >> 4};
      const u32 b[4] = {up(c0, 4 - 2 * gq), up(c0, -4 - 2 * gq), up(c1, 4 - 2 * gq), up(c1, -4 - 2 * gq)};
      const h16x2 sn = scale[cc] * h2(256.0f), an = scale[cc] * h2(-0.001953125f);              // -8 * 2^-12
      const h16x2 sq = scale[cc] * h2(2.0f), aq = scale[cc] * h2(-0.00000286102294921875f);    // -3 * 2^-20
      u32 vn[4], vq[4], va[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const h16x2 n2 = pk_fma_h2(a[k] & 0x00F000F0u, h16x2{sn[H], sn[H]}, h16x2{an[H], an[H]});
        const h16x2 q2 = pk_fma_h2(b[k] & 0x00300030u, h16x2{sq[H], sq[H]}, h16x2{aq[H], aq[H]});
        vn[k] = __builtin_bit_cast(u32, n2);
        vq[k] = __builtin_bit_cast(u32, q2);
        va[k] = __builtin_bit_cast(u32, __builtin_elementwise_fma(n2, h2(0.00048828125f), q2));
      }
      wn = __builtin_bit_cast(h16x8, u32x4{vn[0], vn[1], vn[2], vn[3]});
      wq = __builtin_bit_cast(h16x8, u32x4{vq[0], vq[1], vq[2], vq[3]});
      wa = __builtin_bit_cast(h16x8, u32x4{va[0], va[1], va[2], va[3]});
    };
    f32x16 acc[kTiles], low[kTiles];
    // half a super-block's share of the running sums: the shorter the matrix cores' own sums, the less they round (over
    // whole super-blocks the error was 2 % above the 16-token kernel's for K <= 4096)
    auto add_up = [&]() {
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        u32x4 f0, f1, f2, f3;
        const u32 at_t = aux + t * kAuxBytes + g * 16u;
        lds_read128<1024>(f0, at_t);          // 2^(E+14) of the tokens 8 a + 4 g + {0..3}, a = 0..3
        lds_read128<1056>(f1, at_t);
        lds_read128<1088>(f2, at_t);
        lds_read128<1120>(f3, at_t);
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f0), "+v"(f1), "+v"(f2), "+v"(f3)::"memory");
        const u32 fb[16] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w, f2.x, f2.y, f2.z, f2.w, f3.x, f3.y, f3.z, f3.w};
#pragma unroll
        for (int v = 0; v < 16; ++v) tot[t][v] = fmaf(__uint_as_float(fb[v]), fmaf(512.0f * d, acc[t][v], 0.25f * d * low[t][v]), tot[t][v]);      // 2^(E+14)
      }
    };
    auto step = [&](auto i_c) {
      constexpr int I = decltype(i_c)::value, CH = I / 4, B = I & 1, X = CH + 1;
      auto products = [&](int t) {
        const h16x8 lo = __builtin_bit_cast(h16x8, tok[B][t][0]), hi = __builtin_bit_cast(h16x8, tok[B][t][1]);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, wq, I % 8 == 0 ? zero : acc[t], 0, 0, 0);
        low[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, wa, I % 8 == 0 ? zero : low[t], 0, 0, 0);
        low[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, wn, low[t], 0, 0, 0);
      };
      if constexpr (I % 4 == 3) {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(tok[B][0][0]), "+v"(tok[B][0][1]), "+v"(tok[B][1][0]), "+v"(tok[B][1][1])::"memory");
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(X == 4 ? WD + 1 : 0) : "memory");      // chunk X is there
        asm volatile("s_barrier" ::: "memory");
        tokens.chunk(min(s + (CH + 2) / 4u, ns - 1u), (CH + 2) & 3, CH & 1);      // chunk CH + 2 takes this one's place
        if constexpr (X == 3) {      // all of this weight tile is in registers: its place takes the next one
          issue_w(min(s + 1u, ns - 1u));
          tokens.sums(min(s + 1u, ns - 1u), (s + 1u) & 1u);
        }
        if constexpr (I < 15) read_tokens(1 - B, X & 1, std::integral_constant<int, 0>{});
        build(I);
        products(0);
        products(1);
        if constexpr (I == 7 || I == 15) add_up();
      } else {
        read_tokens(1 - B, CH & 1, std::integral_constant<int, (I + 1) & 3>{});
        build(I);
        asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(tok[B][0][0]), "+v"(tok[B][0][1]), "+v"(tok[B][1][0]), "+v"(tok[B][1][1]) : "n"(2 * kTiles) : "memory");
        products(0);
        products(1);
      }
    };
    __builtin_amdgcn_s_setprio(1);
    for_each_product(step, std::make_integer_sequence<int, 16>{});
    __builtin_amdgcn_s_setprio(0);
    if (--left == 0u) {
      left = run;
#pragma unroll
      for (int t = 0; t < kTiles; ++t) put_by<true>(stash[t], tot[t]);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int t = 0; t < kTiles; ++t) stash[t] += tot[t];
  store_tiles<1, 2>(stash, c + static_cast<size_t>(at.part) * m * n, m, n, row0 + col, at.tile * (kTiles * kTile), g);
}

// c = the parts of K in part order
__device__ __forceinline__ void sum_parts_body(float* __restrict__ c, const float* __restrict__ parts, uint64_t mn, u32 kparts) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < mn; i += stride) {
    float s = 0.0f;
    for (u32 p = 0; p < kparts; ++p) s += parts[p * mn + i];
    c[i] = s;
  }
}

}  // namespace gemm_tall
