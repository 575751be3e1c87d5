// Matrix-core k-quant GEMM for a few sequences decoded together (gfx950, v_mfma_f32_16x16x32_f16), up to 48 tokens:
//   C[m x n] = A[m x k] . dequant(W[n x k])^T,  c[row*n + col]      (trueno-gpu/src/kernels/quantize.rs:568-574)
// with the operands of kquant_gemm_f16.hip.h.  There a workgroup's waves share one super-block's token operands and meet at a barrier for every
// super-block, and a matrix of 4096 columns is cut in parts that meet through memory: 5 us to the first barrier, 1.5-2 a super-block, 3.5 for the sum.
//   * Here a workgroup of eight waves takes 16 RT rows of W against 16 tokens, and each wave whole super-blocks of all those rows: wave w the super-blocks
//     w, w + 8, ...: no wave waits for another until the end, where the eight sums meet in LDS.  Half of the products that come here keep K in one
//     part (1508 of 3111 drawn); in the others the parts meet through memory as there: 4096 x 14336 and 4096 x 4096 with 16 tokens take four, 14 super-blocks
//     of the former's for eight waves, so that two have one and six have two.
//   * A wave's activations go to registers in whole lines (with a token's row a lane, sixteen rows 4 K bytes apart, a load instruction took 70
//     cycles: the rows share an L2 channel), are turned in 8 KB of LDS so that a lane holds 64 values of one token, and become the two f16 pieces there; the
//     next super-block's are asked for before that.  Weights come by copies into LDS, two super-blocks ahead where it holds them (RT <= 2).
//     What does not exist is asked for from a buffer of no bytes: the waits are counted by hand, and the count is the same everywhere.
//   * A lane takes a 32-byte piece of the quants, so it needs two of a row's eight scales; the sums of its own sub-blocks come from products with ones.
//   * Bound by vector instructions (RT = 4: 250 to make the pieces, 125 a tile of 16 rows; a matrix instruction of 16 cycles takes 8 of the
//     SIMD's issue from them) and by latency: a launch of 14336 x 4096, 16 tokens, has its first activations at 1.3 us, the first products at 3 to 6.5,
//     two super-blocks a wave done at 12.
//   * Rounding: as there, hi and lo pieces' sums apart; a wave sums few super-blocks, the waves meet in a tree.  Error against fp64 0.95-0.98 of that
//     kernel's over drawn products, 0.57-0.92 of the GEMV engine's (f32 activations) over 150 of two to eight tokens that the engine had.
//   * Measured (us, 16 tokens, that kernel -> this one): Q4_K 14336 x 4096 15.4 -> 14.7, 4096 x 14336 18.4 -> 16.3-17.0, 4096 x 4096 9.9 -> 8.7, 11008 x 4096 14.2 ->
//     13.0; Q5_K 11008 x 4096 16.6 -> 14.9; 3 tokens, Q4_K 12000 x 1024 13.8 -> 5.4 (the integer cores); Q6_K 32000 x 4096 keeps the other (41 against 48).
//   * q5k_gemm_slices_r1 spills 13 registers and reads them back inside the loop; its times, and so the estimate that chooses it (one product in eight of
//     Q5_K), include that.
// (v_mfma_f32_16x16x16_f16, half as long, gave wrong rows in one build where its result lay over its first operand; the cause was not found, and it is not used.)
#pragma once
#include "kquant_gemm_f16.hip.h"

namespace gemm_slices {

using namespace gemm_f16;      // the LDS helpers, dma16, Geometry, pk_fma_h2, kCounterBytes

constexpr u32 kWaves = 8;
constexpr u32 kTurnBytes = 8192;      // LDS in which a wave turns half a super-block of its sixteen tokens' activations

// a row of a super-block in LDS: PIECES sixteen-byte pieces, PITCH bytes apart (Q6_K: thirteen pieces, then the block's last sixteen bytes)
template <int FMT> struct Block;
template <> struct Block<FMT_Q4K> { static constexpr u32 SB = 144, PITCH = 144, PIECES = 9, HEAD = 0; };
template <> struct Block<FMT_Q5K> { static constexpr u32 SB = 176, PITCH = 176, PIECES = 11, HEAD = 0; };
template <> struct Block<FMT_Q6K> { static constexpr u32 SB = 210, PITCH = 224, PIECES = 14, HEAD = 222; };

// RT tiles of 16 rows
template <int FMT, int RT> struct Shape {
  static constexpr u32 ROWS = 16u * RT, COPIES = (ROWS * Block<FMT>::PIECES + 63u) / 64u, STAGE = COPIES * 1024u;
  static constexpr u32 STAGES = kWaves * (2u * STAGE + kTurnBytes) <= 156u * 1024u ? 2u : 1u;
  static constexpr u32 WAVE = STAGES * STAGE + kTurnBytes, LDS = kWaves * WAVE + 16u;      // of a wave, of a workgroup
};

// two values times `down`, and 2^11 times what f16 leaves out of that (up = 2^11 down), as f16 pairs: the two pieces
__device__ __forceinline__ void pieces(float a, float b, float down, float up, u32& hi, u32& lo) {
  hi = opaque(__builtin_bit_cast(u32, h16x2{static_cast<_Float16>(fmaf(a, down, 0.0f)), static_cast<_Float16>(fmaf(b, down, 0.0f))}));
  const h16x2 h = as_h16x2(hi);
  const h16x2 l = {static_cast<_Float16>(fmaf(static_cast<float>(h.x), -2048.0f, a * up)), static_cast<_Float16>(fmaf(static_cast<float>(h.y), -2048.0f, b * up))};
  lo = __builtin_bit_cast(u32, l);
}

// the activations are there when only the copies asked for behind them are outstanding
template <int BEHIND>
__device__ __forceinline__ void wait_landed(u32x4 (&v)[16]) {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(BEHIND) : "memory");
#pragma unroll
  for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(v[i])::"memory");
}

__device__ __forceinline__ f32x4 mfma32(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h16x8, a), __builtin_bit_cast(h16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ u32 pk(h16x2 v) { return __builtin_bit_cast(u32, v); }
__device__ __forceinline__ h16x2 two(float a, float b) { return h16x2{static_cast<_Float16>(a), static_cast<_Float16>(b)}; }

template <int FMT, int RT>
__device__ __forceinline__ void body(const float* __restrict__ a, const uint8_t* __restrict__ w, float* __restrict__ c, uint8_t* __restrict__ ws,
                                     u32 m, u32 n, u32 nsb, uint64_t geom, u32 lds_base) {
  using B = Block<FMT>;
  using S = Shape<FMT, RT>;
  constexpr int COPIES = static_cast<int>(S::COPIES);
  const Geometry cut(geom);
  const u32 ksb = cut.ksb, kparts = cut.kparts, groups = cut.groups, tiles = cut.tiles;
  const u32 lane = threadIdx.x & 63u, col = lane & 15u, g = lane >> 4;
  const u32 wave = static_cast<u32>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
  const u32 id = blockIdx.x;
  const u32 pair = (id / (8u * tiles)) * 8u + (id & 7u), tile = (id >> 3) % tiles;      // the tiles of a (group, part) on one XCD
  if (pair >= groups * kparts) return;
  const u32 group = pair / kparts, part = pair - group * kparts;
  const u32 sb0 = part * ksb, ns = min(ksb, nsb - sb0);
  const u32 row0 = group * S::ROWS, rows = min(S::ROWS, n - row0), token0 = tile * 16u, tokens = min(16u, m - token0);

  // Activations: instruction 8 h + j brings half h (the lanes' fields r = 2 h and 2 h + 1, below) of the tokens 2 j and 2 j + 1, 512 bytes
  // each in whole lines.  Tokens that are not there lie outside the buffer and read as zeros; a buffer of no bytes stands for a
  // super-block that is not there: nothing is read, and the count of loads in flight is the same.
  const uint8_t* a_at = reinterpret_cast<const uint8_t*>(a) + (static_cast<size_t>(token0) * nsb + sb0) * 1024u;
  const u32 u = lane & 31u, odd = lane >> 5;
  // the lane's piece (16 bytes) of a half, and the unit (8 g + 4 (r % 2) + piece of the field) it is to the lane group g that takes it
  const u32 a_piece = FMT == FMT_Q6K ? 512u * (u >> 4) + 16u * (u & 15u) : 256u * (u >> 3) + 16u * (u & 7u);
  const u32 a_unit = FMT == FMT_Q6K ? 16u * (u >> 4) + 8u * ((u >> 2) & 1u) + 4u * ((u >> 3) & 1u) + (u & 3u) : u;
  constexpr int kHalf = FMT == FMT_Q6K ? 256 : 128;
  const u32 a_off = odd * nsb * 1024u + a_piece, a_bytes = (tokens * nsb - sb0) * 1024u;
  u32x4 raw[16];
  auto load_a = [&](u32 s) {
    const u32 there = s < ns ? a_bytes : 0u, at = s < ns ? s * 1024u : 0u;
    const uintptr_t p = reinterpret_cast<uintptr_t>(a_at);
    const u32x4 rsrc = {static_cast<u32>(p), static_cast<u32>(p >> 32) & 0xFFFFu, there, 0x00020000u};
#pragma unroll
    for (u32 j = 0; j < 8; ++j) {
      const u32 off = a_off + j * (2048u * nsb);
      asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen" : "=&v"(raw[j]) : "v"(off), "s"(rsrc), "s"(at) : "memory");
      asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen offset:%4" : "=&v"(raw[8 + j]) : "v"(off), "s"(rsrc), "s"(at), "n"(kHalf) : "memory");
    }
  };
  // Weights: 64 pieces an instruction, as in kquant_gemm_tall.hip.h
  const size_t row_bytes = static_cast<size_t>(nsb) * B::SB;
  u32 woff[COPIES];
#pragma unroll
  for (int t = 0; t < COPIES; ++t) {
    const u32 p = min(64u * t + lane, S::ROWS * B::PIECES - 1u), r = p / B::PIECES, cc = p - B::PIECES * r;
    woff[t] = min(r, rows - 1u) * static_cast<u32>(row_bytes) + min(16u * cc, B::SB - 16u);
  }
  const uint8_t* w_at = w + static_cast<size_t>(row0) * row_bytes + static_cast<size_t>(sb0) * B::SB;
  const u32 w_bytes = rows * static_cast<u32>(row_bytes) - sb0 * B::SB;
  const u32 lds_w = lds_base + wave * S::WAVE, lds_turn = lds_w + S::STAGES * S::STAGE;
  // unit x of token t lies at x ^ t of the token's 32: writes (two tokens an instruction) and reads (sixteen) meet no bank twice
  const u32 turn_in = lds_turn + 512u * odd + 16u * (a_unit ^ odd), turn_out = lds_turn + 512u * col + 16u * ((8u * g) ^ col);
  auto copy_w = [&](u32 s, u32 stage) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(w_at), 0, static_cast<int>(s < ns ? w_bytes : 0u), 0x00020000);
#pragma unroll
    for (int t = 0; t < COPIES; ++t)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(uintptr_t)(lds_w + stage * S::STAGE + 1024u * t), 16,
                                               static_cast<int>(woff[t]), static_cast<int>(s < ns ? s * B::SB : 0u), 0, 0);
  };

  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 tot[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) tot[t] = zero;
  // where Q4_K keeps the scales and mins of the sub-blocks 2 g and 2 g + 1: for the last four the upper two bits lie apart
  [[maybe_unused]] const u32 sc_shift = 16u * (g & 1u), sc_up = g < 2u ? 0u : 2u, sc_mask = g < 2u ? 0x3F3Fu : 0x3030u, sc_rest = g < 2u ? 0u : 0x0F0Fu;
  // selector of the sums: ones in the rows 4 g .. 4 g + 3, so that lane group g of the result holds the sum over its own sub-block
  const u32 one = FMT != FMT_Q6K && (col >> 2) == g ? 0x3C003C00u : 0u;
  const u32x4 sel = {one, one, one, one};

  if (wave < ns) {
    load_a(wave);
    copy_w(wave, 0u);
    if constexpr (S::STAGES == 2) copy_w(wave + kWaves, 1u);
    u32 stage = 0;
    wait_landed<COPIES * static_cast<int>(S::STAGES)>(raw);
    // one super-block; MORE: this wave has another one behind it
    auto unit = [&](u32 s, auto more_c) {
      constexpr bool MORE = decltype(more_c)::value;
      // Field r of a lane: the sixteen values 64 g + 16 r .. (Q6_K: 128 (g / 2) + 32 r + 16 (g % 2) ..) of its token, as v[4 r .. 4 r + 3].
      // (LDS serves a wave's accesses in order: a half's writes, its reads, the other half's)
      u32x4 vb[16];
#pragma unroll
      for (u32 h = 0; h < 2; ++h) {
#pragma unroll
        for (u32 j = 0; j < 8; ++j) asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(turn_in ^ (32u * j)), "v"(raw[8 * h + j]), "n"(1024 * j) : "memory");
#pragma unroll
        for (u32 x = 0; x < 8; ++x) asm volatile("ds_read_b128 %0, %1" : "=&v"(vb[8 * h + x]) : "v"(turn_out ^ (16u * x)) : "memory");
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(vb[i])::"memory");
      if constexpr (MORE) load_a(s + kWaves);      // into the registers that are free now
      f32x4 v[16];
      float top = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        v[i] = __builtin_bit_cast(f32x4, vb[i]);
        top = fmaxf(fmaxf(top, fabsf(v[i].x)), fmaxf(fabsf(v[i].y), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
      }
      {
        const u32 x = __float_as_uint(top);
        const u32x2 p = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(x, x, false, false));
        const u32 y = __float_as_uint(fmaxf(__uint_as_float(p.x), __uint_as_float(p.y)));
        const u32x2 q = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(y, y, false, false));
        top = fmaxf(__uint_as_float(q.x), __uint_as_float(q.y));
      }
      u32 eb = __float_as_uint(top) >> 23;      // biased exponent of the run's maximum (a NaN beside finite values is its own piece)
      const float factor = eb == 255u ? __uint_as_float(0x7FC00000u) : __uint_as_float(max(eb, 25u) << 23);      // 2^(E+14)
      eb = max(eb, 25u);
      const float down = __uint_as_float((268u - eb) << 23), up = __uint_as_float((279u - eb) << 23);      // 2^-E brings the maximum to [2^14, 2^15)
      // operand of step 2 r + u: values 8 u .. 8 u + 7 of v[r], in the order 0,2,1,3,4,6,5,7
      u32x4 hi[8], lo[8];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const f32x4 p = v[4 * r + 2 * u], q = v[4 * r + 2 * u + 1];
          u32 h0, h1, h2, h3, l0, l1, l2, l3;
          pieces(p.x, p.z, down, up, h0, l0);
          pieces(p.y, p.w, down, up, h1, l1);
          pieces(q.x, q.z, down, up, h2, l2);
          pieces(q.y, q.w, down, up, h3, l3);
          hi[2 * r + u] = u32x4{h0, h1, h2, h3};
          lo[2 * r + u] = u32x4{l0, l1, l2, l3};
        }
      [[maybe_unused]] u32x4 sum_hi = {0u, 0u, 0u, 0u}, sum_lo = {0u, 0u, 0u, 0u};
      if constexpr (FMT != FMT_Q6K) {      // sub-blocks 2 g (r = 0, 1) and 2 g + 1 of the lane's token: their sums in the lane, times 2^-5, two pieces each
        f32x4 part[4] = {zero, zero, zero, zero};      // (four chains: one after the other would wait for each other)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          part[0] = mfma32(sel, hi[q], part[0]);
          part[1] = mfma32(sel, lo[q], part[1]);
          part[2] = mfma32(sel, hi[4 + q], part[2]);
          part[3] = mfma32(sel, lo[4 + q], part[3]);
        }
        const f32x4 t = {part[0].x, part[2].x, part[1].x, part[3].x};
        u32 s_hi, s_lo;
        pieces(fmaf(t.z, 0.00048828125f, t.x), fmaf(t.w, 0.00048828125f, t.y), 0.03125f, 64.0f, s_hi, s_lo);
        sum_hi.x = s_hi;
        sum_lo.x = s_lo;
      }
      // the weights are there: behind them the other tile's copies, the next activations
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(!MORE ? 0 : S::STAGES == 2 ? COPIES + 16 : 16) : "memory");
      const u32 wt = lds_w + stage * S::STAGE + col * B::PITCH, wh = lds_w + stage * S::STAGE + 4u * g * B::PITCH + B::HEAD;
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        constexpr u32 kTileBytes = 16u * B::PITCH;
        u32 dd[4];
        f32x4 acc_hi = zero, acc_lo = zero;
        if constexpr (FMT != FMT_Q6K) {
          [[maybe_unused]] u32x4 hd = {0u, 0u, 0u, 0u};
          [[maybe_unused]] u32x2 fields = {0u, 0u};
          u32x4 q0, q1;
          [[maybe_unused]] u32x2 qh = {0u, 0u};
          const u32 wr = wt + t * kTileBytes + 32u * g;
          if constexpr (FMT == FMT_Q4K) lds_read128<0>(hd, wt + t * kTileBytes);
          else      // the words that bytes 4 + 3 g .. of the block lie in
            asm volatile("ds_read2_b32 %0, %1 offset0:1 offset1:2" : "=&v"(fields) : "v"(wt + t * kTileBytes + (3u * g & ~3u)) : "memory");
          lds_read128<16>(q0, wr);
          lds_read128<32>(q1, wr);
          if constexpr (FMT == FMT_Q5K) lds_read64<144>(qh, wt + t * kTileBytes + 8u * g);
#pragma unroll
          for (int e = 0; e < 4; ++e) asm volatile("ds_read_b32 %0, %1 offset:%2" : "=&v"(dd[e]) : "v"(wh + t * kTileBytes), "n"(e * B::PITCH) : "memory");
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(hd), "+v"(fields), "+v"(q0), "+v"(q1), "+v"(qh), "+v"(dd[0]), "+v"(dd[1]), "+v"(dd[2]), "+v"(dd[3])::"memory");
          // scales and mins of the sub-blocks 2 g and 2 g + 1, in the low two bytes
          u32 s2, m2;
          if constexpr (FMT == FMT_Q4K) {      // get_scale_min_k4, quantize.rs:1306-1385
            const u32 x = hd.w >> sc_shift;
            s2 = ((hd.y >> (sc_shift + sc_up)) & sc_mask) | (x & sc_rest);
            m2 = ((hd.z >> (sc_shift + sc_up)) & sc_mask) | ((x >> 4) & sc_rest);
          } else {                             // eight contiguous 12-bit fields, scale in the low six bits (quantize.rs:1607-1635): two are three bytes at 4 + 3 g
            const u32 f = __builtin_amdgcn_alignbit(fields.y, fields.x, 8u * (3u * g & 3u));
            s2 = (f & 63u) | ((f >> 4) & 0x3F00u);
            m2 = ((f >> 6) & 63u) | ((f >> 10) & 0x3F00u);
          }
          const h16x2 k1024 = two(1024.0f, 1024.0f);
          const h16x2 sc2 = as_h16x2(__builtin_amdgcn_perm(0x64646464u, s2, 0x04010400u)) - k1024;
          const h16x2 mn2 = as_h16x2(__builtin_amdgcn_perm(0x64646464u, m2, 0x04010400u)) - k1024;
          constexpr float kCentre = FMT == FMT_Q4K ? 8.0f : 16.0f;
          const h16x2 scale = sc2 * two(1024.0f, 64.0f);
          const h16x2 add = sc2 * two(-kCentre * 0.00006103515625f, -kCentre * 0.00006103515625f);      // -C * s_j * 2^-14
          // C s_j 2^-9 and -m_j 2^-9 against the sums (which carry 2^-5)
          const h16x2 cs = sc2 * two(kCentre * 0.001953125f, kCentre * 0.001953125f), ms = mn2 * two(-0.001953125f, -0.001953125f);
          const h16x2 sl = {scale.x, scale.x}, al = {add.x, add.x}, sg = {scale.y, scale.y}, ag = {add.y, add.y};
          const u32 dw[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const u32 t0 = dw[2 * u], t1 = dw[2 * u + 1], t0s = t0 >> 8, t1s = t1 >> 8;
            u32 f[4] = {0u, 0u, 0u, 0u}, e[4] = {0u, 0u, 0u, 0u};
            if constexpr (FMT == FMT_Q5K) {      // the fifth bits (kquant_gemm_f16.hip.h)
#pragma unroll
              for (int d = 0; d < 2; ++d) {
                const u32 nl = (qh.x >> (8 * u + 4 * d)) & 15u, nh = (qh.y >> (8 * u + 4 * d)) & 15u;
                f[2 * d] = __umul24(nl, 0x40010u) & 0x00100010u;
                f[2 * d + 1] = __umul24(nl, 0x20008u) & 0x00100010u;
                e[2 * d] = __umul24(nh, 0x400100u) & 0x01000100u;
                e[2 * d + 1] = __umul24(nh, 0x200080u) & 0x01000100u;
              }
            }
            const u32x4 wl = {pk(pk_fma_h2((t0 & 0x000F000Fu) | f[0], sl, al)), pk(pk_fma_h2((t0s & 0x000F000Fu) | f[1], sl, al)),
                              pk(pk_fma_h2((t1 & 0x000F000Fu) | f[2], sl, al)), pk(pk_fma_h2((t1s & 0x000F000Fu) | f[3], sl, al))};
            acc_hi = mfma32(wl, hi[u], acc_hi);
            acc_lo = mfma32(wl, lo[u], acc_lo);
            const u32x4 wg = {pk(pk_fma_h2((t0 & 0x00F000F0u) | e[0], sg, ag)), pk(pk_fma_h2((t0s & 0x00F000F0u) | e[1], sg, ag)),
                              pk(pk_fma_h2((t1 & 0x00F000F0u) | e[2], sg, ag)), pk(pk_fma_h2((t1s & 0x00F000F0u) | e[3], sg, ag))};
            acc_hi = mfma32(wg, hi[4 + u], acc_hi);
            acc_lo = mfma32(wg, lo[4 + u], acc_lo);
          }
          acc_hi = mfma32(u32x4{pk(cs), 0u, 0u, 0u}, sum_hi, acc_hi);
          acc_lo = mfma32(u32x4{pk(cs), 0u, 0u, 0u}, sum_lo, acc_lo);
          const f32x4 min_hi = mfma32(u32x4{pk(ms), 0u, 0u, 0u}, sum_hi, zero), min_lo = mfma32(u32x4{pk(ms), 0u, 0u, 0u}, sum_lo, zero);
          // (what the lo pieces gave comes first: next to no rounding is added at the size of the whole)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const h16x2 h = as_h16x2(dd[e]);
            const float lo_part = fmaf(static_cast<float>(h.y), min_lo[e], static_cast<float>(h.x) * acc_lo[e]) * 0.00048828125f;
            tot[t][e] = fmaf(factor, fmaf(static_cast<float>(h.x), acc_hi[e], fmaf(static_cast<float>(h.y), min_hi[e], lo_part)), tot[t][e]);
          }
        } else {
          u32x4 qa, qb, qc;
          u32x2 sv;
          const u32 wr = wt + t * kTileBytes, at = (g >> 1) * 64u + (g & 1u) * 16u;
          lds_read128<0>(qa, wr + at);
          lds_read128<32>(qb, wr + at);
          lds_read128<128>(qc, wr + (g >> 1) * 32u + (g & 1u) * 16u);
          lds_read64<192>(sv, wr + (g >> 1) * 8u);
#pragma unroll
          for (int e = 0; e < 4; ++e) asm volatile("ds_read_u16 %0, %1 offset:%2" : "=&v"(dd[e]) : "v"(wh + t * kTileBytes), "n"(e * B::PITCH) : "memory");
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(qa), "+v"(qb), "+v"(qc), "+v"(sv), "+v"(dd[0]), "+v"(dd[1]), "+v"(dd[2]), "+v"(dd[3])::"memory");
          // scales of the fields r = 0 .. 3: bytes (g % 2) + 2 r
          const u32 sx = ((sv.x ^ 0x80808080u) >> (8u * (g & 1u))) & 0x00FF00FFu, sy = ((sv.y ^ 0x80808080u) >> (8u * (g & 1u))) & 0x00FF00FFu;
          const h16x2 s01 = as_h16x2(sx | 0x64006400u) - two(1152.0f, 1152.0f), s23 = as_h16x2(sy | 0x64006400u) - two(1152.0f, 1152.0f);
          const u32 da[4] = {qa.x, qa.y, qa.z, qa.w}, db[4] = {qb.x, qb.y, qb.z, qb.w}, dh[4] = {qc.x, qc.y, qc.z, qc.w};
          f32x4 accq_hi = zero, accq_lo = zero;
          auto by = [](u32 x, int n) { return n >= 0 ? x << n : x >> -n; };
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const _Float16 sf = r == 0 ? s01.x : r == 1 ? s01.y : r == 2 ? s23.x : s23.y;
            const h16x2 ss = {sf, sf};
            // (nib - 8) sc 2^-14 and (2 q2 - 3) sc 2^-14 out of bits 4 .. 7 and 4 .. 5 of a 16-bit lane (kquant_gemm_f16.hip.h)
            const h16x2 sn = ss * two(64.0f, 64.0f), an = ss * two(-0.00048828125f, -0.00048828125f);
            const h16x2 sq = ss * two(128.0f, 128.0f), aq = ss * two(-0.00018310546875f, -0.00018310546875f);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const u32 t0 = (r & 1) ? db[2 * u] : da[2 * u], t1 = (r & 1) ? db[2 * u + 1] : da[2 * u + 1], c0 = dh[2 * u], c1 = dh[2 * u + 1];
              const u32x4 wn = {pk(pk_fma_h2(by(t0, r < 2 ? 4 : 0) & 0x00F000F0u, sn, an)), pk(pk_fma_h2(by(t0, r < 2 ? -4 : -8) & 0x00F000F0u, sn, an)),
                                pk(pk_fma_h2(by(t1, r < 2 ? 4 : 0) & 0x00F000F0u, sn, an)), pk(pk_fma_h2(by(t1, r < 2 ? -4 : -8) & 0x00F000F0u, sn, an))};
              const u32x4 wq = {pk(pk_fma_h2(by(c0, 4 - 2 * r) & 0x00300030u, sq, aq)), pk(pk_fma_h2(by(c0, -4 - 2 * r) & 0x00300030u, sq, aq)),
                                pk(pk_fma_h2(by(c1, 4 - 2 * r) & 0x00300030u, sq, aq)), pk(pk_fma_h2(by(c1, -4 - 2 * r) & 0x00300030u, sq, aq))};
              acc_hi = mfma32(wn, hi[2 * r + u], acc_hi);
              accq_hi = mfma32(wq, hi[2 * r + u], accq_hi);
              acc_lo = mfma32(wn, lo[2 * r + u], acc_lo);
              accq_lo = mfma32(wq, lo[2 * r + u], accq_lo);
            }
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = fmaf(fmaf(8.0f, accq_lo[e], acc_lo[e]), 0.00048828125f, fmaf(8.0f, accq_hi[e], acc_hi[e]));
            tot[t][e] = fmaf(factor * half_bits_to_f32(dd[e]), x, tot[t][e]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);      // (the next tile's operands ahead of this one's products would spill)
      }
      if constexpr (MORE) {
        copy_w(s + S::STAGES * kWaves, stage);      // (the tile is in registers)
        if constexpr (S::STAGES == 2) stage ^= 1u;
        wait_landed<COPIES>(raw);
      }
    };
    u32 s = wave;
    for (; s + kWaves < ns; s += kWaves) unit(s, std::true_type{});
    unit(s, std::false_type{});
  }

  // The waves' sums meet in LDS, each in its own wave's place; thread i of the first 64 RT takes 16-byte element i:
  // element 64 t + lane: token lane % 16, rows 16 t + 4 (lane / 16) .. + 3
#pragma unroll
  for (int t = 0; t < RT; ++t) asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(lds_w + lane * 16u), "v"(tot[t]), "n"(1024 * t) : "memory");
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  const u32 i = threadIdx.x;
  const bool mine = i < 64u * RT;
  f32x4 sum = zero;
  if (mine) {
    u32x4 x[kWaves];
#pragma unroll
    for (u32 q = 0; q < kWaves; ++q)
      asm volatile("ds_read_b128 %0, %1" : "=&v"(x[q]) : "v"(lds_base + q * S::WAVE + i * 16u) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (u32 q = 0; q < kWaves; ++q) asm volatile("" : "+v"(x[q])::"memory");
    f32x4 f[kWaves];
#pragma unroll
    for (u32 q = 0; q < kWaves; ++q) f[q] = __builtin_bit_cast(f32x4, x[q]);
    sum = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
  }
  const u32 token = token0 + (i & 15u), row = row0 + 16u * (i >> 6) + 4u * ((i >> 4) & 3u);
  auto store = [&]() {
    if (!mine || token >= m) return;
    float* dst = c + static_cast<size_t>(token) * n + row;
    if ((n & 3u) == 0u && (reinterpret_cast<uintptr_t>(c) & 15u) == 0u) {
      if (row < n) *reinterpret_cast<f32x4*>(dst) = sum;
    } else {
#pragma unroll
      for (u32 e = 0; e < 4; ++e)
        if (row + e < n) dst[e] = sum[e];
    }
  };
  if (kparts == 1u) {
    store();
    return;
  }
  // parts of K: published through to memory, added in part order by the workgroup that arrives last (as in kquant_gemm_f16.hip.h)
  u32* counters = reinterpret_cast<u32*>(ws);
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      ws + kCounterBytes, 0, static_cast<int>(kparts * tiles * groups * (RT * 1024u)), 0x00020000);
  auto slot = [&](u32 p) { return static_cast<int>(((p * tiles + tile) * groups + group) * (RT * 1024u) + i * 16u); };
  if (mine) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum), rsrc, slot(part), 0, 16);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");      // the coherent stores have been acknowledged
  const u32 lds_flag = lds_base + kWaves * S::WAVE;
  if (threadIdx.x == 0u) {
    const u32 old = __hip_atomic_fetch_add(counters + group * tiles + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old == kparts - 1u) __hip_atomic_store(counters + group * tiles + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("ds_write_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" ::"v"(lds_flag), "v"(old) : "memory");
  }
  asm volatile("s_barrier" ::: "memory");
  u32 old;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(old) : "v"(lds_flag) : "memory");
  if (old != kparts - 1u || !mine) return;
  sum = zero;
  auto add_parts = [&](auto width) {
    constexpr u32 W = decltype(width)::value;
    for (u32 p0 = 0; p0 < kparts; p0 += W) {
      u32x4 x[W];
#pragma unroll
      for (u32 p = 0; p < W; ++p) x[p] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, slot(min(p0 + p, kparts - 1u)), 0, 16);
#pragma unroll
      for (u32 p = 0; p < W; ++p)
        if (p0 + p < kparts) sum += __builtin_bit_cast(f32x4, x[p]);
    }
  };
  if (kparts <= 2u) add_parts(std::integral_constant<u32, 2>{});
  else if (kparts <= 4u) add_parts(std::integral_constant<u32, 4>{});
  else add_parts(std::integral_constant<u32, 8>{});
  store();
}

}  // namespace gemm_slices
