// Weight-streaming scaled FP8 matmul for small M (decode): C[M,N] = A[M,K] . B[N,K]^T,
// M <= 16 * MT.
//
// The bytes that matter are the N*K weight bytes, read exactly once, so the kernel is
// shaped by what HBM likes (measured on MI355X with read-only kernels: whole 128-byte lines
// per row and long runs per wave reach ~6.2 TB/s on these shapes; half lines taken by
// alternating waves stay at ~4.6 TB/s):
//
//   * a block owns 16*NTW consecutive weight rows; each of its 4 or 8 waves owns a contiguous
//     share of K and walks it in 128-byte slabs;
//   * weight slabs travel by LDS-DMA (`buffer_load_dwordx4 ... lds`), one instruction per
//     8 rows x 128 bytes (whole cache lines), into a ring of DEPTH slots that is private to
//     the wave -- no barrier in the loop, DEPTH slabs of weights in flight per wave;
//   * the MFMA row operand (16 weight rows x 128 K bytes) is read back from LDS with the
//     same conflict-free chunk swizzle as the tiled kernel; the activations are the column
//     operand, loaded straight from global memory / L2 (tokens >= M read as zero through the
//     buffer descriptor): v_mfma_f32_16x16x128_f8f6f4 computes 16 weight rows x 16 tokens
//     per instruction, so M is never padded to a 128-row tile;
//   * the waves' partial sums meet in LDS in a fixed order (deterministic result).
//
// Scaling follows gemm_tiled.hip: block mode promotes every slab with
// a_s[slab, m] * b_s[n/128, slab]; row/tensor mode scales once at the end
// (max/kernels/src/linalg/fp8_quantization.mojo:1218-1240, 1576-1624).
#include <stdlib.h>

#include <type_traits>
#include <utility>

#include "common.h"
#include "gemm_args.h"
#include "tuning.h"

namespace maxfp8 {

typedef __attribute__((address_space(3))) void* sk_lds_ptr_t;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t sk_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
// Cache policy of the weight copies: non-temporal.  A weight byte is read once per launch; marked so, the stream does not
// displace what the memory-side cache and the L2 hold, and the chip reads 7.0 instead of 6.2 TB/s (a read-only kernel,
// one block of eight 16 KB rings per CU, the same matrix with and without the bit).
constexpr int kWeightStream = 2;

__device__ __forceinline__ v4i sk_load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ float sk_load_f32(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ uint32_t sk_clamp_u32(int64_t v) {
  return v > 0xfffffff0ll ? 0xfffffff0u : (v < 0 ? 0u : (uint32_t)v);
}

// ALDS: the activations of a wave's share of K are copied to LDS once, before the loop (at most kSkinnyALdsBytes per
// wave), instead of two loads per slab and 16-token group: on a launch that is a single round of blocks those loads
// are half of the loop's vector-memory instructions and cost 8 % of the kernel, whatever they fetch.
constexpr int kSkinnyALdsBytes = 8192;
// How the activations reach the loop: loaded per slab, copied to LDS before it, or (any larger value) quantised into LDS
// before it from the bf16 activations by the block itself, that many 16-byte loads per lane.
enum SkinnyActs { kActsPerSlab = 0, kActsLds = 1 };
template <int NTW, int MT, bool BLOCKSCALE, int RING_KB, int NWAVES, int ACTS = kActsPerSlab>
struct SkinnyCfg {
  static constexpr bool ALDS = ACTS != kActsPerSlab, QUANT = ACTS > kActsLds;
  static constexpr int WAVES = NWAVES;
  static constexpr int SLOT = NTW * 2048;                    // one slab of the block's rows
  // VMEM instructions a wave issues per slab, in this order: activations, scales, weight DMA
  static constexpr int PER = (ALDS ? 0 : 2 * MT) + (BLOCKSCALE ? (QUANT ? 1 : MT + 1) : 0) + 2 * NTW;
  // slabs in flight per wave: RING_KB of weights, limited by the 6-bit vmcnt counter and by the
  // registers the activation fragments of the in-flight slabs take (96)
  static constexpr int D_BYTES = RING_KB * 1024 / SLOT, D_CNT = 63 / PER + 1, D_REGS = 96 / (MT * 8);
  static constexpr int D_MIN = D_BYTES < D_CNT ? (D_BYTES < D_REGS ? D_BYTES : D_REGS) : (D_CNT < D_REGS ? D_CNT : D_REGS);
  static constexpr int DEPTH = D_MIN < 2 ? 2 : D_MIN;
  static constexpr int RING = DEPTH * SLOT;                  // per wave
  static constexpr int RED = WAVES * MT * NTW * 4 * 64 * 4;  // reduction buffer (reuses the rings)
  static constexpr int RINGS = WAVES * RING > RED ? WAVES * RING : RED;
  static constexpr int ROW_TABLE = 16 * MT * 8;              // fused QKV only, behind everything else: the cache row of every token
  static constexpr int SMEM = RINGS;  // (ALDS: plus WAVES * M * the share's bytes, added at the launch)
};

// LDS of the activations a wave keeps for its share of K (per_wave slabs), beside the rings: M rows, one after the other
template <int ACTS>
__host__ __device__ constexpr uint32_t skinny_acts_row(uint32_t per_wave) {
  // (quantised in place: rows 16 bytes apart in the bank order, so that 16 tokens read without conflicts; copied: whole
  // 1024-byte copies)
  return ACTS > kActsLds ? per_wave * 128u + 16u : (per_wave * 128u + 1023u) & ~1023u;
}
// ... and the scales that the quantisation leaves there: one per token and slab (block scaling), or the waves' largest values
// and the scale per token
template <int ACTS, bool BLOCKSCALE>
__host__ __device__ constexpr uint32_t skinny_acts_bytes(uint32_t M, uint32_t per_wave) {
  if (ACTS == kActsPerSlab) return 0;
  const uint32_t rows = M * skinny_acts_row<ACTS>(per_wave);
  return ACTS > kActsLds ? rows + (BLOCKSCALE ? (M * per_wave * 4u + 15u) & ~15u : 128u) : rows;
}

// The fused QKV projection's form has a wave of its own for the page look-ups where the tokens are one group of 16.  (With five waves two share
// a SIMD, so each has half of its registers: 256, which two or four groups do not fit.)
__host__ __device__ constexpr int skinny_page_waves(int mt, bool kv) { return kv && mt == 1 ? 1 : 0; }

// One block: columns [n0, n0 + 16 * NTW) of C.
// KV: the fused QKV projection's epilogue (a kernel of its own: the plain one would load its arguments all the same, 1 to 2 per cent)
// c_rows (GROUPED, may be null): row m of the result goes to row c_rows[m] of C
template <int NTW, int MT, bool BLOCKSCALE, int RING_KB, int NWAVES, int ACTS, bool KV, bool GROUPED = false, class Args>
__device__ __forceinline__ void skinny_body(const Args& p, uint8_t* smem, const int n0, [[maybe_unused]] const uint32_t* c_rows = nullptr) {
  using Cfg = SkinnyCfg<NTW, MT, BLOCKSCALE, RING_KB, NWAVES, ACTS>;
  constexpr bool ALDS = Cfg::ALDS, QUANT = Cfg::QUANT;
  static_assert(!ALDS || MT == 1, "activations in LDS: one 16-token group");
  constexpr int WAVES = Cfg::WAVES, DEPTH = Cfg::DEPTH, SLOT = Cfg::SLOT, PER = Cfg::PER;
  static_assert((DEPTH - 1) * PER < 64, "vmcnt is a 6-bit counter");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lq = lane >> 4;
  const int cols_here = (p.N - n0) < 16 * NTW ? (p.N - n0) : 16 * NTW;

  const uint8_t* b_tile = p.b + (int64_t)n0 * p.ldb;
  const __amdgpu_buffer_rsrc_t b_rsrc = sk_rsrc(b_tile, sk_clamp_u32((int64_t)(cols_here - 1) * p.ldb + p.K));
  const __amdgpu_buffer_rsrc_t a_rsrc = sk_rsrc(p.a, sk_clamp_u32((int64_t)(p.M - 1) * p.lda + p.K));

  const int nslab = (p.K + 127) / 128;
  const bool k_tail = (p.K & 127) != 0;
  // this wave's slabs: [s_begin, s_end)
  const int per_wave = (nslab + WAVES - 1) / WAVES;
  const int s_begin = wave * per_wave;
  const int s_end = (s_begin + per_wave) < nslab ? (s_begin + per_wave) : nslab;

  // Fused QKV: a wave of its own looks up the rows' pages while the others walk their slabs.  Its loads depend on one another (a search
  // among the sequences and two more) and stood at the end of the kernel before: 10 tokens, 6144 x 4096, 11.5 -> 11.1 us, quantiser
  // included.
  [[maybe_unused]] int64_t* row_table = reinterpret_cast<int64_t*>(smem + Cfg::RINGS + WAVES * skinny_acts_bytes<ACTS, BLOCKSCALE>((uint32_t)p.M, (uint32_t)per_wave));
  constexpr bool PAGE_WAVE = skinny_page_waves(MT, KV) > 0;
  if constexpr (PAGE_WAVE) {
    if (wave == WAVES) {
      if (lane < 16 * MT) row_table[lane] = lane < p.M ? kv_row_offset(p.kv, lane) : -1;
      if constexpr (QUANT && !BLOCKSCALE) {
        if (!p.x_static) __builtin_amdgcn_s_barrier();  // (the waves' meeting below)
      }
      __syncthreads();
      __syncthreads();
      return;
    }
  }

  // weight DMA: lane (cr = lane >> 3, cp = lane & 7) moves logical chunk cp ^ cr of row cr (then
  // row 8 + cr) of a 16-row group to LDS position lane * 16: row r, chunk c is stored at c ^ (r & 7)
  const int cr = lane >> 3, cp = lane & 7;
  const int cchunk = cp ^ cr;
  const uint32_t w_voff = (uint32_t)cr * (uint32_t)p.ldb + cchunk * 16;
  const uint32_t w_half = 8u * (uint32_t)p.ldb;
  const uint32_t w_tile = 16u * (uint32_t)p.ldb;
  // activation operand: lane (m = lm, lq) holds K bytes [16*lq, +16) and [64 + 16*lq, +16) of token m
  uint32_t a_off[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) a_off[t] = (uint32_t)(t * 16 + lm) * (uint32_t)p.lda + lq * 16;
  // fragment read: row lm of a 16-row group, logical chunks lq and lq + 4
  const uint32_t frag0 = lm * 128 + ((lq ^ (lm & 7)) << 4);
  const uint32_t frag1 = lm * 128 + (((lq + 4) ^ (lm & 7)) << 4);
  uint8_t* ring = smem + wave * Cfg::RING;
  // ALDS: token t's bytes of this wave's share of K sit at a_lds + t * a_tok; lane (lm, lq) reads token min(lm, M - 1)
  // (the columns of C past M are never stored, so what their lanes multiply does not matter)
  [[maybe_unused]] const uint32_t a_tok = skinny_acts_row<ACTS>((uint32_t)per_wave);
  [[maybe_unused]] uint8_t* a_lds = smem + Cfg::RINGS + wave * skinny_acts_bytes<ACTS, BLOCKSCALE>((uint32_t)p.M, (uint32_t)per_wave);
  [[maybe_unused]] float* a_sc = reinterpret_cast<float*>(a_lds + (uint32_t)p.M * a_tok);  // QUANT
  [[maybe_unused]] const uint32_t a_rd = (uint32_t)(lm < p.M ? lm : p.M - 1) * a_tok + lq * 16;
  // QUANT: this lane's bf16 activations, load i = 512 consecutive elements of the share of token i / pieces (zeros past it).
  // They go out before the first weight copies, so that waiting for them is not waiting for those.
  constexpr int NLOADS = QUANT ? ACTS : 1;
  [[maybe_unused]] v4i xv[NLOADS];
  [[maybe_unused]] const int pieces = (per_wave + 3) / 4, n_loads = p.M * pieces;
  if constexpr (QUANT) {
    const __amdgpu_buffer_rsrc_t x_rsrc = sk_rsrc(p.x, sk_clamp_u32(((int64_t)(p.M - 1) * p.ldx + p.K) * 2));
    const uint32_t share_end = (uint32_t)(s_end > s_begin ? s_end : s_begin) * 128u;
    const uint32_t k_end = share_end < (uint32_t)p.K ? share_end : (uint32_t)p.K;
    int t = 0, piece = 0;
#pragma unroll
    for (int i = 0; i < NLOADS; ++i) {
      if (i < n_loads) {
        const uint32_t k = (uint32_t)s_begin * 128u + (uint32_t)piece * 512u + (uint32_t)lane * 8u;
        xv[i] = sk_load16(x_rsrc, k < k_end ? k * 2u : 0x80000000u, (uint32_t)t * (uint32_t)p.ldx * 2u);
        if (++piece == pieces) { piece = 0; ++t; }
      }
    }
  }
  if constexpr (ALDS && !QUANT) {
    // one instruction moves 1024 consecutive bytes of a token; bytes past K or past the share are not fetched (zeros)
    const uint32_t share_begin = (uint32_t)s_begin * 128u, share_end = (uint32_t)(s_end > s_begin ? s_end : s_begin) * 128u;
    const uint32_t k_end = share_end < (uint32_t)p.K ? share_end : (uint32_t)p.K;
    for (int t = 0; t < p.M; ++t)
      for (uint32_t piece = 0; piece < a_tok; piece += 1024u) {
        const uint32_t k = share_begin + piece + lane * 16u;
        const uint32_t kill = k < k_end ? 0u : 0x80000000u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (sk_lds_ptr_t)(a_lds + t * a_tok + piece), 16, ((uint32_t)t * (uint32_t)p.lda + k) | kill, 0, 0, 0);
      }
  }

  __amdgpu_buffer_rsrc_t as_rsrc = sk_rsrc(nullptr, 0), bs_rsrc = sk_rsrc(nullptr, 0);
  uint32_t as_voff[MT];
  if constexpr (BLOCKSCALE && !QUANT) {
    as_rsrc = sk_rsrc(p.a_scales, sk_clamp_u32(((int64_t)(nslab - 1) * p.a_scales_ld + p.M) * 4));
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = t * 16 + lm;
      as_voff[t] = (uint32_t)(m < p.M ? m : p.M - 1) * 4u;
    }
  }

  if constexpr (BLOCKSCALE) bs_rsrc = sk_rsrc(p.b_scales + (int64_t)(n0 / 128) * p.b_scales_ld, (uint32_t)nslab * 4u);

  v4f acc[MT][NTW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  v8i af[DEPTH][MT];
  float as_v[DEPTH][MT], bs_v[DEPTH];

  // Issues the PER loads of one slab into pipeline slot d.  Slabs past the wave's range are
  // issued "out of range" (zeros, no traffic), so every slot always carries exactly PER
  // instructions and the wait counts below are exact.
  auto issue = [&](int slab, auto d_c) {
    constexpr int d = decltype(d_c)::value;
    const bool live = slab < s_end;
    const int sl = live ? slab : s_begin;
    // (wave-uniform by construction; said so explicitly, or the loads' scalar offsets end up in vector registers
    // and every load in a loop over the lanes' values)
    const uint32_t koff = __builtin_amdgcn_readfirstlane((uint32_t)sl * 128u);
    const uint32_t koff_hi = __builtin_amdgcn_readfirstlane(koff + 64u);
    uint32_t kill0 = live ? 0u : 0x80000000u, kill1 = kill0, killw = kill0;
    if (k_tail) {
      if (koff + lq * 16 >= (uint32_t)p.K) kill0 = 0x80000000u;
      if (koff + 64 + lq * 16 >= (uint32_t)p.K) kill1 = 0x80000000u;
      if (koff + cchunk * 16 >= (uint32_t)p.K) killw = 0x80000000u;
    }
    if constexpr (!ALDS) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const v4i lo = sk_load16(a_rsrc, a_off[t] | kill0, koff);
        const v4i hi = sk_load16(a_rsrc, a_off[t] | kill1, koff_hi);
        af[d][t] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      }
    }
    if constexpr (BLOCKSCALE) {
      if constexpr (!QUANT) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
          as_v[d][t] = sk_load_f32(as_rsrc, as_voff[t], (uint32_t)sl * (uint32_t)p.a_scales_ld * 4u);
      }
      bs_v[d] = sk_load_f32(bs_rsrc, 0, (uint32_t)sl * 4u);
    }
    uint8_t* slot = ring + d * SLOT;
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (sk_lds_ptr_t)(slot + t * 2048), 16, w_voff | killw,
                                               koff + t * w_tile, 0, kWeightStream);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (sk_lds_ptr_t)(slot + t * 2048 + 1024), 16, w_voff | killw,
                                               koff + t * w_tile + w_half, 0, kWeightStream);
    }
    // (the slabs' loads stay in this order: with another one in front of the loop, the waits the compiler adds for registers have to hold for
    // both and were for everything in flight, once a round of the ring; 1 to 4 tokens, 102 matmuls, 3.6 per cent, up to 25.  Not in the form
    // that has no registers to spare for the order: it spilled a fifth more.)
    if constexpr (NTW * MT < 16) __builtin_amdgcn_sched_barrier(0);
  };
  auto compute = [&](auto d_c, [[maybe_unused]] int slab) {
    constexpr int d = decltype(d_c)::value;
    // the slot's loads are the oldest in flight: everything issued for the DEPTH-1 younger slots may stay
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * PER) : "memory");
    const uint8_t* slot = ring + d * SLOT;
    if constexpr (ALDS) {
      // (a slab past the share's end multiplies zeros -- its weights were not fetched -- with whatever this reads)
      const uint32_t at = (uint32_t)(slab < s_end ? slab - s_begin : 0) * 128u;
      const v4i lo = *reinterpret_cast<const v4i*>(a_lds + a_rd + at);
      const v4i hi = *reinterpret_cast<const v4i*>(a_lds + a_rd + at + 64);
      af[d][0] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      if constexpr (QUANT && BLOCKSCALE) as_v[d][0] = a_sc[(lm < p.M ? lm : p.M - 1) * per_wave + (slab < s_end ? slab - s_begin : 0)];
    }
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      const v4i lo = *reinterpret_cast<const v4i*>(slot + nt * 2048 + frag0);
      const v4i hi = *reinterpret_cast<const v4i*>(slot + nt * 2048 + frag1);
      const v8i wf = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if constexpr (BLOCKSCALE) {
          const v4f zero = {0.f, 0.f, 0.f, 0.f};
          const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, af[d][mt], zero, 0, 0, 0, 0, 0, 0);
          acc[mt][nt] += part * (as_v[d][mt] * bs_v[d]);
        } else {
          acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, af[d][mt], acc[mt][nt], 0, 0, 0, 0, 0, 0);
        }
      }
    }
    // the fragment reads must have left LDS before the slot is refilled
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  auto for_each_slot = [&](auto&& f) {
    [&]<int... D>(std::integer_sequence<int, D...>) { (f(std::integral_constant<int, D>{}), ...); }
    (std::make_integer_sequence<int, DEPTH>{});
  };

  for_each_slot([&](auto d_c) { issue(s_begin + decltype(d_c)::value, d_c); });
  if constexpr (QUANT) {
    // While the first weight slabs are on their way: the arithmetic of quantize_dynamic_scaled_fp8 (quant.hip), so that the
    // codes and scales are those that kernel would have left in memory.
    auto unpack = [](const v4i& w, float (&f)[8]) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f[2 * j] = __uint_as_float((uint32_t)w[j] << 16);
        f[2 * j + 1] = __uint_as_float((uint32_t)w[j] & 0xffff0000u);
      }
    };
    auto store = [&](const float (&f)[8], float recip, int t, int piece) {
      int lo = 0, hi = 0;
      lo = cvt_pk_e4m3fn(clamp448(f[0] * recip), clamp448(f[1] * recip), lo, false);
      lo = cvt_pk_e4m3fn(clamp448(f[2] * recip), clamp448(f[3] * recip), lo, true);
      hi = cvt_pk_e4m3fn(clamp448(f[4] * recip), clamp448(f[5] * recip), hi, false);
      hi = cvt_pk_e4m3fn(clamp448(f[6] * recip), clamp448(f[7] * recip), hi, true);
      const uint32_t at = (uint32_t)piece * 512u + (uint32_t)lane * 8u;
      if (at < (uint32_t)per_wave * 128u)
        *reinterpret_cast<uint2*>(a_lds + (uint32_t)t * a_tok + at) = make_uint2((uint32_t)lo, (uint32_t)hi);
    };
    auto amax8 = [](const float (&f)[8]) {
      float m = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(f[j]));
      return m;
    };
    int t = 0, piece = 0;
    if constexpr (BLOCKSCALE) {
#pragma unroll
      for (int i = 0; i < NLOADS; ++i) {
        if (i < n_loads) {
          float f[8], scale, recip;
          unpack(xv[i], f);
          dynamic_scale_f32(row16_max(amax8(f)), p.x_scale_ub, scale, recip);
          store(f, recip, t, piece);
          const int slab = piece * 4 + lq;
          if (lm == 0 && slab < per_wave) a_sc[t * per_wave + slab] = scale;
          if (++piece == pieces) { piece = 0; ++t; }
        }
      }
    } else {
      // one scale per token: the waves' shares meet in LDS (word t of each wave's scale area)
      float* meet = reinterpret_cast<float*>(smem + Cfg::RINGS + (uint32_t)p.M * a_tok);
      constexpr uint32_t kWaveStep = 16;  // (each wave's area holds 32 words: 16 for the waves' values of ITS tokens, 16 scales)
      const uint32_t area = skinny_acts_bytes<ACTS, BLOCKSCALE>((uint32_t)p.M, (uint32_t)per_wave) / 4u;
      if (!p.x_static) {
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < NLOADS; ++i) {
          if (i < n_loads) {
            float f[8];
            unpack(xv[i], f);
            m = fmaxf(m, amax8(f));
            if (++piece == pieces) {
              m = wave_max(m);
              if (lane == 0) meet[wave * area + t] = m;
              m = 0.0f;
              piece = 0;
              ++t;
            }
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      t = piece = 0;
      float scale = 0.f, recip = p.x_recip;
#pragma unroll
      for (int i = 0; i < NLOADS; ++i) {
        if (i < n_loads) {
          if (piece == 0 && !p.x_static) {
            float m = meet[t];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) m = fmaxf(m, meet[w * area + t]);
            dynamic_scale_f32(m, p.x_scale_ub, scale, recip);
            if (lane == 0) a_sc[kWaveStep + t] = scale;
          }
          float f[8];
          unpack(xv[i], f);
          store(f, recip, t, piece);
          if (++piece == pieces) { piece = 0; ++t; }
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  for (int base = s_begin; base < s_end; base += DEPTH) {
    for_each_slot([&](auto d_c) {
      constexpr int d = decltype(d_c)::value;
      compute(d_c, base + d);
      issue(base + DEPTH + d, d_c);
    });
  }
  // drain: the last DEPTH issues were out of range, but they still target LDS slots
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // ---- reduce the 4 waves' partial sums (fixed order) and store ----------------------
  float* red = reinterpret_cast<float*>(smem);  // [WAVES][MT*NTW*4][64]
  constexpr int RSTRIDE = MT * NTW * 4 * 64;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[wave * RSTRIDE + ((mt * NTW + nt) * 4 + v) * 64 + lane] = acc[mt][nt][v];
  __syncthreads();

  // (mt, nt) pairs are dealt to the waves round-robin
  for (int pair = wave; pair < MT * NTW; pair += WAVES) {
    const int mt = pair / NTW, nt = pair - mt * NTW;
    const int m = mt * 16 + lm;
    const int n = n0 + nt * 16 + lq * 4;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = (pair * 4 + i) * 64 + lane;
      float sum = red[r];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) sum += red[w * RSTRIDE + r];
      v[i] = sum;
    }
    if (m >= p.M || n >= p.N) continue;
    if constexpr (KV) {
      // fused QKV: the reference's bf16 roundings, then C or the row's K / V page (see tile_body)
      int64_t row_off;
      if constexpr (PAGE_WAVE) row_off = row_table[m];
      else row_off = kv_row_offset(p.kv, m);
      float a_s = 1.f;
      if constexpr (!BLOCKSCALE) a_s = QUANT ? a_sc[16 + m] : p.a_scales[(int64_t)m * p.a_scale_stride];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int nn = (n + i < p.N) ? n + i : p.N - 1;
        float r = bf16_round(v[i]);
        if constexpr (!BLOCKSCALE) {
          const float sc = bf16_round(bf16_round(a_s) * bf16_round(p.b_scales[(int64_t)nn * p.b_scale_stride]));
          r = bf16_round(r * sc);
        }
        if (p.kv.bias) r = bf16_round(r + bf16_bits_to_f32(p.kv.bias[nn]));
        v[i] = r;
      }
      if (row_off < 0 && n >= p.kv.q_dim) continue;
      uint16_t* dst = kv_dst(p.kv, p.c, p.ldc, m, row_off, n);
      if (p.c_vec_ok && n + 3 < p.N) {
        const uint32_t lo = pack_bf16x2(v[0], v[1]);
        const uint32_t hi = pack_bf16x2(v[2], v[3]);
        *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < p.N) dst[i] = (uint16_t)f32_to_bf16_bits(v[i]);
      }
      continue;
    }
    if (!BLOCKSCALE && QUANT && p.x_static) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] *= p.x_scale;
    } else if constexpr (!BLOCKSCALE) {
      float b_s[4];
      scales_at(b_s, p.b_scales, p.scales_dtype, [&](int i) { return (int64_t)(n + i < p.N ? n + i : p.N - 1) * p.b_scale_stride; });
      const float a_s = QUANT ? a_sc[16 + m] : scale_at(p.a_scales, (int64_t)m * p.a_scale_stride, p.scales_dtype);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float t = v[i] * a_s;
        v[i] = t * b_s[i];
      }
    }
    int64_t cm = m;
    if constexpr (GROUPED) {
      if (c_rows) cm = c_rows[m];
    }
    if (p.c_dtype == MAXFP8_BF16) {
      uint16_t* dst = reinterpret_cast<uint16_t*>(p.c) + cm * p.ldc + n;
      if (p.c_vec_ok && n + 3 < p.N) {
        const uint32_t lo = pack_bf16x2(v[0], v[1]);
        const uint32_t hi = pack_bf16x2(v[2], v[3]);
        *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < p.N) dst[i] = (uint16_t)f32_to_bf16_bits(v[i]);
      }
    } else {
      float* dst = reinterpret_cast<float*>(p.c) + cm * p.ldc + n;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < p.N) dst[i] = v[i];
    }
  }
}

template <int NTW, int MT, bool BLOCKSCALE, int RING_KB, int NWAVES, int ACTS = kActsPerSlab, bool KV = false>
__global__ __launch_bounds__((NWAVES + skinny_page_waves(MT, KV)) * 64) void gemm_skinny_kernel(std::conditional_t<KV, GemmArgs, MatmulArgs> p_in) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const auto p = gridDim.y == 1 ? p_in : batch_view(p_in, blockIdx.y);
  skinny_body<NTW, MT, BLOCKSCALE, RING_KB, NWAVES, ACTS, KV>(p, smem, (int)blockIdx.x * (16 * NTW));
}

int compute_units();
template <int NTW, int MT, bool BLOCKSCALE, int RING_KB, int NWAVES, int ACTS = kActsPerSlab, bool KV = false>
static int launch_skinny_r(const GemmArgs& p, int64_t batch, hipStream_t stream) {
  if constexpr (!KV && ACTS != kActsLds) {
    if (p.kv_on) return launch_skinny_r<NTW, MT, BLOCKSCALE, RING_KB, NWAVES, ACTS, true>(p, batch, stream);
  }
  if constexpr (MT == 1 && ACTS == kActsPerSlab && !KV) {
    // few tokens, a share of K per wave that fits, and a weight matrix small enough that the launch is about one round of
    // blocks: the activations go to LDS once (84 MB, M = 1: 17.8 -> 17.0 us; on a 470 MB matrix, where blocks come and
    // go, the per-slab loads cost nothing and this form measured 1 % slower).  Not for the fused QKV epilogue's build, a
    // rare caller at these sizes, to keep the number of kernels down.
    // The extra LDS must not cost a resident block: all blocks of such a launch sit on the chip at once, and a CU's share
    // of them has to fit its 160 KB with the activations added (10240 x 8192 at M = 2: 18.3 -> 16.6 us; at M = 4, where
    // a CU's three blocks would need 192 KB: 18.5 -> 20.2, so that case keeps the per-slab loads).
    const int64_t per_wave = ceil_div(ceil_div(p.K, 128), NWAVES);
    const int64_t a_bytes = (int64_t)p.M * ((per_wave * 128 + 1023) / 1024 * 1024);  // per wave
    const int64_t blocks_per_cu = ceil_div(ceil_div((int64_t)p.N, 16 * NTW) * batch, (int64_t)compute_units());
    using Plain = SkinnyCfg<NTW, MT, BLOCKSCALE, RING_KB, NWAVES>;
    if (tuning().skinny_alds && (int64_t)p.N * p.K < ((int64_t)1 << 27) && a_bytes <= kSkinnyALdsBytes &&
        blocks_per_cu * (Plain::SMEM + NWAVES * a_bytes) <= 160 * 1024)
      return launch_skinny_r<NTW, MT, BLOCKSCALE, RING_KB, NWAVES, kActsLds>(p, batch, stream);
  }
  using Cfg = SkinnyCfg<NTW, MT, BLOCKSCALE, RING_KB, NWAVES, ACTS>;
  auto kern = gemm_skinny_kernel<NTW, MT, BLOCKSCALE, RING_KB, NWAVES, ACTS, KV>;
  static PerDeviceFlag attr;
  bool& attr_done = attr.here();
  constexpr int smem_all = Cfg::QUANT ? 160 * 1024 : Cfg::SMEM + Cfg::ROW_TABLE + (Cfg::ALDS ? NWAVES * kSkinnyALdsBytes : 0);
  constexpr int smem_max = smem_all < 160 * 1024 ? smem_all : 160 * 1024;  // (what a launch asks for was checked against the CU's LDS)
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem_max);
    if (e != hipSuccess) MAXFP8_FAIL(MAXFP8_ERR_LAUNCH, "gemm_skinny: cannot reserve %d bytes of LDS: %s", smem_max, hipGetErrorString(e));
    attr_done = true;
  }
  const uint32_t per_wave = (uint32_t)ceil_div(ceil_div(p.K, 128), NWAVES);
  const int smem = Cfg::SMEM + NWAVES * (int)skinny_acts_bytes<ACTS, BLOCKSCALE>((uint32_t)p.M, per_wave) + (KV ? Cfg::ROW_TABLE : 0);
  const int64_t blocks = ceil_div(p.N, 16 * NTW);
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, (unsigned)batch), dim3((NWAVES + skinny_page_waves(MT, KV)) * 64), smem, stream, static_cast<const std::conditional_t<KV, GemmArgs, MatmulArgs>&>(p));
  return launch_status("gemm_skinny");
}

// Shape choice.  A block re-reads its M x K activations for every 16 * NTW weight rows, through L1 and L2, so the
// activation traffic is M / (16 * NTW) times the weight traffic, and all blocks are resident at once, so a CU's
// share is ceil(blocks / CUs) blocks.  The shape with the smallest
//     ceil(blocks / CUs) * (16 * NTW + M + 8)        (8: ring fill and the epilogue of a block, in the same unit)
// wins; 64-row blocks count 25 % more (one block per CU: 32 KB of weights in flight per wave, but fewer waves to
// hide latency with) and need K >= 4096 (with few slabs per wave the long epilogue shows).  Measured on Llama-70B /
// Llama-8B / DeepSeek-V3 decode shapes in both scale modes the rule lands on the fastest shape or within 4 % of it;
// e.g. M = 64, N = 8192, K = 28672: 32 rows per block, 75 us (16 rows: 122); M = 32, N = 10240, K = 8192: 64 rows,
// 23 us (16 rows: 33); M = 32, N = 5120, K = 5120: 32 rows, 12 us (16 rows: 18); N = 4096: 16 rows, one block per CU.
// 32-row blocks keep 16 KB per wave in flight when M <= 16 and the weights exceed 256 MB, else 8 KB.
// (8 waves per block were tried for the small-N shapes and were no faster.)  Every shape splits K over its four waves
// in the same way and adds the partial sums in the same order: the result does not depend on the choice.
// The tuning switch `skinny` = <ntw>4<ringKB>, e.g. 1408 or 2416, forces a shape for tuning runs.
int compute_units();
static int skinny_shape(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = compute_units();
  int best = 1;
  float best_cost = 0.f;
  for (int ntw = 1; ntw <= 4; ntw *= 2) {
    if (ntw == 4 && K < 4096) break;
    const int64_t blocks = ceil_div(N, 16 * ntw);
    float cost = (float)ceil_div(blocks, cus) * (float)(16 * ntw + M + 8);
    if (ntw == 4) cost *= K >= 8192 ? 1.25f : 1.35f;  // (one block per CU: its start and end weigh more the shorter K is)
    if (ntw == 1 || cost < best_cost) { best = ntw; best_cost = cost; }
  }
  // (16 KB rings for 32-row blocks -- the selector 2416 -- were ahead on the largest matrices while the chip read 6.2
  // TB/s; with the weight copies marked non-temporal 8 KB rings are: 68.6 against 72.2 us on 57344 x 8192 at M = 1)
  if (best == 4) return 4432;
  if (best == 2) return 2408;
  return 1408;
}

template <int MT, bool BLOCKSCALE>
static int pick_ntw(const GemmArgs& p, int64_t batch, hipStream_t stream) {
  int sel = tuning().skinny;
  if (!sel) sel = skinny_shape(p.M, p.N, p.K);
  switch (sel) {
    case 1408: return launch_skinny_r<1, MT, BLOCKSCALE, 8, 4>(p, batch, stream);
    case 1416: return launch_skinny_r<1, MT, BLOCKSCALE, 16, 4>(p, batch, stream);
    case 2416: return launch_skinny_r<2, MT, BLOCKSCALE, 16, 4>(p, batch, stream);
    case 2408: return launch_skinny_r<2, MT, BLOCKSCALE, 8, 4>(p, batch, stream);
    case 4432: return launch_skinny_r<4, MT, BLOCKSCALE, 32, 4>(p, batch, stream);
    default: MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "skinny matmul: unknown shape selector %d", sel);
  }
}

// ---- with the quantisation inside -------------------------------------------------------------------------------
// A block quantises the activations of its waves' shares of K itself, from bf16, while its first weight slabs are on their
// way: no quantisation launch in front and no fp8 activations in memory.  Linear of one token, graph timing, against the
// quantiser and the plain kernel behind it: 4096 x 4096 8.5 -> 6.2 us, 28672 x 4096 24.1 -> 20.0, 10240 x 8192 19.7 -> 15.6 (block
// scaling; row scaling 7.9 -> 6.2, 23.6 -> 20.4, 18.8 -> 15.8).
// Every block repeats the work, a third of a microsecond per 512 elements of a wave (its conversions come one after the
// other, one wave per SIMD): with eight loads per wave the two ways are level (4 tokens of 4096: 9.1 and 8.6 us; 8 tokens 9.5
// and 11.7).  With row scales every token costs a meeting of the waves on top, once per block of a CU: at most four tokens,
// on at most three blocks per CU, and with those at most eight (2 tokens on 24576 x 4096, three blocks, 20.0 and 17.9 us; on 28672 x
// 4096, four, 22.8 and 24.5; 4 tokens on 16384 x 4096, two blocks, 15.8 and 14.2).
constexpr int kQuantLoads = 8;
static int skinny_quant_loads(int64_t M, int64_t K) {
  return (int)(M * ceil_div(ceil_div(ceil_div(K, 128), 4), 4));
}
template <int NTW, bool BLOCKSCALE, int RING_KB>
static bool skinny_quant_fits(int64_t M, int64_t N, int64_t K) {
  const int64_t per_cu = ceil_div(ceil_div(N, 16 * NTW), (int64_t)compute_units());
  if (skinny_quant_loads(M, K) > kQuantLoads || (!BLOCKSCALE && M > 1 && (M > 4 || per_cu > 3 || M * per_cu > 8))) return false;
  // (the quantised activations of the blocks that are on a CU together -- three keep the weight stream full -- fit its LDS)
  const uint32_t per_wave = (uint32_t)ceil_div(ceil_div(K, 128), 4);
  using Cfg = SkinnyCfg<NTW, 1, BLOCKSCALE, RING_KB, 4, kQuantLoads>;
  const int64_t smem = Cfg::SMEM + Cfg::ROW_TABLE +
                       4 * (int64_t)skinny_acts_bytes<kQuantLoads, BLOCKSCALE>((uint32_t)M, per_wave);
  return (per_cu < 3 ? per_cu : 3) * smem <= 160 * 1024;
}
static int skinny_quant_shape(int64_t M, int64_t N, int64_t K) {
  const int sel = tuning().skinny ? tuning().skinny : skinny_shape(M, N, K);
  return sel == 1408 || sel == 2408 || sel == 4432 ? sel : 0;
}
bool gemm_skinny_quant_ok(int64_t M, int64_t N, int64_t K, bool blockscale) {
  if (M < 1 || M > 16 || !tuning().skinny_quant || K % (blockscale ? 128 : 16) != 0) return false;
  switch (skinny_quant_shape(M, N, K)) {
    case 1408: return blockscale ? skinny_quant_fits<1, true, 8>(M, N, K) : skinny_quant_fits<1, false, 8>(M, N, K);
    case 2408: return blockscale ? skinny_quant_fits<2, true, 8>(M, N, K) : skinny_quant_fits<2, false, 8>(M, N, K);
    case 4432: return blockscale ? skinny_quant_fits<4, true, 32>(M, N, K) : skinny_quant_fits<4, false, 32>(M, N, K);
    default: return false;
  }
}
template <bool BLOCKSCALE>
static int pick_quant(const GemmArgs& p, hipStream_t stream) {
  switch (skinny_quant_shape(p.M, p.N, p.K)) {
    case 1408: return launch_skinny_r<1, 1, BLOCKSCALE, 8, 4, kQuantLoads>(p, 1, stream);
    case 2408: return launch_skinny_r<2, 1, BLOCKSCALE, 8, 4, kQuantLoads>(p, 1, stream);
    default: return launch_skinny_r<4, 1, BLOCKSCALE, 32, 4, kQuantLoads>(p, 1, stream);
  }
}
int gemm_skinny_quant_dispatch(const GemmArgs& p, bool blockscale, hipStream_t stream) {
  if (skinny_quant_loads(p.M, p.K) > kQuantLoads)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "decode matmul with the quantisation inside: M = %d, K = %d do not fit", p.M, p.K);
  return blockscale ? pick_quant<true>(p, stream) : pick_quant<false>(p, stream);
}

// ---- grouped: the experts of a few tokens ------------------------------------------------------------------------
// The MoE matmul (rows sorted by expert, slot z = rows [offsets[z], offsets[z + 1]) times the weights of expert expert_ids[z], zeros where that is
// -1: max/kernels/src/linalg/grouped_matmul_sm100_blockwise_fp8.mojo:2938-3105) when its slots hold a few rows each: the decode matmul of every
// slot in use, 16 * NTW weight rows per tile, K split over the block's waves.  Bound by the weights of the experts in use.  A block works out from
// the offsets which slots are in use (a list in LDS, once), then takes every gridDim.x-th tile: no claims, and four blocks per CU, so that one
// block's start and end hide behind the others' streams.  The persistent launch of gemm_tiled.hip, made for mixed sizes, gives
// a CU tiles of 512 weight rows that its block claims from counters in memory: a tile is 21 us and more for one CU however few there are.
// A slot of more than 32 rows is computed 32 rows at a time, its weights read again for each, and each 32 rows are tiles of their own: one slot of most
// of the rows is spread over the chip like many.  (Four groups of 16 rows per pass take 168 registers,
// three blocks per CU and spills: one token of 8 experts 7168 x 2048 70 -> 93 us, 64 tokens 467 -> 560.)
template <int NTW, bool BLOCKSCALE>
struct GroupedSkinnyCfg {
  static constexpr int WAVES = 4, RING_KB = NTW == 1 ? 6 : 8, THREADS = 64 * WAVES;
  using One = SkinnyCfg<NTW, 1, BLOCKSCALE, RING_KB, WAVES>;
  using Two = SkinnyCfg<NTW, 2, BLOCKSCALE, RING_KB, WAVES>;
  static constexpr int LIST = One::SMEM > Two::SMEM ? One::SMEM : Two::SMEM;  // the units of work, behind the rings and sums
  static constexpr int MAX_SLOTS = 512, MAX_ROWS = 16384, MAX_UNITS = MAX_SLOTS + MAX_ROWS / 32, SMEM = LIST + MAX_UNITS * 4 + 2 * WAVES * 4;
};
template <int NTW, bool BLOCKSCALE>
__global__ __launch_bounds__(256, 4) void gemm_grouped_skinny_kernel(GemmArgs g, int ncol) {
  using Cfg = GroupedSkinnyCfg<NTW, BLOCKSCALE>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t* const list = reinterpret_cast<uint32_t*>(smem + Cfg::LIST);  // slot, and which 32 of its rows << 16
  int* const counts = reinterpret_cast<int*>(list + Cfg::MAX_UNITS);
  // (rows held inside [0, M): a stale routing tensor must not turn into accesses outside the operands)
  auto rows_of = [&](int z, int64_t& begin) {
    const int64_t M = g.M, b = g.offsets[z], e = g.offsets[z + 1];
    begin = b < M ? b : M;
    const int64_t end = e < M ? e : M;
    return (int)(end > begin ? end - begin : 0);
  };
  int units = 0;
#pragma unroll
  for (int half = 0; half < Cfg::MAX_SLOTS / Cfg::THREADS; ++half) {
    const int z = half * Cfg::THREADS + tid;
    int64_t begin;
    const int mine = z < g.num_active ? (rows_of(z, begin) + 31) >> 5 : 0;
    // (the sums over the lanes bit by bit: mostly there is one)
    int in_front = 0, of_wave = 0;
    for (int bit = 0; __ballot(mine >> bit) != 0; ++bit) {
      const uint64_t with = __ballot(mine >> bit & 1);
      in_front += __popcll(with & (((uint64_t)1 << lane) - 1)) << bit;
      of_wave += __popcll(with) << bit;
    }
    if (lane == 0) counts[half * Cfg::WAVES + wave] = of_wave;
    __syncthreads();
    int at = units + in_front;
    for (int w = 0; w < Cfg::WAVES; ++w) {
      const int c = counts[half * Cfg::WAVES + w];
      if (w < wave) at += c;
      units += c;
    }
    // (more than fit only with stale offsets that overlap)
    for (int i = 0; i < mine && at + i < Cfg::MAX_UNITS; ++i) list[at + i] = (uint32_t)z | (uint32_t)i << 16;
  }
  units = __builtin_amdgcn_readfirstlane(units < Cfg::MAX_UNITS ? units : Cfg::MAX_UNITS);
  for (int t = (int)blockIdx.x; t < units * ncol; t += (int)gridDim.x) {
    __syncthreads();  // the list is there; the last tile's sums have been read
    const int j = t / ncol, n0 = (t - j * ncol) * 16 * NTW;
    const uint32_t unit = __builtin_amdgcn_readfirstlane(list[j]);
    const int slot = (int)(unit & 0xffffu), r0 = (int)(unit >> 16) * 32;
    int64_t begin;
    const int all = rows_of(slot, begin), rows = all - r0 < 32 ? all - r0 : 32;
    begin += r0;
    const int e = g.expert_ids[slot];
    const int64_t esize = g.c_dtype == MAXFP8_BF16 ? 2 : 4;
    if (e < 0) {
      const int cols = g.N - n0 < 16 * NTW ? g.N - n0 : 16 * NTW;
      for (int i = tid; i < rows * cols; i += Cfg::THREADS) {
        const int r = i / cols;
        const int64_t m = begin + r, at = (g.c_row_index ? (int64_t)g.c_row_index[m] : m) * g.ldc + n0 + (i - r * cols);
        if (esize == 2) reinterpret_cast<uint16_t*>(g.c)[at] = 0;
        else reinterpret_cast<float*>(g.c)[at] = 0.f;
      }
      continue;
    }
    MatmulArgs p = g;
    p.b = g.b + (int64_t)e * g.b_expert_stride;
    p.b_scales = g.b_scales + (int64_t)e * g.bs_expert_stride;
    p.M = rows;
    p.a = g.a + begin * g.lda;
    p.a_scales = g.a_scales + (BLOCKSCALE ? begin : begin * g.a_scale_stride);
    const uint32_t* c_rows = g.c_row_index ? g.c_row_index + begin : nullptr;
    p.c = g.c_row_index ? g.c : reinterpret_cast<uint8_t*>(g.c) + begin * g.ldc * esize;
    if (rows <= 16) skinny_body<NTW, 1, BLOCKSCALE, Cfg::RING_KB, Cfg::WAVES, kActsPerSlab, false, true>(p, smem, n0, c_rows);
    else skinny_body<NTW, 2, BLOCKSCALE, Cfg::RING_KB, Cfg::WAVES, kActsPerSlab, false, true>(p, smem, n0, c_rows);
  }
}

template <int NTW, bool BLOCKSCALE>
static int launch_grouped_skinny(const GemmArgs& p, int64_t most_tiles, hipStream_t stream) {
  using Cfg = GroupedSkinnyCfg<NTW, BLOCKSCALE>;
  auto kern = gemm_grouped_skinny_kernel<NTW, BLOCKSCALE>;
  static PerDeviceFlag attr;
  bool& attr_done = attr.here();
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::SMEM);
    if (e != hipSuccess) MAXFP8_FAIL(MAXFP8_ERR_LAUNCH, "gemm_grouped_skinny: cannot reserve %d bytes of LDS: %s", Cfg::SMEM, hipGetErrorString(e));
    attr_done = true;
  }
  const int64_t resident = 4 * (int64_t)compute_units();
  hipLaunchKernelGGL(kern, dim3((unsigned)(most_tiles < resident ? most_tiles : resident)), dim3(Cfg::THREADS), Cfg::SMEM, stream, p,
                     (int)ceil_div(p.N, 16 * NTW));
  return launch_status("gemm_grouped_skinny");
}

// Total rows up to which a grouped matmul comes here.  The experts' two matmuls with what is around them, persistent launch and this one, us: 256
// experts of 7168 x 2048, 8 per token, 1 / 8 / 32 / 48 / 64 / 128 tokens 137 / 213 / 395 / 408 / 453 / 565 and 71 / 173 / 323 / 401 / 469 / 713; 128 of 4096 x 1536,
// 8 per token, 1 / 16 / 64 / 80 tokens 95 / 146 / 251 / 254 and 45 / 116 / 240 / 274; 64 of 2048 x 1408, 6 per token, 1 / 16 / 80 / 96 tokens 70 / 88 / 121 /
// 121 and 32 / 52 / 115 / 126.  Level at 400, 576 and 510 rows: what turns it is the slots of more than 32 rows, whose weights are read more than once.
// So few slots turn it at fewer rows: one matmul of 7168 x 2048, 2 slots with 64 / 128 / 256 rows in all 42 / 28 / 29 us and 17 / 30 / 57, 4 slots with 128 / 256
// 44 / 29 and 27 / 50, 8 with 256 / 448 41 / 40 and 31 / 57; 4096 x 7168, 4 slots with 128 / 256 / 448 123 / 64 / 70 and 41 / 79 / 143.  (Those were measured with a slot's
// 32-row parts one after the other in a block.)  Skewed routings, whose host knows no better, one matmul, weights from memory, persistent launch, this one, and with the parts
// one after the other: 448 rows all in one of 64 slots, 3072 x 4096 70 / 40 / 94 us, 4096 x 7168 115 / 81 / 160, 7168 x 2048 43 / 49 / 58; half of them in one of 20 slots 74 / 65 / 88,
// 125 / 140 / 166, 85 / 83 / 85; half of 300 in one of 64 155 / 134 / 149, 349 / 300 / 320, 165 / 170 / 169.  Over 440 routings of 64 to 448 rows the worst is 14 per cent behind, at 448 rows (40 before).
// max_rows: the caller's bound on a slot's rows; all rows there are stands for one that does not know.
bool gemm_grouped_skinny_ok(const GemmArgs& p, int64_t max_rows) {
  if (p.num_active > GroupedSkinnyCfg<2, true>::MAX_SLOTS || p.M > GroupedSkinnyCfg<2, true>::MAX_ROWS) return false;
  if (((int64_t)p.num_active + p.M / 32) * ceil_div(p.N, 16) >= (int64_t)1 << 30) return false;  // (the tiles' numbers)
  const int forced = tuning().grouped_decode;
  if (forced >= 0) return p.M <= forced;
  return p.M <= 448 && p.M <= 64 + 20 * p.num_active && (max_rows <= 128 || max_rows >= p.M);
}
int gemm_grouped_skinny_dispatch(const GemmArgs& p, bool blockscale, hipStream_t stream) {
  const int64_t slots = p.M < p.num_active ? p.M : p.num_active, units = slots + p.M / 32;  // (at most)
  if (slots * ceil_div(p.N, 32) >= 4 * (int64_t)compute_units()) {
    const int64_t wide = units * ceil_div(p.N, 32);
    return blockscale ? launch_grouped_skinny<2, true>(p, wide, stream) : launch_grouped_skinny<2, false>(p, wide, stream);
  }
  const int64_t narrow = units * ceil_div(p.N, 16);
  return blockscale ? launch_grouped_skinny<1, true>(p, narrow, stream) : launch_grouped_skinny<1, false>(p, narrow, stream);
}

// ---- read-only probe ---------------------------------------------------------------------------
// The weight traffic of gemm_skinny_kernel and nothing else: same grid, block size, rows per block, split of K over
// the waves, LDS ring, ring depth, DMA instructions and wait counts as the matmul of an M <= 16 row-scaled problem, but
// no activations, no MFMA, no reduction and no stores (one dword per slab is read back from LDS so that the ring is
// consumed in order).  Its time is what this access pattern can reach on the memory system: the matmul is measured
// against it.
template <int NTW, int RING_KB, int NWAVES>
__global__ __launch_bounds__(NWAVES * 64) void skinny_read_probe_kernel(const uint8_t* b, int N, int K, int64_t ldb, uint32_t* sink) {
  using Cfg = SkinnyCfg<NTW, 1, false, RING_KB, NWAVES>;
  constexpr int WAVES = Cfg::WAVES, DEPTH = Cfg::DEPTH, SLOT = Cfg::SLOT, PER = 2 * NTW;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * (16 * NTW);
  const int cols_here = (N - n0) < 16 * NTW ? (N - n0) : 16 * NTW;
  const __amdgpu_buffer_rsrc_t b_rsrc = sk_rsrc(b + (int64_t)n0 * ldb, sk_clamp_u32((int64_t)(cols_here - 1) * ldb + K));
  const int nslab = (K + 127) / 128;
  const int per_wave = (nslab + WAVES - 1) / WAVES;
  const int s_begin = wave * per_wave;
  const int s_end = (s_begin + per_wave) < nslab ? (s_begin + per_wave) : nslab;
  const int cr = lane >> 3, cp = lane & 7;
  const uint32_t w_voff = (uint32_t)cr * (uint32_t)ldb + (cp ^ cr) * 16;
  const uint32_t w_half = 8u * (uint32_t)ldb, w_tile = 16u * (uint32_t)ldb;
  uint8_t* ring = smem + wave * Cfg::RING;
  uint32_t seen = 0;
  auto issue = [&](int slab, auto d_c) {
    constexpr int d = decltype(d_c)::value;
    const bool live = slab < s_end;
    const uint32_t koff = (uint32_t)(live ? slab : s_begin) * 128u;
    const uint32_t killw = live ? 0u : 0x80000000u;
    uint8_t* slot = ring + d * SLOT;
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (sk_lds_ptr_t)(slot + t * 2048), 16, w_voff | killw, koff + t * w_tile, 0, kWeightStream);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (sk_lds_ptr_t)(slot + t * 2048 + 1024), 16, w_voff | killw, koff + t * w_tile + w_half, 0, kWeightStream);
    }
  };
  auto consume = [&](auto d_c) {
    constexpr int d = decltype(d_c)::value;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * PER) : "memory");
    seen ^= *reinterpret_cast<const uint32_t*>(ring + d * SLOT + lane * 4);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  auto for_each_slot = [&](auto&& f) {
    [&]<int... D>(std::integer_sequence<int, D...>) { (f(std::integral_constant<int, D>{}), ...); }
    (std::make_integer_sequence<int, DEPTH>{});
  };
  for_each_slot([&](auto d_c) { issue(s_begin + decltype(d_c)::value, d_c); });
  for (int base = s_begin; base < s_end; base += DEPTH) {
    for_each_slot([&](auto d_c) {
      constexpr int d = decltype(d_c)::value;
      consume(d_c);
      issue(base + DEPTH + d, d_c);
    });
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // (never true for the data the benchmark streams; keeps the reads alive)
  if (seen == 0x9e3779b9u && sink) sink[0] = seen;
}

template <int NTW, int RING_KB, int NWAVES>
static int launch_read_probe(const void* b, int64_t N, int64_t K, int64_t ldb, hipStream_t stream) {
  using Cfg = SkinnyCfg<NTW, 1, false, RING_KB, NWAVES>;
  auto kern = skinny_read_probe_kernel<NTW, RING_KB, NWAVES>;
  static PerDeviceFlag attr;
  bool& attr_done = attr.here();
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::SMEM);
    if (e != hipSuccess) MAXFP8_FAIL(MAXFP8_ERR_LAUNCH, "read probe: cannot reserve %d bytes of LDS: %s", Cfg::SMEM, hipGetErrorString(e));
    attr_done = true;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(N, 16 * NTW)), dim3(NWAVES * 64), Cfg::SMEM, stream, (const uint8_t*)b, (int)N, (int)K,
                     ldb, (uint32_t*)nullptr);
  return launch_status("skinny_read_probe");
}

int gemm_skinny_read_probe(const void* b, int64_t M, int64_t N, int64_t K, int64_t ldb, hipStream_t stream) {
  int sel = tuning().skinny;
  if (!sel) sel = skinny_shape(M, N, K);
  switch (sel) {
    case 1408: return launch_read_probe<1, 8, 4>(b, N, K, ldb, stream);
    case 1416: return launch_read_probe<1, 16, 4>(b, N, K, ldb, stream);
    case 2416: return launch_read_probe<2, 16, 4>(b, N, K, ldb, stream);
    case 2408: return launch_read_probe<2, 8, 4>(b, N, K, ldb, stream);
    case 4432: return launch_read_probe<4, 32, 4>(b, N, K, ldb, stream);
    default: MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "read probe: unknown shape selector %d", sel);
  }
}

int gemm_skinny_max_m() { return 64; }

// Where streaming the weights is preferred to the tiles by size alone: every matmul of at most 32 rows (but see below), and those
// of 33 to 64 rows whose weights take less than 32 MB.  (Batches, and what the small tiles of gemm_mid.hip do not take, go by it; the choice
// between those, the tiles and this kernel is made in api.hip.)  With four 16-token groups per weight fragment every block re-reads 64 rows of
// activations through its L1 (about 8 TB/s over the chip) and its time grows with M, while the three-stage 128 x 128
// tiles share the activations through LDS, split K over the chip when their column tiles are few, and take the same
// time from 1 to 128 rows: at M = 64 they measured 54 us against 75 (N = 8192, K = 28672), 19 against 36 (2304 x
// 16384), 25 against 32 (10240 x 8192), 30 against 40 (28672 x 4096).  Their floor is two launches, 16 to 17 us:
// below 32 MB of weights the streaming kernel stays ahead (4096 x 4096: 12 us; 6144 x 4096: 14).
// From 25 rows on the tiles are already ahead where K is long and N narrow (M = 32: 48 us against 53 on 8192 x 28672,
// 17 against 21 on 4096 x 14336 and on 2304 x 16384); at 24 rows and below the streaming kernel wins or ties.
bool gemm_skinny_preferred(int64_t M, int64_t N, int64_t K) {
  const bool small_weights = N * K < ((int64_t)1 << 25);
  if (M <= 24) return true;
  if (M <= 32) return small_weights || K < 12288 || N >= 10240;
  return M <= 64 && small_weights;
}

// Estimated microseconds at 17 to 32 rows with row scales, fitted to 700 matmuls with the weights from memory and, with less weight, in the memory-side cache: within 3 per cent
// for half of the launches, 7 for nine in ten.  *alone: a CU has one block, of at most 32 weight rows
float gemm_skinny_cost(int64_t M, int64_t N, int64_t K, bool* alone) {
  const int ntw = skinny_shape(M, N, K) / 1000;
  const int64_t per_cu = ceil_div(ceil_div(N, 16 * ntw), (int64_t)compute_units());
  *alone = per_cu == 1 && ntw <= 2;
  const float blocks = (float)per_cu, k = (float)K * 1e-4f, weights = (float)N * (float)K * 1e-6f;
  return 3.07f + blocks * (0.76f + (3.32f * (float)ntw + 0.42f + 0.192f * (float)M) * k) + 0.025f * weights;
}

int gemm_skinny_dispatch(const GemmArgs& p, bool blockscale, int64_t batch, hipStream_t stream) {
  if (p.M > 64) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "skinny matmul: M = %d exceeds 64", p.M);
  const int mt = (p.M + 15) / 16;
  if (blockscale) {
    if (mt <= 1) return pick_ntw<1, true>(p, batch, stream);
    if (mt <= 2) return pick_ntw<2, true>(p, batch, stream);
    return pick_ntw<4, true>(p, batch, stream);
  }
  if (mt <= 1) return pick_ntw<1, false>(p, batch, stream);
  if (mt <= 2) return pick_ntw<2, false>(p, batch, stream);
  return pick_ntw<4, false>(p, batch, stream);
}

}  // namespace maxfp8
