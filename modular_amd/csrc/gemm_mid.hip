// Scaled FP8 matmul for batches between decode and prefill (a few to a thousand tokens): C[M,N] = A[M,K] . B[N,K]^T.
//
// Such a matmul is a few dozen 128 x 128 tiles: too few for the chip, so the tile kernels cut K over blocks and pay for it
// with a second launch (or a hand-over) and the partial sums' way to memory and back.  Here the K split stays inside a
// block: a block owns a small tile, 16 * MT tokens x 16 * NT weight rows, its waves a share of K each, and their
// partial tiles meet in LDS.  Small tiles make enough blocks for the chip without a cut.
//
//   * Each wave has an LDS ring of its own: a slot holds one 128-wide slab of the tile's weight rows AND token rows (and
//     their scales), copied by LDS-DMA in whole 128-byte lines.  No barrier in the loop; waits are exact counts.  (Token rows
//     loaded straight into the MFMA's operand layout instead, 16 rows x 64 bytes per instruction, come in at 38 GB/s
//     per CU, out of L2 too; copies of 8 rows x 128 bytes at 117.)
//   * A slot's fragments are read into registers at once, and the copies that refill it go out between the MFMAs that multiply
//     them: a CU takes a copy of 1 KB every 18 cycles, so a slab's copies sent together stop their wave for as long as its
//     MFMAs take (117 x 6144 x 4096 in 64 x 48 tiles 12.5 -> 10.6 us).
//   * How a CU is filled (BLOCKS per CU): one block of eight waves with the whole LDS, all on one tile where there is one for each CU (the same
//     shape 10.2 us); or two, three or four blocks of four waves on a share of it, so that one block's start and end hide
//     behind another's loop (432 x 3648 x 2432 in 64 x 64 tiles 16.3 -> 12.5 us, 730 x 1824 x 1536 12.1 -> 9.3).
//   * Epilogue: partial sums to LDS as [token][column], a thread adds them (in wave order) for eight columns of a token,
//     scales, converts and stores 16 bytes.  Row scales are loaded in front of the copies (their first use was the longest
//     wait of the epilogue); a wave of its own makes the fused QKV projection's page look-ups during the loop.
//
// Bound: what a CU can pull out of the L2s -- every block fetches its tokens and weights itself, 16 * (MT + NT) * K bytes.
// Measured (graph timing, operands in the memory-side cache) against what ran these shapes before: 117 x 6144 x 4096 12.1 -> 10.2 us,
// 432 x 3648 x 2432 20.1 -> 12.5, 730 x 1824 x 1536 17.2 -> 8.8, 18 x 4096 x 14336 15.6 -> 13.4, 28 x 6144 x 4096 8.9 -> 7.3.  Bytes at
// 7 TB/s: 3.9, 2.1, 1.1, 8.4 and 3.7.  64 x 10240 x 8192 with row scales, whose weights pass the L2s by (`once` below), stays at 23.7 (12.2).
#include <type_traits>
#include <utility>

#include "common.h"
#include "gemm_args.h"
#include "gemm_device.h"
#include "tuning.h"

namespace maxfp8 {

// BLOCKS blocks per CU: their waves and their share of its LDS
__host__ __device__ constexpr int mid_waves(int blocks) { return blocks == 1 ? 8 : 4; }
__host__ __device__ constexpr int mid_lds(int blocks) { return (blocks == 1 ? 160 : blocks == 2 ? 79 : blocks == 3 ? 53 : 39) * 1024; }
// Slabs in flight per wave: what the block's LDS holds and the 6-bit wait counter counts -- of the shapes below one, or two in the smaller tiles of four waves
__host__ __device__ constexpr int mid_depth(int mt, int nt, bool blockscale, int blocks) {
  const int groups = blockscale ? (mt + 3) / 4 : 0, slot = (mt + nt) * 2048 + 256 * groups, per = 2 * (mt + nt) + groups;
  const int lds = (mid_lds(blocks) - 16 * mt * 8) / mid_waves(blocks) / slot, counter = 63 / per + 1;
  return lds < counter ? lds : counter;
}

template <int MT, int NT, bool BLOCKSCALE, int BLOCKS>
struct MidCfg {
  static constexpr int NWAVES = mid_waves(BLOCKS), BM = 16 * MT, BN = 16 * NT;
  static constexpr int SCALES = BLOCKSCALE ? 256 : 0;        // 64 activation scales: one copy
  static constexpr int SLOT = (MT + NT) * 2048 + SCALES;
  static constexpr int PER = 2 * (MT + NT) + (BLOCKSCALE ? 1 : 0);  // copies per wave and slab
  static constexpr int ROW_TABLE = BM * 8;                   // fused QKV: the cache row of every token
  static constexpr int DEPTH = mid_depth(MT, NT, BLOCKSCALE, BLOCKS);
  static constexpr int RING = DEPTH * SLOT;
  static constexpr int RED_LD = BN + 4;                      // floats per token row of a partial tile
  static constexpr int RED = NWAVES * BM * RED_LD * 4;
  static constexpr int SMEM = (NWAVES * RING > RED ? NWAVES * RING : RED) + ROW_TABLE;
  static_assert(MT <= 4 && NT <= 4 && DEPTH >= 1 && SMEM <= mid_lds(BLOCKS));
};

// Where the copies of a slab read
struct MidSlabAt { uint32_t koff, kill, scales; };

// KV: the fused QKV projection's epilogue and its wave of page look-ups
template <int MT, int NT, bool BLOCKSCALE, int W_POLICY, int BLOCKS, bool KV>
__global__ __launch_bounds__((BLOCKS == 1 ? 512 : 256) + (KV ? 64 : 0)) __attribute__((amdgpu_waves_per_eu(1, (BLOCKS == 1 ? 2 : BLOCKS) + (KV ? 1 : 0)))) void gemm_mid_kernel(std::conditional_t<KV, GemmArgs, MatmulArgs> p, int tiles_m, int tiles_n) {
  using Cfg = MidCfg<MT, NT, BLOCKSCALE, BLOCKS>;
  constexpr int NWAVES = Cfg::NWAVES, BM = Cfg::BM, BN = Cfg::BN, DEPTH = Cfg::DEPTH, PER = Cfg::PER, SLOT = Cfg::SLOT;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  // block id -> tile: every XCD (id mod 8) takes a contiguous run of tiles, the row tiles of a column tile next to each
  // other: its L2 holds their weights
  const int total = tiles_m * tiles_n, xcd = blockIdx.x & 7, share = total >> 3, extra = total & 7;
  const int index = xcd * share + (xcd < extra ? xcd : extra) + (int)(blockIdx.x >> 3);
  const int tn = index / tiles_m, tm = index - tn * tiles_m;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lq = lane >> 4;
  const int m0 = tm * BM, n0 = tn * BN;
  const int rows_here = p.M - m0 < BM ? p.M - m0 : BM;
  const int cols_here = p.N - n0 < BN ? p.N - n0 : BN;
  int64_t* row_table = reinterpret_cast<int64_t*>(smem + Cfg::SMEM - Cfg::ROW_TABLE);

  const __amdgpu_buffer_rsrc_t a_rsrc = t2_rsrc(p.a + (int64_t)m0 * p.lda, t2_clamp_u32((int64_t)(rows_here - 1) * p.lda + p.K));
  const __amdgpu_buffer_rsrc_t b_rsrc = t2_rsrc(p.b + (int64_t)n0 * p.ldb, t2_clamp_u32((int64_t)(cols_here - 1) * p.ldb + p.K));
  const int nslab = (p.K + 127) / 128;
  const bool k_tail = (p.K & 127) != 0;
  const int per_wave = (nslab + NWAVES - 1) / NWAVES;
  const int s_begin = wave * per_wave;
  const int s_end = s_begin + per_wave < nslab ? s_begin + per_wave : nslab;

  // copies: lane (cr, cp) moves logical chunk cp ^ cr of row cr of an 8-row group; row r keeps chunk c at c ^ (r & 7)
  const int cr = lane >> 3, cchunk = (lane & 7) ^ cr;
  const uint32_t a_voff = (uint32_t)cr * (uint32_t)p.lda + cchunk * 16;
  const uint32_t b_voff = (uint32_t)cr * (uint32_t)p.ldb + cchunk * 16;
  const uint32_t a_step = 8u * (uint32_t)p.lda, b_step = 8u * (uint32_t)p.ldb;
  const uint32_t frag0 = lm * 128 + ((lq ^ (lm & 7)) << 4);
  const uint32_t frag1 = lm * 128 + (((lq + 4) ^ (lm & 7)) << 4);
  uint8_t* ring = smem + wave * Cfg::RING;

  // Block scaling: activation scale i of a slab's copy is that of token 16 * (i % 4) + i / 4, so that a lane reads its MT
  // scales (tokens lm, lm + 16, ...) with one 16-byte read.  The weight scales of the wave's slabs sit in a register, one
  // slab per lane (a column tile of 48 touches two scale rows).
  __amdgpu_buffer_rsrc_t s_rsrc = t2_rsrc(nullptr, 0);
  uint32_t s_voff = 0x80000000u;
  float bs_lo = 0.f, bs_hi = 0.f;
  if constexpr (BLOCKSCALE) {
    s_rsrc = t2_rsrc(p.a_scales + m0, t2_clamp_u32(((int64_t)(nslab - 1) * p.a_scales_ld + rows_here) * 4));
    const int token = 16 * (lane & 3) + (lane >> 2);
    if (token < rows_here) s_voff = (uint32_t)token * 4u;
    const int s = s_begin + lane;
    if (lane < per_wave && s < nslab) {
      bs_lo = p.b_scales[(int64_t)(n0 / 128) * p.b_scales_ld + s];
      bs_hi = NT == 3 && n0 / 128 != (n0 + cols_here - 1) / 128 ? p.b_scales[(int64_t)(n0 / 128 + 1) * p.b_scales_ld + s] : bs_lo;
    }
  }
  // 16-row groups of weights from here on belong to the second scale row
  const int nt_hi = NT == 3 ? (128 - n0 % 128) / 16 : NT;

  // Row scaling: what the epilogue multiplies this thread's results by (eight columns of a token per item), loaded before
  // the copies
  constexpr int CHUNKS = BN / 8, ITEMS = (BM * CHUNKS + NWAVES * 64 - 1) / (NWAVES * 64);
  float row_s[ITEMS], col_s[ITEMS][8];
  if (!BLOCKSCALE && (!KV || wave < NWAVES)) {
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int item = it * NWAVES * 64 + tid, row = item / CHUNKS, col = (item - row * CHUNKS) * 8;
      scales_at(col_s[it], p.b_scales, p.scales_dtype, [&](int i) { return (int64_t)(n0 + col + i < p.N ? n0 + col + i : p.N - 1) * p.b_scale_stride; });
      float one[1];
      scales_at(one, p.a_scales, p.scales_dtype, [&](int) { return (int64_t)(m0 + (row < rows_here ? row : 0)) * p.a_scale_stride; });
      row_s[it] = one[0];
    }
  }

  v4f acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  auto slab_at = [&](int slab) {
    MidSlabAt at;
    at.koff = __builtin_amdgcn_readfirstlane((uint32_t)slab * 128u);
    at.kill = k_tail && at.koff + cchunk * 16 >= (uint32_t)p.K ? 0x80000000u : 0u;
    at.scales = (uint32_t)slab * (uint32_t)p.a_scales_ld * 4u;
    return at;
  };
  // copy i (0 .. PER - 1, known at compile time) of a slab into slot d: weight rows, token rows, token scales
  auto copy = [&](const MidSlabAt& at, int d, int i) {
    uint8_t* slot = ring + d * SLOT;
    if (i < 2 * NT)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (lds_ptr_t)(slot + i * 1024), 16, b_voff | at.kill, at.koff + i * b_step, 0, W_POLICY);
    else if (i < 2 * (NT + MT))
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(slot + i * 1024), 16, a_voff | at.kill, at.koff + (i - 2 * NT) * a_step, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(s_rsrc, (lds_ptr_t)(slot + (MT + NT) * 2048), 4, s_voff, at.scales, 0, 0);
  };
  // One slab, in slot d.  REFILLS: slab + DEPTH is one of the wave's too and takes the slot.  behind: DEPTH - 1 slabs are in flight behind this one
  // (fewer only at the end of the share, where the wait is for everything).
  auto step = [&](int slab, int d, auto refills_c, bool behind) {
    constexpr bool REFILLS = decltype(refills_c)::value;
    if (DEPTH > 1 && behind) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * PER) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const uint8_t* slot = ring + d * SLOT;
    v8i wf[NT], af[MT];
    auto frag = [&](const uint8_t* g) {
      const v4i lo = *reinterpret_cast<const v4i*>(g + frag0);
      const v4i hi = *reinterpret_cast<const v4i*>(g + frag1);
      return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    };
#pragma unroll
    for (int i = 0; i < NT; ++i) wf[i] = frag(slot + i * 2048);
#pragma unroll
    for (int i = 0; i < MT; ++i) af[i] = frag(slot + (NT + i) * 2048);
    v4f as = {0.f, 0.f, 0.f, 0.f};
    float b0 = 0.f, b1 = 0.f;
    if constexpr (BLOCKSCALE) {
      as = *reinterpret_cast<const v4f*>(slot + (MT + NT) * 2048 + lm * 16);
      const int at = __builtin_amdgcn_readfirstlane(slab - s_begin);
      b0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, bs_lo), at));
      b1 = NT == 3 ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, bs_hi), at)) : b0;
    }
    // the slot's bytes are in registers before it is refilled
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    // MFMA i, in front of it its share of the copies of the slab that takes this slot, and behind it the promotion of the
    // product LAG MFMAs back, which has left the matrix pipe
    const MidSlabAt next = slab_at(slab + DEPTH);
    constexpr int NM = MT * NT, LAG = 3;
    v4f part[LAG + 1];
    auto promote = [&](auto j_c) {
      constexpr int j = decltype(j_c)::value, mt = j / NT, nt = j % NT;
      // (fused by name: the loop's copies of this have parts in common, and a product and a sum the compiler would merge one by one, each rounded)
      const float scale = as[mt] * (NT == 3 && nt >= nt_hi ? b1 : b0);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[mt][nt][i] = fmaf(part[j % (LAG + 1)][i], scale, acc[mt][nt][i]);
    };
    static_for<NM>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value, mt = i / NT, nt = i % NT, c0 = i * PER / NM, c1 = (i + 1) * PER / NM;
      if constexpr (REFILLS) static_for<c1 - c0>([&](auto c_c) { copy(next, d, c0 + decltype(c_c)::value); });
      if constexpr (BLOCKSCALE) {
        const v4f zero = {0.f, 0.f, 0.f, 0.f};
        part[i % (LAG + 1)] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[nt], af[mt], zero, 0, 0, 0, 0, 0, 0);
        if constexpr (i >= LAG) promote(std::integral_constant<int, i - LAG>{});
      } else {
        acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[nt], af[mt], acc[mt][nt], 0, 0, 0, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (BLOCKSCALE) {
      constexpr int left = NM < LAG ? NM : LAG;
      static_for<left>([&](auto j_c) { promote(std::integral_constant<int, NM - left + decltype(j_c)::value>{}); });
    }
  };

  if ((!KV || wave < NWAVES) && s_begin < s_end) {
    // (copies are sent for the wave's own slabs only: those of a slab past its share, of nothing, kept the counts of the waits exact and
    // took a CU's 18 cycles each all the same, a fifth of the copies of a share of four slabs)
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (d > 0 && s_begin + d >= s_end) break;
      const MidSlabAt at = slab_at(s_begin + d);
#pragma unroll
      for (int i = 0; i < PER; ++i) copy(at, d, i);
    }
    if constexpr (BLOCKSCALE)  // (the weight scales are older than the copies: they arrive without waiting for those)
      asm volatile("s_waitcnt vmcnt(%2)" : "+v"(bs_lo), "+v"(bs_hi) : "n"(DEPTH * PER < 63 ? DEPTH * PER : 63));
    int slab = s_begin;
    for (; slab + 2 * DEPTH <= s_end; slab += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) step(slab + d, d, std::true_type{}, true);
    }
    const int left = s_end - slab;  // 1 .. 2 DEPTH - 1
    static_for<2 * DEPTH - 1>([&](auto t_c) {
      constexpr int t = decltype(t_c)::value;
      if (t + 1 < DEPTH && t + DEPTH < left) step(slab + t, t % DEPTH, std::true_type{}, true);
      else if (t < left) step(slab + t, t % DEPTH, std::false_type{}, t + DEPTH <= left);
    });
  } else if (KV && wave >= NWAVES && lane < BM) {
    // fused QKV: a wave of its own looks up the rows' pages.  Its loads depend on one another, a search among the sequences and two
    // more; in one of the other waves each of them waited for all copies in front of it, and the wave's share of K for them
    // (64 tokens of 64 sequences, 10240 x 8192 with row scales, quantiser and the new tiles included: 30.9 -> 30.5 us).
    if constexpr (KV) row_table[lane] = lane < rows_here ? kv_row_offset(p.kv, m0 + lane) : -1;
  }
  __syncthreads();

  // ---- the waves' partial tiles meet ------------------------------------------------------------------------------
  float* red = reinterpret_cast<float*>(smem);
  constexpr int LD = Cfg::RED_LD;
  if (!KV || wave < NWAVES) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        *reinterpret_cast<v4f*>(red + (wave * BM + mt * 16 + lm) * LD + nt * 16 + lq * 4) = acc[mt][nt];
  }
  __syncthreads();
  if (KV && wave >= NWAVES) return;
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int item = it * NWAVES * 64 + tid, row = item / CHUNKS, col = (item - row * CHUNKS) * 8;
    if (row >= rows_here || col >= cols_here) continue;
    float v[8];
    {
      const float* at = red + row * LD + col;
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = at[i];
#pragma unroll
      for (int w = 1; w < NWAVES; ++w)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] += at[w * BM * LD + i];
    }
    const int64_t m = m0 + row;
    const int n = n0 + col;
    if constexpr (KV) {
      // fused QKV: the reference's bf16 roundings, then C or the row's K / V page (see tile_body)
      const int64_t row_off = row_table[row];
      if (row_off < 0 && n >= p.kv.q_dim) continue;
      float a_s = 1.f;
      if constexpr (!BLOCKSCALE) a_s = bf16_round(row_s[it]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int nn = n + i < p.N ? n + i : p.N - 1;
        float r = bf16_round(v[i]);
        if constexpr (!BLOCKSCALE) r = bf16_round(r * bf16_round(a_s * bf16_round(col_s[it][i])));
        if (p.kv.bias) r = bf16_round(r + bf16_bits_to_f32(p.kv.bias[nn]));
        v[i] = r;
      }
      *reinterpret_cast<uint4*>(kv_dst(p.kv, p.c, p.ldc, m, row_off, n)) =
          make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
      continue;
    }
    if constexpr (!BLOCKSCALE) {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = (v[i] * row_s[it]) * col_s[it][i];
    }
    if (p.c_dtype == MAXFP8_BF16) {
      uint16_t* dst = reinterpret_cast<uint16_t*>(p.c) + m * p.ldc + n;
      if (p.c_vec8_ok && n + 7 < p.N) {
        *reinterpret_cast<uint4*>(dst) =
            make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (n + i < p.N) dst[i] = (uint16_t)f32_to_bf16_bits(v[i]);
      }
    } else {
      float* dst = reinterpret_cast<float*>(p.c) + m * p.ldc + n;
      if (p.c_vec_ok && n + 7 < p.N) {
        *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(dst + 4) = make_float4(v[4], v[5], v[6], v[7]);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (n + i < p.N) dst[i] = v[i];
      }
    }
  }
}

template <int MT, int NT, bool BLOCKSCALE, int BLOCKS, bool KV>
static int launch_mid(const GemmArgs& p, hipStream_t stream) {
  using Cfg = MidCfg<MT, NT, BLOCKSCALE, BLOCKS>;
  // weights that are read once and are more than a quarter of the memory-side cache: non-temporal (10240 x 8192 at 64 tokens
  // 24.1 -> 23.2 us; smaller ones may still sit in that cache and then come quicker without: 1536 x 7168 9.4 against 12.8; from 2^23 on for tiles of
  // up to 32 tokens: 1.7 per cent from memory, -5 from the cache)
  const bool once = p.M <= Cfg::BM && (int64_t)p.N * p.K >= ((int64_t)1 << 26);
  using Args = std::conditional_t<KV, GemmArgs, MatmulArgs>;
  void (*kern)(Args, int, int) = gemm_mid_kernel<MT, NT, BLOCKSCALE, 0, BLOCKS, KV>;
  if (once) kern = gemm_mid_kernel<MT, NT, BLOCKSCALE, kStreamOnce, BLOCKS, KV>;
  static PerDeviceFlag attrs[2];
  PerDeviceFlag& attr = attrs[once];
  bool& attr_done = attr.here();
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::SMEM);
    if (e != hipSuccess) MAXFP8_FAIL(MAXFP8_ERR_LAUNCH, "gemm_mid: cannot reserve %d bytes of LDS: %s", Cfg::SMEM, hipGetErrorString(e));
    attr_done = true;
  }
  const int64_t tiles_m = ceil_div(p.M, Cfg::BM), tiles_n = ceil_div(p.N, Cfg::BN);
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3((Cfg::NWAVES + (KV ? 1 : 0)) * 64), Cfg::SMEM, stream, static_cast<const Args&>(p), (int)tiles_m, (int)tiles_n);
  return launch_status("gemm_mid");
}

int compute_units();

// The shapes that are built: 16 mt tokens x 16 nt weight rows, blocks per CU.  Of 78 measured on 300 matmuls (1 to 1000 tokens, K 512 ...
// 28672, N 512 ... 57344, both scalings), these lose 1 per cent against choosing among all of them.
struct MidShape { int mt, nt, blocks; };
#define MAXFP8_MID_SHAPES(S)                                                                                               \
  S(1, 1, 4) S(1, 2, 3) S(2, 1, 3) S(2, 2, 4) S(2, 2, 2) S(2, 3, 3) S(2, 3, 1) S(2, 4, 3) S(2, 4, 1) S(3, 1, 2) S(3, 2, 1) S(3, 3, 1) \
  S(3, 4, 2) S(3, 4, 1) S(4, 1, 1) S(4, 2, 1) S(4, 3, 1) S(4, 4, 2)
#define MAXFP8_MID_ROW(mt, nt, blocks) {mt, nt, blocks},
static const MidShape kMidShapes[] = {MAXFP8_MID_SHAPES(MAXFP8_MID_ROW)};
#undef MAXFP8_MID_ROW

// Estimated microseconds, one estimate for all shapes.  Fitted to the launches above with the operands in the memory-side cache where they fit:
// within 8 per cent for half of the launches, 19 for nine in ten; what the shapes have in common cancels where they are
// compared: the one it picks is 0.4 per cent behind the best of them on average there, 10 at most, and 0.8 with the weights from memory.  From memory a launch takes
// 1.07 to 1.2 times as long, the more the longer K is; the rules that compare it with other kernels (api.hip) were made for that.  An estimate fitted to times from
// memory instead picked no better there beyond 64 tokens (1066 matmuls: 0.6 per cent behind the best kernel and shape with either) and worse in the cache.
// Its terms: a launch; per round of blocks on the chip a start and end, the waits of the ring's rounds, and the MFMAs of a wave; per block of a CU the bytes of its
// slabs and its MFMAs; the weights' way.
static float mid_cost(const MidShape& t, int64_t M, int64_t N, int64_t K, bool blockscale) {
  const int64_t cus = compute_units(), blocks = ceil_div(M, 16 * t.mt) * ceil_div(N, 16 * t.nt);
  const float rounds = (float)ceil_div(blocks, cus * t.blocks), per_cu = (float)ceil_div(blocks, cus);
  const int64_t slabs = ceil_div(K, 128), wave_slabs = ceil_div(slabs, mid_waves(t.blocks)), depth = mid_depth(t.mt, t.nt, blockscale, t.blocks);
  const float turns = (float)ceil_div(wave_slabs, depth), walked = turns * (float)depth, mfmas = (float)(t.mt * t.nt);
  const float fetched = per_cu * (float)slabs * (float)(t.mt + t.nt), multiplied = per_cu * (float)slabs * mfmas, weights = (float)N * (float)K;
  if (blockscale)
    return 1.35f + rounds * (1.93f + 0.060f * turns + 0.0045f * walked * mfmas) + 0.0179f * fetched + 0.0033f * multiplied + 6.2e-8f * weights;
  return 1.31f + rounds * (2.60f + 0.043f * turns + 0.0023f * walked * mfmas) + 0.0160f * fetched + 0.0033f * multiplied +
         0.023f * per_cu * mfmas + 9.0e-8f * weights;
}

// What the kernel takes (with block scaling a wave's weight scales sit in its 64 lanes) and where it may be the quicker one: at most 2048 tokens
bool gemm_mid_ok(int64_t M, int64_t N, int64_t K) { return M <= 2048 && K <= 4 * 64 * 128 && ceil_div(M, 16) * ceil_div(N, 16) < ((int64_t)1 << 31); }

// The shape for an M x N x K matmul (100 * blocks per CU + 10 * mt + nt) and what it is estimated to take
int gemm_mid_shape(int64_t M, int64_t N, int64_t K, bool blockscale, float* us) {
  const MidShape* best = nullptr;
  for (const MidShape& t : kMidShapes) {
    if (t.mt > 1 && M <= 16 * (t.mt - 1)) continue;
    const float c = mid_cost(t, M, N, K, blockscale);
    if (!best || c < *us) { best = &t; *us = c; }
  }
  return 100 * best->blocks + 10 * best->mt + best->nt;
}

template <bool BLOCKSCALE, bool KV>
static int pick_mid(const GemmArgs& p, int sel, hipStream_t stream) {
#define MAXFP8_MID_CASE(mt, nt, blocks) if (sel == 100 * blocks + 10 * mt + nt) return launch_mid<mt, nt, BLOCKSCALE, blocks, KV>(p, stream);
  MAXFP8_MID_SHAPES(MAXFP8_MID_CASE)
#undef MAXFP8_MID_CASE
  MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "mid matmul: unknown shape selector %d", sel);
}

// The tuning switch names a shape as <blocks per CU><mt><nt>, or a tile as <mt><nt>: the first shape above with that tile
int gemm_mid_forced_shape() {
  const int sel = tuning().mid;
  if (sel >= 100) return sel;
  for (const MidShape& t : kMidShapes)
    if (10 * t.mt + t.nt == sel) return 100 * t.blocks + sel;
  return sel;
}

// sel: the shape, as gemm_mid_shape names it
int gemm_mid_dispatch(const GemmArgs& p, bool blockscale, int sel, hipStream_t stream) {
  if (p.kv_on) return blockscale ? pick_mid<true, true>(p, sel, stream) : pick_mid<false, true>(p, sel, stream);
  return blockscale ? pick_mid<true, false>(p, sel, stream) : pick_mid<false, false>(p, sel, stream);
}

}  // namespace maxfp8
