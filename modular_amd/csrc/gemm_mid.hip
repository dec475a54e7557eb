// Scaled FP8 matmul for batches between decode and prefill (tens to a few hundred tokens): C[M,N] = A[M,K] . B[N,K]^T.
//
// Such a matmul is a few dozen 128 x 128 tiles: too few for the chip, so the tile kernels cut K over blocks and pay for it
// with a second launch (or a hand-over) and the partial sums' way to memory and back.  Here the K split stays inside a
// block: a block owns a small tile, 16 * MT tokens x 16 * NT weight rows, its four waves a quarter of K each, and the
// four partial tiles meet in LDS.  Small tiles make enough blocks for the chip without a cut.
//
//   * Each wave has an LDS ring of its own: a slot holds one 128-wide slab of the tile's weight rows AND token rows (and
//     their scales), copied by LDS-DMA in whole 128-byte lines.  No barrier in the loop; waits are exact counts.
//   * A slot's fragments are read into registers at once and the slot is refilled before they are multiplied, so DEPTH
//     slabs stay in flight per wave nearly all the time.
//   * Epilogue: partial sums to LDS as [token][column], a thread adds the four (in wave order) for eight columns of a token,
//     scales, converts and stores 16 bytes.  The fused QKV projection's page look-ups are made before the loop.
//
// Bound: what a CU can pull out of the L2s -- every block fetches its tokens and weights itself, 16 * (MT + NT) * K bytes, and
// 40 KB per wave hold two to six slabs in flight.  Measured (graph timing, operands cold) against what ran these shapes
// before: 117 x 6144 x 4096 20.0 -> 13.1 us, 117 x 4096 x 4096 19.9 -> 10.7, 64 x 4096 x 4096 12.3 -> 8.3, 256 x 1536 x 7168 16.9 ->
// 11.2, 256 x 576 x 7168 15.2 -> 9.0; the fused QKV projection of 64 tokens (10240 x 8192) 36.9 -> 23.6.  Bytes at 6 TB/s: 4.5,
// 3.0, 2.9, 2.3, 1.0 and 14.3.
#include <type_traits>
#include <utility>

#include "common.h"
#include "gemm_args.h"
#include "gemm_device.h"
#include "tuning.h"

namespace maxfp8 {

// Slabs in flight per wave: a quarter of the LDS, the 6-bit wait counter, at most six
__host__ __device__ constexpr int mid_depth(int mt, int nt, bool blockscale) {
  const int slot = (mt + nt) * 2048 + (blockscale ? 256 : 0), per = 2 * (mt + nt) + (blockscale ? 1 : 0);
  const int lds = (160 * 1024 - 16 * mt * 8) / 4 / slot, counter = 63 / per + 1, least = lds < counter ? lds : counter;
  return least > 6 ? 6 : least;
}

template <int MT, int NT, bool BLOCKSCALE>
struct MidCfg {
  static constexpr int BM = 16 * MT, BN = 16 * NT;
  static constexpr int SCALES = BLOCKSCALE ? 256 : 0;        // 64 activation scales: one copy
  static constexpr int SLOT = (MT + NT) * 2048 + SCALES;
  static constexpr int PER = 2 * (MT + NT) + (BLOCKSCALE ? 1 : 0);  // copies per wave and slab
  static constexpr int ROW_TABLE = BM * 8;                   // fused QKV: the cache row of every token
  static constexpr int DEPTH = mid_depth(MT, NT, BLOCKSCALE);
  static constexpr int RING = DEPTH * SLOT;
  static constexpr int RED_LD = BN + 4;                      // floats per token row of a partial tile
  static constexpr int RED = 4 * BM * RED_LD * 4;
  static constexpr int SMEM = (4 * RING > RED ? 4 * RING : RED) + ROW_TABLE;
  static_assert(MT <= 4 && DEPTH >= 2 && SMEM <= 160 * 1024);
};

template <int MT, int NT, bool BLOCKSCALE, int W_POLICY>
__global__ __launch_bounds__(256) void gemm_mid_kernel(GemmArgs p, int tiles_m, int tiles_n) {
  using Cfg = MidCfg<MT, NT, BLOCKSCALE>;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, DEPTH = Cfg::DEPTH, PER = Cfg::PER, SLOT = Cfg::SLOT;
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
  const int per_wave = (nslab + 3) / 4;
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

  v4f acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // the PER copies of a slab; a slab past the wave's share fetches nothing (and writes zeros), so the counts stay exact
  auto issue = [&](int slab, int d) {
    const bool live = slab < s_end;
    const int sl = live ? slab : s_begin;
    const uint32_t koff = __builtin_amdgcn_readfirstlane((uint32_t)sl * 128u);
    uint32_t kill = live ? 0u : 0x80000000u;
    const uint32_t kill_s = kill;
    if (k_tail && koff + cchunk * 16 >= (uint32_t)p.K) kill = 0x80000000u;
    uint8_t* slot = ring + d * SLOT;
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (lds_ptr_t)(slot + i * 1024), 16, b_voff | kill, koff + i * b_step, 0, W_POLICY);
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(slot + (2 * NT + i) * 1024), 16, a_voff | kill, koff + i * a_step, 0, 0);
    if constexpr (BLOCKSCALE)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(s_rsrc, (lds_ptr_t)(slot + (MT + NT) * 2048), 4, s_voff | kill_s,
                                               (uint32_t)sl * (uint32_t)p.a_scales_ld * 4u, 0, 0);
  };
  auto step = [&](int slab, int d) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * PER) : "memory");
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
    if constexpr (BLOCKSCALE) as = *reinterpret_cast<const v4f*>(slot + (MT + NT) * 2048 + lm * 16);
    // the slot's bytes are in registers before it is refilled
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    issue(slab + DEPTH, d);
    if constexpr (BLOCKSCALE) {
      // (a slab past the share's end multiplies zeros; its scales are finite)
      const int at = __builtin_amdgcn_readfirstlane(slab - s_begin);
      const float b0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, bs_lo), at));
      const float b1 = NT == 3 ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, bs_hi), at)) : b0;
      const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[nt], af[mt], zero, 0, 0, 0, 0, 0, 0);
          acc[mt][nt] += part * (as[mt] * (NT == 3 && nt >= nt_hi ? b1 : b0));
        }
    } else {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[nt], af[mt], acc[mt][nt], 0, 0, 0, 0, 0, 0);
    }
  };

#pragma unroll
  for (int d = 0; d < DEPTH; ++d) issue(s_begin + d, d);
  if constexpr (BLOCKSCALE)  // (the weight scales are older than the copies: they arrive without waiting for those)
    asm volatile("s_waitcnt vmcnt(%2)" : "+v"(bs_lo), "+v"(bs_hi) : "n"(DEPTH * PER < 63 ? DEPTH * PER : 63));
  if (p.kv_on && tid < BM) row_table[tid] = tid < rows_here ? kv_row_offset(p.kv, m0 + tid) : -1;
  for (int base = s_begin; base < s_end; base += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) step(base + d, d);
  }
  // drain: the last DEPTH copies fetched nothing but still write their slots
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // ---- the four partial tiles meet ------------------------------------------------------------------------------
  float* red = reinterpret_cast<float*>(smem);
  constexpr int LD = Cfg::RED_LD;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      *reinterpret_cast<v4f*>(red + (wave * BM + mt * 16 + lm) * LD + nt * 16 + lq * 4) = acc[mt][nt];
  __syncthreads();
  constexpr int CHUNKS = BN / 8;
  for (int item = tid; item < BM * CHUNKS; item += 256) {
    const int row = item / CHUNKS, col = (item - row * CHUNKS) * 8;
    if (row >= rows_here || col >= cols_here) continue;
    float v[8];
    {
      const float* at = red + row * LD + col;
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = at[i];
#pragma unroll
      for (int w = 1; w < 4; ++w)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] += at[w * BM * LD + i];
    }
    const int64_t m = m0 + row;
    const int n = n0 + col;
    if (p.kv_on) {
      // fused QKV: the reference's bf16 roundings, then C or the row's K / V page (see tile_body)
      const int64_t row_off = row_table[row];
      if (row_off < 0 && n >= p.kv.q_dim) continue;
      float a_s = 1.f;
      if constexpr (!BLOCKSCALE) a_s = bf16_round(p.a_scales[m * p.a_scale_stride]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int nn = n + i < p.N ? n + i : p.N - 1;
        float r = bf16_round(v[i]);
        if constexpr (!BLOCKSCALE) r = bf16_round(r * bf16_round(a_s * bf16_round(p.b_scales[(int64_t)nn * p.b_scale_stride])));
        if (p.kv.bias) r = bf16_round(r + bf16_bits_to_f32(p.kv.bias[nn]));
        v[i] = r;
      }
      *reinterpret_cast<uint4*>(kv_dst(p.kv, p.c, p.ldc, m, row_off, n)) =
          make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
      continue;
    }
    if constexpr (!BLOCKSCALE) {
      const float a_s = scale_at(p.a_scales, m * p.a_scale_stride, p.scales_dtype);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int nn = n + i < p.N ? n + i : p.N - 1;
        v[i] = (v[i] * a_s) * scale_at(p.b_scales, (int64_t)nn * p.b_scale_stride, p.scales_dtype);
      }
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

template <int MT, int NT, bool BLOCKSCALE>
static int launch_mid(const GemmArgs& p, hipStream_t stream) {
  using Cfg = MidCfg<MT, NT, BLOCKSCALE>;
  // weights that are read once and are more than a quarter of the memory-side cache: non-temporal (10240 x 8192 at 64 tokens
  // 24.1 -> 23.2 us; smaller ones may still sit in that cache and then come quicker without: 1536 x 7168 9.4 against 12.8)
  const bool once = p.M <= Cfg::BM && (int64_t)p.N * p.K >= ((int64_t)1 << 26);
  auto kern = once ? gemm_mid_kernel<MT, NT, BLOCKSCALE, kStreamOnce> : gemm_mid_kernel<MT, NT, BLOCKSCALE, 0>;
  static PerDeviceFlag attrs[2];
  PerDeviceFlag& attr = attrs[once];
  bool& attr_done = attr.here();
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::SMEM);
    if (e != hipSuccess) MAXFP8_FAIL(MAXFP8_ERR_LAUNCH, "gemm_mid: cannot reserve %d bytes of LDS: %s", Cfg::SMEM, hipGetErrorString(e));
    attr_done = true;
  }
  const int64_t tiles_m = ceil_div(p.M, Cfg::BM), tiles_n = ceil_div(p.N, Cfg::BN);
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3(256), Cfg::SMEM, stream, p, (int)tiles_m, (int)tiles_n);
  return launch_status("gemm_mid");
}

int compute_units();
float gemm_skinny_cost(int64_t M, int64_t N, int64_t K, bool blockscale);

// Estimated times (microseconds), fitted to launches of every kernel on 26 weight matrices (K 512 ... 28672, N 576 ... 32768)
// at 4 to 400 tokens in both scale modes, operands cold: within 15 per cent for nine launches in ten.
//
// This kernel: a start, per round of blocks a fixed part and a slab's time of the tile shape, the bytes of all blocks'
// operands (out of the L2s), and not less than the weights take from memory.
struct MidShape { int mt, nt; float start, round, slab, traffic; };
static const MidShape kMidShapes[12] = {
    {2, 1, 1.84f, 3.33f, 0.037f, 3.32f}, {2, 2, 1.82f, 2.93f, 0.066f, 2.91f}, {2, 3, 2.07f, 2.97f, 0.093f, 3.17f}, {2, 4, 2.17f, 3.25f, 0.121f, 2.89f},
    {3, 1, 2.01f, 2.75f, 0.061f, 2.31f}, {3, 2, 1.91f, 2.98f, 0.091f, 2.44f}, {3, 3, 2.55f, 3.87f, 0.115f, 2.80f}, {3, 4, 1.69f, 4.01f, 0.166f, 2.16f},
    {4, 1, 1.75f, 2.91f, 0.069f, 2.30f}, {4, 2, 1.90f, 3.56f, 0.104f, 2.13f}, {4, 3, 1.45f, 4.38f, 0.144f, 1.90f}, {4, 4, 1.43f, 4.97f, 0.181f, 2.27f}};
static float mid_cost(const MidShape& t, int64_t M, int64_t N, int64_t K) {
  const int64_t blocks = ceil_div(M, 16 * t.mt) * ceil_div(N, 16 * t.nt);
  const float slabs = (float)(ceil_div(K, 512) * 4);
  float us = t.start + (float)ceil_div(blocks, compute_units()) * (t.round + slabs * t.slab) +
                   t.traffic * (float)(blocks * 16 * (t.mt + t.nt)) * (float)K * 1e-8f;
  // (the fit reads long K on weights from 32 MB short: 9728 x 5328 at 59 tokens 22.7 us against the K split's 19.7; on smaller
  // ones it does not: 9600 x 2416 at 45 tokens 14.5 against the decode kernel's 19.3)
  if (K > 9216 && N * K >= ((int64_t)1 << 25)) us *= 1.25f;
  const float stream = 4.0f + (float)N * (float)K / 5.2e6f;
  return us > stream ? us : stream;
}

// What the estimate holds for: at most 320 tokens, K up to 12288 (beyond, the decode kernel and the K split's tiles win from
// both sides: 14336 x 4096 at 24 tokens 17.4 against 20 us, at 117 tokens 26.6 against 28.4) and weights under 128 MB (25024 x
// 6400 at 45 tokens 40 against 44).  (In any case at most 58 slabs per wave: their weight scales sit in its 64 lanes.)
bool gemm_mid_ok(int64_t M, int64_t N, int64_t K) { return M <= 320 && K <= 12288 && N * K < ((int64_t)1 << 27); }

// The shape for an M x N x K matmul (10 * MT + NT) and what it is estimated to take
int gemm_mid_shape(int64_t M, int64_t N, int64_t K, float* us) {
  int best = 0;
  *us = 0.f;
  for (const MidShape& t : kMidShapes) {
    if (t.mt > 2 && M <= 16 * (t.mt - 1)) continue;
    const float c = mid_cost(t, M, N, K);
    if (best == 0 || c < *us) { best = 10 * t.mt + t.nt; *us = c; }
  }
  return best;
}

// What that shape takes at 33 to 64 rows, for the comparison with the decode kernel: one estimate per scaling, with the slabs of
// a wave in whole rounds of its ring (the launches of gemm_skinny_cost: within 9 per cent for nine in ten)
float gemm_mid_cost(int64_t M, int64_t N, int64_t K, bool blockscale) {
  float us;
  const int sel = gemm_mid_shape(M, N, K, &us), mt = sel / 10, nt = sel % 10, depth = mid_depth(mt, nt, blockscale);
  const float rounds = (float)ceil_div(ceil_div(M, 16 * mt) * ceil_div(N, 16 * nt), compute_units());
  const int64_t slabs = ceil_div(K, 512);
  const float walked = (float)(ceil_div(slabs, depth) * depth), stream = (float)N * (float)K * 1e-8f;
  if (blockscale) return 1.91f + 12.6f * stream + rounds * (1.46f + 0.139f * (float)(mt * nt) + 0.049f * (float)(slabs * (mt + nt)) + 0.214f * walked);
  return 1.58f + 10.9f * stream + rounds * (2.15f + 0.188f * (float)(mt * nt) + 0.058f * (float)(slabs * (mt + nt)) + 0.162f * walked);
}

// The kernel here or the decode kernel, 17 to 64 rows.
// Up to 32 rows the decode kernel reads the tokens with half the loads and is ahead or level nearly everywhere (17 / 24 / 32 x 1536 x
// 7168 8.8 / 9.9 / 11.0 us against 10.2 / 10.7 / 11.4, 20 x 5040 x 6528 11.0 against 12.4, 28 x 24624 x 2560 20.8 against 21.8) but
// where its third block per CU runs all but alone: 22 x 9648 x 6912 0.81 of its time, 27 x 11328 x 1152 0.87 (shorter K: 1.0 to 1.1).
// Beyond, by the estimates: 33 x 4096 x 4096 9.7 against 8.2 us, 47 x 9152 x 1024 9.9 against 7.1 -- but 36 x 6272 x 512 5.0 against
// 5.8 and, with row scales, 39 x 21600 x 896 11.6 against 15.2 (block scales: 14.4 and 12.8).
bool gemm_mid_before_skinny(int64_t M, int64_t N, int64_t K, bool blockscale, bool qkv) {
  if (!gemm_mid_ok(M, N, K)) return false;
  if (M <= 32) return K > 1024 && ceil_div(ceil_div(N, 16), compute_units()) == 3;
  // (Beyond 3072 the estimate here is the higher one of the two by 6 per cent.  The fused QKV projection's epilogue costs more here, a
  // microsecond per block and round: 48 x 2048 x 1536 7.0 against 7.7 us, 56 x 7168 x 5120 17.7 against 18.8, with row scales 18.2, 48 x
  // 17408 x 2048 with row scales 20.9 against 26.7.)
  const float margin = qkv ? (K < 3072 ? 0.90f : blockscale ? 0.95f : 1.06f) : K > 3072 ? 1.06f : 1.0f;
  return gemm_mid_cost(M, N, K, blockscale) < margin * gemm_skinny_cost(M, N, K, blockscale);
}

template <bool BLOCKSCALE>
static int pick_mid(const GemmArgs& p, int sel, hipStream_t stream) {
  switch (sel) {
    case 21: return launch_mid<2, 1, BLOCKSCALE>(p, stream);
    case 22: return launch_mid<2, 2, BLOCKSCALE>(p, stream);
    case 23: return launch_mid<2, 3, BLOCKSCALE>(p, stream);
    case 24: return launch_mid<2, 4, BLOCKSCALE>(p, stream);
    case 31: return launch_mid<3, 1, BLOCKSCALE>(p, stream);
    case 32: return launch_mid<3, 2, BLOCKSCALE>(p, stream);
    case 33: return launch_mid<3, 3, BLOCKSCALE>(p, stream);
    case 34: return launch_mid<3, 4, BLOCKSCALE>(p, stream);
    case 41: return launch_mid<4, 1, BLOCKSCALE>(p, stream);
    case 42: return launch_mid<4, 2, BLOCKSCALE>(p, stream);
    case 43: return launch_mid<4, 3, BLOCKSCALE>(p, stream);
    case 44: return launch_mid<4, 4, BLOCKSCALE>(p, stream);
    default: MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "mid matmul: unknown shape selector %d", sel);
  }
}

int gemm_mid_dispatch(const GemmArgs& p, bool blockscale, hipStream_t stream) {
  float us;
  const int sel = tuning().mid > 0 ? tuning().mid : gemm_mid_shape(p.M, p.N, p.K, &us);
  return blockscale ? pick_mid<true>(p, sel, stream) : pick_mid<false>(p, sel, stream);
}

}  // namespace maxfp8
