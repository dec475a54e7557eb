// Batched block-scaled FP8 matmul for short K, one to four 128-wide slabs: the products of latent attention, whose weights are one small matrix
// per head.  Such a matmul has next to no arithmetic per byte and no pipeline fills: the decode kernel splits K over four waves, of
// which one slab of K leaves three idle, and the tiles' stages along K have nothing to hide behind.  Two kernels:
//   gemm_one_slab_kernel   one slab, any number of tokens
//   gemm_short_k_kernel    two to four slabs, at most 32 tokens
#include <utility>

#include "common.h"
#include "gemm_args.h"
#include "gemm_device.h"
#include "tuning.h"

namespace maxfp8 {

// ---- two to four slabs, at most 32 tokens ----------------------------------------------------------------------
// A wave takes 32 weight rows and 16 tokens with ALL of their K into registers, straight in the MFMA's operand layout: no LDS, no
// barrier, no split, every load of the wave in flight at once.
//
// Bound: the bytes (weights and activations once, bf16 results once) and one trip to memory and back.  Measured, graph
// timing, operands cold, 128 heads, K = 512, N = 128: M = 1 / 16 / 32 tokens 4.9 / 5.6 / 5.7 us where the decode kernel took 5.9 / 8.5 / 11.8
// and the 128 x 128 tiles take 6.2 / 6.4 / 6.3.
// NS slabs of K.  grid: (128-column blocks, groups of 16 tokens, batches)
template <int NS>
__global__ __launch_bounds__(256) void gemm_short_k_kernel(MatmulArgs p_in) {
  const MatmulArgs p = batch_view(p_in, blockIdx.z);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lq = lane >> 4;
  const int n0 = ((int)blockIdx.x * 4 + wave) * 32;
  if (n0 >= p.N) return;
  const uint32_t m = blockIdx.y * 16 + lm;

  const __amdgpu_buffer_rsrc_t a_rsrc = t2_rsrc(p.a, t2_clamp_u32((int64_t)(p.M - 1) * p.lda + p.K));
  const __amdgpu_buffer_rsrc_t b_rsrc = t2_rsrc(p.b + (int64_t)n0 * p.ldb, t2_clamp_u32((int64_t)(p.N - n0 - 1) * p.ldb + p.K));
  const __amdgpu_buffer_rsrc_t s_rsrc = t2_rsrc(p.a_scales, t2_clamp_u32(((int64_t)(NS - 1) * p.a_scales_ld + p.M) * 4));
  // lane (lm, lq) of a fragment holds K bytes [16 * lq, +16) and [64 + 16 * lq, +16) of its row, as in the other kernels
  auto load_frag = [](__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t k) -> v8i {
    const v4i lo = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, voff, k * 128u, 0));
    const v4i hi = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, voff, k * 128u + 64u, 0));
    return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  };

  // Weight fragments in pairs over 32 rows: MFMA row i of the even fragment is weight row 8 * (i / 4) + i % 4, of the odd
  // one 4 more, which leaves a lane eight consecutive columns of one token.
  v8i w[2][NS], a[NS];
  float as[NS], bs[NS];
  const uint32_t wrow = 8u * (lm >> 2) + (lm & 3);
#pragma unroll
  for (int k = 0; k < NS; ++k)
#pragma unroll
    for (int h = 0; h < 2; ++h) w[h][k] = load_frag(b_rsrc, (wrow + 4u * h) * (uint32_t)p.ldb + (uint32_t)lq * 16u, k);
#pragma unroll
  for (int k = 0; k < NS; ++k) {  // (tokens past M read as zero)
    a[k] = load_frag(a_rsrc, m * (uint32_t)p.lda + (uint32_t)lq * 16u, k);
    as[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, m < (uint32_t)p.M ? m * 4u : 0x80000000u,
                                                                            (uint32_t)k * (uint32_t)p.a_scales_ld * 4u, 0));
  }
  const float* bs_row = p.b_scales + (int64_t)(n0 / 128) * p.b_scales_ld;
#pragma unroll
  for (int k = 0; k < NS; ++k) bs[k] = bs_row[k];

  v4f acc[2];
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    const float s = as[k] * bs[k];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[h][k], a[k], zero, 0, 0, 0, 0, 0, 0);
      if (k == 0) acc[h] = part * s;
      else acc[h] += part * s;
    }
  }
  if (m < (uint32_t)p.M)
    *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p.c) + (int64_t)m * p.ldc + n0 + lq * 8) =
        make_uint4(pack_bf16x2(acc[0][0], acc[0][1]), pack_bf16x2(acc[0][2], acc[0][3]), pack_bf16x2(acc[1][0], acc[1][1]),
                   pack_bf16x2(acc[1][2], acc[1][3]));
}

// ---- one slab of K ----------------------------------------------------------------------------------------------
// A block owns 128 columns of one matrix of the batch, a wave 32 of them, whose weights (a 128-byte row each) sit in registers; the tokens come by in
// chunks of 16 * MT through LDS, copied whole lines at a time for the four waves together (straight into the MFMA's layout, 16 rows x 64 bytes per
// instruction, an L1 delivers 16 bytes a clock), the next chunk's copies in front of this one's MFMAs and stores.
//
// Bound: the bytes, of which the bf16 results are most, and a start of three microseconds.  The tiles of gemm_tiled.hip stage 128 or 256 rows, whole or not,
// and their results again, and store in bursts; with all operands in a wave's registers, as below, an L1 delivers the tokens once per 32 columns.
//   * The column blocks of a matrix's rows sit on one XCD, one behind the other (blocks go to the XCDs round-robin): its L2 reads the tokens once and holds whole
//     rows of the result, where four of them each wrote every fourth 256 bytes.  128 heads of 1000 tokens, 128 -> 512, results from the cache 39.0 -> 26.3 us.
//   * Stores pass the L2 (device scope) without staying in it: 48.6 -> 30.3 us with the results going to memory, and 26.3 -> 28.3 from the cache; non-temporal alone 41 and 40,
//     device scope alone 58 and 26.  112 tokens 9.2 -> 7.7 and 7.4 -> 6.1.  Non-temporal alone where four blocks per CU and more take two chunks at most (of more than 16 tokens): all of their
//     stores come at once, and 100 tokens of 128 -> 1024 are 13.1 and 9.0 us with it, 14.4 and 8.2 at device scope, 13.1 and 10.1 with neither.
//   * Two blocks per CU walk the chunks of more: the weights are read once per block, and a mostly empty last chunk costs little.  80 tokens 7.4 -> 5.5 and 6.0 -> 4.9.
// Graph timing, 128 heads of 128 -> 512, results to memory (four sets of operands in turn) / from the cache (one), the tiles and this kernel: 48 tokens 6.9 / 6.2 and 4.6 / 4.2,
// 80 8.1 / 6.9 and 5.5 / 4.9, 200 12.6 / 11.0 and 8.1 / 7.4, 400 21.3 / 20.3 and 13.1 / 12.4, 1000 42.3 / 38.5 and 27.8 / 27.3, 1500 59.5 / 50.5 and 45.6 / 44.5 (bytes at
// 6 TB/s: 2.6, 3.7, 7.1, 13, 28, 41).  Before the three: 5.5 / 4.9, 9.5 / 8.1, 14.5 / 11.9, 23.1 / 17.5, 51.5 / 38.7, 78.1 / 51.3.
constexpr int kNonTemporal = 2, kPastL2 = 18;  // (device scope and non-temporal)
// grid: (XCDs, 128-column blocks, the walkers of all matrices over the XCDs)
template <int MT, int STORE_POLICY>
__global__ __launch_bounds__(256) void gemm_one_slab_kernel(MatmulArgs p_in, int walkers, int batch) {
  constexpr int CHUNK = 16 * MT, A_BYTES = MT * 2048, COPIES = 2 * MT;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[16384 + 2 * (A_BYTES + 256)];
  // (all arguments at once: behind the branches their loads would begin when those of the two counts are back, 0.1 us of the shortest launches)
  asm volatile("" ::"s"(p_in.a), "s"(p_in.b), "s"(p_in.c), "s"(p_in.a_scales), "s"(p_in.b_scales), "s"(p_in.M), "s"(p_in.N), "s"(p_in.K), "s"(p_in.lda), "s"(p_in.ldb),
               "s"(p_in.ldc), "s"(p_in.b_scales_ld), "s"(p_in.a_batch), "s"(p_in.b_batch), "s"(p_in.c_batch), "s"(p_in.a_scales_batch), "s"(p_in.b_scales_batch), "s"(walkers), "s"(batch));
  const int walker = (int)blockIdx.z * 8 + (int)blockIdx.x;
  int matrix = walker, first = 0;
  if (walkers > 1) {
    matrix = walker / walkers;
    first = walker - matrix * walkers;
  }
  if (matrix >= batch) return;
  const MatmulArgs p = batch_view(p_in, matrix);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lq = lane >> 4, cr = lane >> 3, cp = lane & 7;
  const int n0 = ((int)blockIdx.y * 4 + wave) * 32;
  const int chunks = (p.M + CHUNK - 1) / CHUNK;

  // rows past M, columns past N (whole waves: N is a multiple of 32) and scales past M read as zero through the descriptors
  const __amdgpu_buffer_rsrc_t a_rsrc = t2_rsrc(p.a, t2_clamp_u32((int64_t)(p.M - 1) * p.lda + p.K));
  const __amdgpu_buffer_rsrc_t b_rsrc = t2_rsrc(p.b + (int64_t)n0 * p.ldb, n0 < p.N ? t2_clamp_u32(31 * p.ldb + p.K) : 0u);
  const __amdgpu_buffer_rsrc_t s_rsrc = t2_rsrc(p.a_scales, (uint32_t)p.M * 4u);
  const __amdgpu_buffer_rsrc_t c_rsrc = t2_rsrc(p.c, t2_clamp_u32(((int64_t)(p.M - 1) * p.ldc + p.N) * 2));
  // copies of 8 rows x 128 bytes; row r of the tokens keeps its chunk c at c ^ (r & 7), of the weights as the pairs of fragments below read them
  uint8_t* const w_lds = smem + wave * 4096;
  auto a_lds = [&](int buf) { return smem + 16384 + buf * (A_BYTES + 256); };
  const uint32_t a_voff = (uint32_t)cr * (uint32_t)p.lda + (uint32_t)((cp ^ cr) * 16);
  auto send = [&](int chunk, int buf) {
    const uint32_t row = (uint32_t)chunk * CHUNK;
    for (int i = wave; i < COPIES; i += 4)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(a_lds(buf) + i * 1024), 16, a_voff, (row + i * 8) * (uint32_t)p.lda, 0, 0);
    if (wave == 3) __builtin_amdgcn_raw_ptr_buffer_load_lds(s_rsrc, (lds_ptr_t)(a_lds(buf) + A_BYTES), 4, (uint32_t)lane * 4u, row * 4u, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t chunk = (uint32_t)(cp ^ (((i & 1) << 2) | (cr & 3)));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (lds_ptr_t)(w_lds + i * 1024), 16, (uint32_t)cr * (uint32_t)p.ldb + chunk * 16u, (uint32_t)(i * 8) * (uint32_t)p.ldb, 0, 0);
  }
  int chunk = first;
  send(chunk, 0);
  const float bs = n0 < p.N ? p.b_scales[(int64_t)(n0 / 128) * p.b_scales_ld] : 0.f;

  auto frag = [](const uint8_t* row, int lo, int hi) {
    const v4i l = *reinterpret_cast<const v4i*>(row + lo * 16), h = *reinterpret_cast<const v4i*>(row + hi * 16);
    return v8i{l.x, l.y, l.z, l.w, h.x, h.y, h.z, h.w};
  };
  // Weight fragments in pairs over the 32 rows, as above: a lane is left with eight consecutive columns of one token
  const int wrow = 8 * (lm >> 2) + (lm & 3), wsw = (((wrow >> 3) & 1) << 2) | (wrow & 3);
  v8i w[2];
  const uint32_t c_voff = ((uint32_t)lm * (uint32_t)p.ldc + (uint32_t)(n0 + lq * 8)) * 2u | (n0 < p.N ? 0u : 0x80000000u);
  for (int buf = 0;; buf ^= 1) {
    // this wave's copies of the chunk have landed (behind them only the MT stores of the chunk before), then everyone's
    if (chunk == first) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MT) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (chunk == first) {
#pragma unroll
      for (int h = 0; h < 2; ++h) w[h] = frag(w_lds + (wrow + 4 * h) * 128, lq ^ wsw, (lq + 4) ^ wsw);
    }
    v8i a[MT];
    float as[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      a[t] = frag(a_lds(buf) + (t * 16 + lm) * 128, lq ^ (lm & 7), (lq + 4) ^ (lm & 7));
      as[t] = *reinterpret_cast<const float*>(a_lds(buf) + A_BYTES + (t * 16 + lm) * 4);
    }
    const int next = chunk + walkers;
    // (the other buffer: every wave has read it before this chunk's barrier)
    if (next < chunks) send(next, buf ^ 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const v4f zero = {0.f, 0.f, 0.f, 0.f};
      const float s = as[t] * bs;
      float v[8];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[h], a[t], zero, 0, 0, 0, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[4 * h + i] = fmaf(part[i], s, 0.0f);  // (the tiles' sum of one slab)
      }
      const uint32_t m = (uint32_t)(chunk * CHUNK + t * 16);
      const uint32_t at = (c_voff + m * (uint32_t)p.ldc * 2u) | (m + (uint32_t)lm < (uint32_t)p.M ? 0u : 0x80000000u);
      __builtin_amdgcn_raw_buffer_store_b128(v4u_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])}, c_rsrc, at, 0, STORE_POLICY);
    }
    if (next >= chunks) break;
    chunk = next;
  }
}

int compute_units();

// Batches of one slab of K and whole 32-column groups, bf16 results with 16-byte rows, offsets of 31 bits
bool gemm_one_slab_ok(const GemmArgs& p, bool blockscale, int64_t batch) {
  const int64_t rows = (int64_t)p.M + 64, lim = (int64_t)1 << 31;
  return blockscale && tuning().short_k && batch > 1 && !p.kv_on && p.K == 128 && p.N % 32 == 0 && p.N <= 128 * 65535 && p.c_dtype == MAXFP8_BF16 && p.c_vec8_ok &&
         rows * p.lda < lim && 32 * p.ldb < lim && rows * p.ldc * 2 < lim;
}
template <int MT>
static int launch_one_slab(const GemmArgs& p, int64_t batch, hipStream_t stream) {
  // a walker per chunk up to two blocks per CU; beyond, so many walk the chunks, the same number each (see above)
  const int64_t cus = compute_units(), columns = ceil_div(p.N, 128), chunks = ceil_div(p.M, 16 * MT), fit = 2 * cus / (columns * batch);
  const int64_t walkers = ceil_div(chunks, ceil_div(chunks, fit > 1 ? fit : 1));
  const bool at_once = columns * batch >= 4 * cus && chunks <= 2 && p.M > 16;
  hipLaunchKernelGGL((at_once ? gemm_one_slab_kernel<MT, kNonTemporal> : gemm_one_slab_kernel<MT, kPastL2>), dim3(8, (unsigned)columns, (unsigned)ceil_div(walkers * batch, 8)), dim3(256), 0, stream, static_cast<const MatmulArgs&>(p), (int)walkers, (int)batch);
  return launch_status("gemm_one_slab");
}
int gemm_one_slab_dispatch(const GemmArgs& p, int64_t batch, hipStream_t stream) {
  if (p.M <= 32) return p.M <= 16 ? launch_one_slab<1>(p, batch, stream) : launch_one_slab<2>(p, batch, stream);
  return p.M <= 48 ? launch_one_slab<3>(p, batch, stream) : launch_one_slab<4>(p, batch, stream);
}

// Batches of at most 32 tokens, two to four whole slabs and whole 32-column groups, bf16 results with 16-byte rows; every other shape
// keeps the other kernels.  With three or four slabs the decode kernel's waves all have a share, and it stays ahead while its
// 16-row blocks are at most two per CU (16 heads of 512 -> 128: 3.1 against 4.0 us at M = 1; 128 heads: 5.9 against 4.9) and,
// with two groups of tokens, which are a wave each here and one pass over the weights there, at most one (17 to 32 tokens: 16 and
// 32 heads of 512 -> 128 4.5 and 4.7 us against 5.4 and 5.3, 48 heads 6.3 against 5.9).
bool gemm_short_k_ok(const GemmArgs& p, bool blockscale, int64_t batch) {
  if (!blockscale || !tuning().short_k || batch < 2 || p.kv_on || p.M > 32 || p.K % 128 != 0 || p.K < 256 || p.K > 512 || p.N % 32 != 0 ||
      p.c_dtype != MAXFP8_BF16 || !p.c_vec8_ok)
    return false;
  return p.K <= 256 || ceil_div(p.N, 16) * batch > (p.M > 16 ? 1 : 2) * (int64_t)compute_units();
}

template <int NS>
static int launch_short_k(const GemmArgs& p, int64_t batch, hipStream_t stream) {
  hipLaunchKernelGGL(gemm_short_k_kernel<NS>, dim3((unsigned)ceil_div(p.N, 128), (unsigned)ceil_div(p.M, 16), (unsigned)batch), dim3(256), 0, stream, static_cast<const MatmulArgs&>(p));
  return launch_status("gemm_short_k");
}

int gemm_short_k_dispatch(const GemmArgs& p, int64_t batch, hipStream_t stream) {
  switch (p.K / 128) {
    case 2: return launch_short_k<2>(p, batch, stream);
    case 3: return launch_short_k<3>(p, batch, stream);
    default: return launch_short_k<4>(p, batch, stream);
  }
}

}  // namespace maxfp8
