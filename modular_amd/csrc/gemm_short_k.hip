// Batched block-scaled FP8 matmul for short K (one to four 128-wide slabs) and at most 32 tokens: the products of latent
// attention in decode, whose weights are one small matrix per head.
//
// Such a matmul has next to no arithmetic per byte and no pipeline fills: the decode kernel splits K over four waves, of
// which one slab of K leaves three idle.  Here a wave takes 32 weight rows and 16 or 32 tokens with ALL of their K into
// registers, straight in the MFMA's operand layout: no LDS, no barrier, no split, every load of the wave in flight at once.
//
// Bound: the bytes (weights and activations once, bf16 results once) and one trip to memory and back.  Measured, graph
// timing, operands cold, 128 heads, K = 128, N = 512: M = 1 / 16 / 32 tokens 3.9 / 4.6 / 5.6 us where the decode kernel took
// 14.6 / 15.7 / 27.3 and the 128 x 128 tiles take 5.4 / 5.8 / 6.2 (bytes at 5 TB/s: 1.7 / 2.2 / 2.6); K = 512, N = 128:
// 4.9 / 5.6 / 5.7 against 5.9 / 8.5 / 11.8 and 6.2 / 6.4 / 6.3.  Beyond 32 tokens the tiles, which share the tokens through LDS
// instead of re-reading them for every 32 columns, are level (48: 6.5 against 6.6) and then ahead (100: 10.5 against 8.2).
// Wider waves (64 columns, whole 128-byte lines per store) and three or four 16-token groups per wave were slower.
#include <utility>

#include "common.h"
#include "gemm_args.h"
#include "gemm_device.h"
#include "tuning.h"

namespace maxfp8 {

// NS slabs of K, MT groups of 16 tokens.  grid: (128-column blocks, groups of 16 * MT tokens, batches)
template <int NS, int MT>
__global__ __launch_bounds__(256) void gemm_short_k_kernel(GemmArgs p_in) {
  const GemmArgs p = batch_view(p_in, blockIdx.z);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lq = lane >> 4;
  const int n0 = ((int)blockIdx.x * 4 + wave) * 32;
  if (n0 >= p.N) return;
  const int m0 = (int)blockIdx.y * (16 * MT);

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
  v8i w[2][NS], a[MT][NS];
  float as[MT][NS], bs[NS];
  const uint32_t wrow = 8u * (lm >> 2) + (lm & 3);
#pragma unroll
  for (int k = 0; k < NS; ++k)
#pragma unroll
    for (int h = 0; h < 2; ++h) w[h][k] = load_frag(b_rsrc, (wrow + 4u * h) * (uint32_t)p.ldb + (uint32_t)lq * 16u, k);
#pragma unroll
  for (int t = 0; t < MT; ++t) {  // (tokens past M read as zero)
    const uint32_t m = (uint32_t)(m0 + t * 16 + lm);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      a[t][k] = load_frag(a_rsrc, m * (uint32_t)p.lda + (uint32_t)lq * 16u, k);
      as[t][k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, m < (uint32_t)p.M ? m * 4u : 0x80000000u,
                                                                              (uint32_t)k * (uint32_t)p.a_scales_ld * 4u, 0));
    }
  }
  const float* bs_row = p.b_scales + (int64_t)(n0 / 128) * p.b_scales_ld;
#pragma unroll
  for (int k = 0; k < NS; ++k) bs[k] = bs_row[k];

#pragma unroll
  for (int t = 0; t < MT; ++t) {
    v4f acc[2];
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const float s = as[t][k] * bs[k];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[h][k], a[t][k], zero, 0, 0, 0, 0, 0, 0);
        if (k == 0) acc[h] = part * s;
        else acc[h] += part * s;
      }
    }
    const int m = m0 + t * 16 + lm;
    if (m < p.M)
      *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p.c) + (int64_t)m * p.ldc + n0 + lq * 8) =
          make_uint4(pack_bf16x2(acc[0][0], acc[0][1]), pack_bf16x2(acc[0][2], acc[0][3]), pack_bf16x2(acc[1][0], acc[1][1]),
                     pack_bf16x2(acc[1][2], acc[1][3]));
  }
}

int compute_units();

// Batches of at most 32 tokens, whole slabs and whole 32-column groups, bf16 results with 16-byte rows; every other shape
// keeps the other kernels.  With three or four slabs the decode kernel's waves all have a share, and it stays ahead while its
// 16-row blocks are at most two per CU (16 heads of 512 -> 128: 3.1 against 4.0 us at M = 1; 128 heads: 5.9 against 4.9) and,
// with two groups of tokens, which are a wave each here and one pass over the weights there, at most one (17 to 32 tokens: 16 and
// 32 heads of 512 -> 128 4.5 and 4.7 us against 5.4 and 5.3, 48 heads 6.3 against 5.9).
bool gemm_short_k_ok(const GemmArgs& p, bool blockscale, int64_t batch) {
  if (!blockscale || !tuning().short_k || batch < 2 || p.kv_on || p.M > 32 || p.K % 128 != 0 || p.K > 512 || p.N % 32 != 0 ||
      p.c_dtype != MAXFP8_BF16 || !p.c_vec8_ok)
    return false;
  return p.K <= 256 || ceil_div(p.N, 16) * batch > (p.M > 16 ? 1 : 2) * (int64_t)compute_units();
}

template <int NS, int MT>
static int launch_short_k(const GemmArgs& p, int64_t batch, hipStream_t stream) {
  hipLaunchKernelGGL((gemm_short_k_kernel<NS, MT>), dim3((unsigned)ceil_div(p.N, 128), (unsigned)ceil_div(p.M, 16 * MT), (unsigned)batch),
                     dim3(256), 0, stream, p);
  return launch_status("gemm_short_k");
}

// One slab: both 16-token groups in one wave (M = 32: 5.6 us against 6.5 with a wave each); longer K: a wave each (5.7 against 6.5)
int gemm_short_k_dispatch(const GemmArgs& p, int64_t batch, hipStream_t stream) {
  switch (p.K / 128) {
    case 1: return p.M > 16 ? launch_short_k<1, 2>(p, batch, stream) : launch_short_k<1, 1>(p, batch, stream);
    case 2: return launch_short_k<2, 1>(p, batch, stream);
    case 3: return launch_short_k<3, 1>(p, batch, stream);
    default: return launch_short_k<4, 1>(p, batch, stream);
  }
}

}  // namespace maxfp8
