// The MoE steps on either side of the grouped FP8 matmul:
//
//   * moe_create_indices: groups the (token, expert) assignments by expert -- a stable bucket
//     sort of topk_ids (semantics: max/kernels/src/nn/moe.mojo:435-590).  The reference hands
//     out expert slots in the order in which its blocks reach an atomic lock, so its
//     expert_ids is some permutation of 0..E-1; here slot z is expert z and tokens keep their
//     order inside a slot, which is one of the reference's possible results and the same on
//     every run.  One block up to 4096 assignments, beyond that three small launches (count,
//     scan, scatter; no atomics, the counts travel in expert_start_indices); no scratch memory.
//   * fused_silu / fused_silu_quantized: silu(gate) * up on the rows that row_offsets says
//     are in use, written as the input dtype or quantised to e4m3fn with one scale per
//     128 outputs, scales transposed (max/kernels/src/shmem/ep_comm.mojo:4409-4500, 4505-4624).
//     Note the quantiser of this op: scale = max(amax, 1e-4) / 448 and out / scale (a division),
//     not the min(amax, ub) / 448 and x * (1 / scale) of quantize_dynamic_scaled_fp8.
#include <type_traits>

#include "common.h"

namespace maxfp8 {

// ---- moe_create_indices -----------------------------------------------------------------------
// An id that is no expert's: its assignment has no position, and a consumer of restore_token_order skips it as out of range.
constexpr uint32_t kMoeNoPosition = 0xffffffffu;

// block e counts the assignments to expert e; the count waits in expert_start_indices[e + 1].  The block behind
// the last expert's marks the assignments to none.
// V ids per thread and iteration: a multiple of 4 (16-byte loads, topk_ids 16-byte aligned) or 1.  Every block reads all of topk_ids from
// L2, so what counts is loads in flight: one id per load and iteration took 49 us for 32768 ids, four per load with
// four loads in flight take a fifth of that.
template <int V>
__device__ __forceinline__ void moe_load_ids(const int32_t* __restrict__ topk_ids, int i, int n, int (&id)[V]) {
  if constexpr (V % 4 == 0) {
    if (i + V - 1 < n) {
#pragma unroll
      for (int q = 0; q < V / 4; ++q) {
        const int4 v = *reinterpret_cast<const int4*>(topk_ids + i + 4 * q);
        id[4 * q] = v.x; id[4 * q + 1] = v.y; id[4 * q + 2] = v.z; id[4 * q + 3] = v.w;
      }
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < V; ++j) id[j] = i + j < n ? topk_ids[i + j] : -1;  // (-1: no expert)
}
template <int V>
__global__ __launch_bounds__(256) void moe_count_kernel(uint32_t* __restrict__ expert_start_indices,
                                                        uint32_t* __restrict__ restore_token_order,
                                                        const int32_t* __restrict__ topk_ids, int n) {
  __shared__ int red[4];
  const int e = blockIdx.x, tid = threadIdx.x, num_experts = (int)gridDim.x - 1;
  if (e == num_experts) {
#pragma unroll 4
    for (int i = tid * V; i < n; i += 256 * V) {
      int id[V];
      moe_load_ids<V>(topk_ids, i, n, id);
#pragma unroll
      for (int j = 0; j < V; ++j)
        if ((uint32_t)id[j] >= (uint32_t)num_experts && i + j < n) restore_token_order[i + j] = kMoeNoPosition;
    }
    return;
  }
  int cnt = 0;
#pragma unroll 4
  for (int i = tid * V; i < n; i += 256 * V) {
    int id[V];
    moe_load_ids<V>(topk_ids, i, n, id);
#pragma unroll
    for (int j = 0; j < V; ++j) cnt += id[j] == e;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
  if ((tid & 63) == 0) red[tid >> 6] = cnt;
  __syncthreads();
  if (tid == 0) {
    expert_start_indices[e + 1] = (uint32_t)(red[0] + red[1] + red[2] + red[3]);
    if (e == 0) expert_start_indices[0] = 0;
  }
}
__global__ __launch_bounds__(1024) void moe_scan_kernel(uint32_t* __restrict__ expert_start_indices,
                                                        int32_t* __restrict__ expert_ids,
                                                        uint32_t* __restrict__ expert_usage_stats, int num_experts) {
  __shared__ uint32_t wave_sum[16], wave_max_s[16];
  __shared__ uint32_t carry;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) carry = 0;
  uint32_t mx = 0;
  __syncthreads();
  for (int base = 0; base < num_experts; base += 1024) {
    const int z = base + tid;
    const uint32_t c = z < num_experts ? expert_start_indices[z + 1] : 0u;
    mx = c > mx ? c : mx;
    uint32_t incl = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t up = __shfl_up(incl, o, 64);
      if (lane >= o) incl += up;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    uint32_t before = carry;
    for (int w = 0; w < wave; ++w) before += wave_sum[w];
    if (z < num_experts) {
      expert_start_indices[z + 1] = before + incl;
      expert_ids[z] = z;
    }
    __syncthreads();
    if (tid == 1023) carry = before + incl;
    __syncthreads();
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t other = __shfl_xor(mx, o, 64);
    mx = other > mx ? other : mx;
  }
  if (lane == 0) wave_max_s[wave] = mx;
  __syncthreads();
  if (tid == 0) {
    uint32_t m = 0;
    for (int w = 0; w < 16; ++w) m = wave_max_s[w] > m ? wave_max_s[w] : m;
    expert_usage_stats[0] = m;                       // most tokens on one expert
    expert_usage_stats[1] = (uint32_t)num_experts;   // every expert keeps a slot (moe.mojo:584-588)
  }
}

// block e writes the positions of its assignments, in order, from expert_start_indices[e] on: 256 * V ids per
// iteration, thread t the V consecutive ids from 256 * V * iteration + V * t, a prefix sum of the threads' hit counts
// (shuffles inside a wave, LDS across the four waves; the two halves of wave_cnt take turns, so one barrier per iteration).
// An iteration costs 0.7 us whatever it holds -- the scan and the barrier, with one block of four waves per CU -- so V = 16 where
// the pointer allows: 32768 ids in 8 iterations (41 us with one id per thread and iteration, 23 with four, 12 with sixteen)
template <int V>
__global__ __launch_bounds__(256) void moe_scatter_kernel(uint32_t* __restrict__ token_expert_order,
                                                          uint32_t* __restrict__ restore_token_order,
                                                          const uint32_t* __restrict__ expert_start_indices,
                                                          const int32_t* __restrict__ topk_ids, int n) {
  __shared__ int wave_cnt[2][4];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t base = expert_start_indices[e];
  if (expert_start_indices[e + 1] == base) return;
  int turn = 0;
  for (int i0 = 0; i0 < n; i0 += 256 * V, turn ^= 1) {
    const int i = i0 + tid * V;
    int id[V];
    moe_load_ids<V>(topk_ids, i, n, id);
    int c = 0;
#pragma unroll
    for (int j = 0; j < V; ++j) c += id[j] == e;
    int incl = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(incl, o, 64);
      if (lane >= o) incl += up;
    }
    if (lane == 63) wave_cnt[turn][wave] = incl;
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wave) before += wave_cnt[turn][w];
      total += wave_cnt[turn][w];
    }
    uint32_t pos = base + (uint32_t)(before + incl - c);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      if (id[j] == e) {
        token_expert_order[pos] = (uint32_t)(i + j);
        restore_token_order[i + j] = pos;
        ++pos;
      }
    }
    base += (uint32_t)total;
  }
}

// Up to 4096 assignments and 512 experts: the three steps in one block, one launch.  The three small launches are latency, and
// the whole list fits one block's registers: wave w holds the 64 * STEPS ids from
// 64 * STEPS * w on.  Lanes with the same id find each other by ballots over the id's nine bits, the lowest of them counts the
// group into the wave's own histogram in LDS, and its count before is the group's rank inside the wave; a thread per expert
// then turns the sixteen waves' counts into start offsets.  The order stays that of the list: steps of a wave one after the
// other, waves by their place, lanes by their number.  Graph timing, three launches -> one block: 512 ids of 256 experts 7.6 ->
// 3.2 us, 2048 of 128 7.8 -> 4.6, 4096 of 256 8.0 -> 7.1.  Bound: the latency of a step's LDS atomic and of its scattered stores
// on one CU, a microsecond per step; 8192 ids were 11.6 us against the three launches' 9.1, so the line is at 4096.
constexpr int kMoeOneBlockExperts = 512, kMoeOneBlockSteps = 4;
template <int STEPS>
__global__ __launch_bounds__(1024) void moe_indices_one_block_kernel(uint32_t* __restrict__ token_expert_order,
                                                                     uint32_t* __restrict__ expert_start_indices,
                                                                     uint32_t* __restrict__ restore_token_order,
                                                                     int32_t* __restrict__ expert_ids,
                                                                     uint32_t* __restrict__ expert_usage_stats,
                                                                     const int32_t* __restrict__ topk_ids, int n, int num_experts) {
  __shared__ uint32_t counts[16][kMoeOneBlockExperts];
  __shared__ uint32_t wave_sum[16], wave_max[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int first = wave * 64 * STEPS + lane;
  int id[STEPS];
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const int i = first + 64 * s;
    id[s] = i < n ? topk_ids[i] : -1;
  }
  for (int i = tid; i < 16 * kMoeOneBlockExperts; i += 1024) (&counts[0][0])[i] = 0;
  __syncthreads();
  uint32_t rank[STEPS];  // among the wave's assignments to the same expert
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const bool valid = (uint32_t)id[s] < (uint32_t)num_experts;  // (others belong to no expert)
    uint64_t same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 9; ++b) {
      const bool set = (id[s] >> b) & 1;
      const uint64_t with = __ballot(set);
      same &= set ? with : ~with;
    }
    const int leader = valid ? __ffsll((unsigned long long)same) - 1 : lane;
    uint32_t before = 0;
    if (valid && lane == leader) before = atomicAdd(&counts[wave][id[s]], (uint32_t)__popcll(same));
    before = __shfl(before, leader, 64);
    rank[s] = before + (uint32_t)__popcll(same & (((uint64_t)1 << lane) - 1));
    if (!valid) id[s] = -1;
  }
  __syncthreads();
  uint32_t mine = 0;  // thread e: assignments to expert e; counts[w][e] becomes those of the waves before w
  if (tid < num_experts) {
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const uint32_t c = counts[w][tid];
      counts[w][tid] = mine;
      mine += c;
    }
  }
  uint32_t incl = mine, most = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t up = __shfl_up(incl, o, 64);
    if (lane >= o) incl += up;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t other = __shfl_xor(most, o, 64);
    most = other > most ? other : most;
  }
  if (lane == 63) {
    wave_sum[wave] = incl;
    wave_max[wave] = most;
  }
  __syncthreads();
  for (int w = 0; w < wave; ++w) incl += wave_sum[w];
  if (tid < num_experts) {
#pragma unroll
    for (int w = 0; w < 16; ++w) counts[w][tid] += incl - mine;
    expert_start_indices[tid + 1] = incl;
    expert_ids[tid] = tid;
  }
  if (tid == 0) {
    expert_start_indices[0] = 0;
    uint32_t m = 0;
    for (int w = 0; w < 16; ++w) m = wave_max[w] > m ? wave_max[w] : m;
    expert_usage_stats[0] = m;
    expert_usage_stats[1] = (uint32_t)num_experts;
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    if (id[s] >= 0) {
      const uint32_t pos = counts[wave][id[s]] + rank[s];
      token_expert_order[pos] = (uint32_t)(first + 64 * s);
      restore_token_order[first + 64 * s] = pos;
    } else if (first + 64 * s < n) {
      restore_token_order[first + 64 * s] = kMoeNoPosition;
    }
  }
}

int moe_create_indices_dispatch(uint32_t* token_expert_order, uint32_t* expert_start_indices, uint32_t* restore_token_order,
                                int32_t* expert_ids, uint32_t* expert_usage_stats, const int32_t* topk_ids, int64_t n,
                                int64_t num_experts, hipStream_t stream) {
  if (n <= 1024 * kMoeOneBlockSteps && num_experts <= kMoeOneBlockExperts) {
    auto* const kernel = n <= 1024 ? moe_indices_one_block_kernel<1> : n <= 2048 ? moe_indices_one_block_kernel<2> :
                         moe_indices_one_block_kernel<kMoeOneBlockSteps>;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(1024), 0, stream, token_expert_order, expert_start_indices, restore_token_order, expert_ids,
                       expert_usage_stats, topk_ids, (int)n, (int)num_experts);
    return launch_status("moe_create_indices");
  }
  const bool vec = (reinterpret_cast<uintptr_t>(topk_ids) & 15) == 0;
  if (vec) hipLaunchKernelGGL(moe_count_kernel<4>, dim3((unsigned)num_experts + 1), dim3(256), 0, stream, expert_start_indices, restore_token_order,
                              topk_ids, (int)n);
  else hipLaunchKernelGGL(moe_count_kernel<1>, dim3((unsigned)num_experts + 1), dim3(256), 0, stream, expert_start_indices, restore_token_order,
                          topk_ids, (int)n);
  hipLaunchKernelGGL(moe_scan_kernel, dim3(1), dim3(1024), 0, stream, expert_start_indices, expert_ids, expert_usage_stats,
                     (int)num_experts);
  if (n > 0) {
    if (vec)
      hipLaunchKernelGGL(moe_scatter_kernel<16>, dim3((unsigned)num_experts), dim3(256), 0, stream, token_expert_order,
                         restore_token_order, expert_start_indices, topk_ids, (int)n);
    else
      hipLaunchKernelGGL(moe_scatter_kernel<1>, dim3((unsigned)num_experts), dim3(256), 0, stream, token_expert_order,
                         restore_token_order, expert_start_indices, topk_ids, (int)n);
  }
  return launch_status("moe_create_indices");
}

// ---- fused SiLU(gate) * up --------------------------------------------------------------------
// a / b, correctly rounded (the IEEE quotient), at a third of the IEEE sequence's cost on the common path.  One Newton
// step turns the hardware's reciprocal (within an ulp) into the correctly rounded one -- unless b's mantissa is all ones --
// and with that, a quotient estimate, its exact residual and one correction give the correctly rounded quotient
// (Markstein's sequence) as long as no product underflows or overflows.  Everything outside those conditions takes the
// IEEE division, in a branch the wave skips unless one of its lanes needs it.  (Checked on the CPU against the IEEE
// quotient: the same operations and acceptance tests on 1.8e9 operand pairs -- random, bf16 numerators, divisors whose
// mantissa is (nearly) all ones, zeros and tiny numerators, quotients of the quantiser's size -- with the reciprocal
// off by -1, 0 and +1 ulp: no difference.)
__device__ __forceinline__ float refined_rcp(float b) {
  const float y0 = __builtin_amdgcn_rcpf(b);
  return fmaf(fmaf(-b, y0, 1.0f), y0, y0);
}
// a / b given y = refined_rcp(b); to be trusted where div_b_ok(b) and div_q_ok(a, result)
__device__ __forceinline__ float div_by(float a, float b, float y) {
  const float q0 = a * y;
  const float q = fmaf(fmaf(-b, q0, a), y, q0);
  return a == 0.0f ? q0 : q;  // (keeps the sign of a zero quotient)
}
__device__ __forceinline__ bool div_b_ok(float b) {
  return (b >= 0x1p-63f) & (b < 0x1p64f) & ((__float_as_uint(b) & 0x007fffffu) != 0x007fffffu);
}
__device__ __forceinline__ bool div_q_ok(float a, float q) {
  return (a == 0.0f) | ((fabsf(a) >= 0x1p-63f) & (fabsf(q) >= 0x1p-63f) & (fabsf(q) < 0x1p64f));
}
// Eight quotients a[j] / b by one divisor, with one test for the lane and one branch for the wave
__device__ __forceinline__ void exact_div8(const float (&a)[8], float b, float (&q)[8]) {
  const float y = refined_rcp(b);
  bool ok = div_b_ok(b);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    q[j] = div_by(a[j], b, y);
    ok = ok & div_q_ok(a[j], q[j]);
  }
  if (__builtin_amdgcn_ballot_w64(!ok) != 0ull) {
    if (!ok) {
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = a[j] / b;
    }
  }
}

__device__ __forceinline__ void unpack_bf16x8(const uint4& v, float (&f)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f[2 * j] = __uint_as_float(w[j] << 16);
    f[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
  }
}

__device__ __forceinline__ uint4 pack_bf16x8(const float (&f)[8]) {
  return make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
}

// gate / (1 + exp(-gate)), every step rounded to f32 (ep_comm.mojo:4494-4497), of eight gates that are bf16 values.
//   BF16 = false: the bits of expf and the IEEE division in 13 instructions instead of 30.  log2(e) comes in two parts, the first of
//     16 bits, whose product t with the gate's 8 is exact: the argument of the power of two has one rounding and no range checks.  The
//     quotient is corrected once by its exact residual (v_div_fixup: signed zeros, NaN).
//   BF16 = true, for a caller that rounds the result to bf16: 7 instructions, some ulp of f32 away, which bf16 does not show.
// Gates of 86 and beyond, where the exponential leaves the range, and infinities take expf and the division, in a branch the wave
// skips unless one of its lanes needs it.  (There are 65536 gates: all of them have been compared with that path, BF16 after
// the rounding: the same bits.)
template <bool BF16>
__device__ __forceinline__ void silu8(const uint4& bits, const float (&gate)[8], float (&sig)[8]) {
  constexpr float kHi = 0x1.7154p+0f, kLo = (float)(1.4426950408889634074 - 0x1.7154p+0);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if constexpr (BF16) {
      sig[j] = gate[j] * refined_rcp(1.0f + __builtin_amdgcn_exp2f(gate[j] * -1.4426950408889634074f));
    } else {
      const float t = gate[j] * -kHi, n = rintf(t);
      const float d = 1.0f + ldexpf(__builtin_amdgcn_exp2f(fmaf(gate[j], -kLo, t - n)), (int)n);
      const float y = __builtin_amdgcn_rcpf(d), q0 = gate[j] * y;
      sig[j] = __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q0, gate[j]), y, q0), d, gate[j]);
    }
  }
  // (compared as integers, two a word: a NaN is larger than every number, where a float maximum may lose the largest to it)
  typedef unsigned short u2 __attribute__((ext_vector_type(2)));
  auto size = [](uint32_t w) { return __builtin_bit_cast(u2, w & 0x7fff7fffu); };
  const u2 most = __builtin_elementwise_max(__builtin_elementwise_max(size(bits.x), size(bits.y)), __builtin_elementwise_max(size(bits.z), size(bits.w)));
  const bool beyond = (most.x >= 0x42acu) | (most.y >= 0x42acu);
  if (__builtin_amdgcn_ballot_w64(beyond) != 0ull) {
    if (beyond) {
#pragma unroll
      for (int j = 0; j < 8; ++j) sig[j] = gate[j] / (1.0f + expf(-gate[j]));
    }
  }
}

// silu(gate) * up for eight outputs.
// ROUND_ACT: the activation is rounded to bf16 before the product, as where silu and the multiplication are two bf16
// operations (the dense gated MLP, max/python/max/nn/linear.py:1072: ops.silu(gate) * up).
template <bool ROUND_ACT>
__device__ __forceinline__ void silu_mul8(const uint4& gate_bits, const uint4& up_bits, float (&f)[8]) {
  float gate[8], up[8], sig[8];
  unpack_bf16x8(gate_bits, gate);
  unpack_bf16x8(up_bits, up);
  silu8<ROUND_ACT>(gate_bits, gate, sig);
  if constexpr (ROUND_ACT) unpack_bf16x8(pack_bf16x8(sig), sig);
#pragma unroll
  for (int j = 0; j < 8; ++j) f[j] = sig[j] * up[j];
}

// What the silu kernel does with its eight products.
enum SiluOut {
  kSiluBf16,       // stores them as bf16
  kSiluQuant,      // quantises the f32 products with the op's own recipe: max(amax, 1e-4) / 448, value / scale
  kSiluBf16Quant,  // rounds them to bf16 and quantises that like quantize_dynamic_scaled_fp8 with groups of 128: the bytes
                   // and scales of kSiluBf16 followed by the quantiser, without the bf16 tensor between them
};

__device__ __forceinline__ uint2 pack_e4m3fn8(const float (&q)[8]) {
  int lo = 0, hi = 0;
  lo = cvt_pk_e4m3fn(q[0], q[1], lo, false);
  lo = cvt_pk_e4m3fn(q[2], q[3], lo, true);
  hi = cvt_pk_e4m3fn(q[4], q[5], hi, false);
  hi = cvt_pk_e4m3fn(q[6], q[7], hi, true);
  return make_uint2((uint32_t)lo, (uint32_t)hi);
}

// A block takes tiles of ROWS rows x U groups of 128 outputs: 16 lanes own a row's group (8 outputs each, one 16-byte load of gate
// and of up per lane), a thread the tile's U groups of its row, whose loads go out together; quantised: amax over the 16 lanes by
// DPP, 8-byte packed fp8 store.  A group's scales leave as ROWS consecutive floats: with 32 rows a whole line, which no other XCD's L2
// holds a part of (32768 x 2048: 16 groups of a row per block, every scale alone, 73 us; 4 rows 113; 16 rows 68; 32 rows 62).
// Bound by the bytes (5 per output where the result is quantised) and, as close, by the arithmetic: 30 instructions per output, two of
// them four times as long.  Graph timing, operands from memory, before this form and now: 2048 x 14336 rounding twice and quantising 38.6 -> 29.9 us
// (147 MB: 4.9 TB/s), 32768 x 2048 rounding once 82 -> 65, 512 x 14336 rounding twice 13.7 -> 10.8, 16 x 14336 4.6 -> 3.6 (from the cache 3.8 -> 2.8).
template <SiluOut OUT, bool ROUND_ACT, int ROWS, int U>
__global__ __launch_bounds__(16 * ROWS) void fused_silu_bf16_kernel(void* __restrict__ out, float* __restrict__ scales,
                                                              const uint16_t* __restrict__ in,
                                                              const uint32_t* __restrict__ row_offsets, int num_offsets,
                                                              int64_t max_rows, int inter, int64_t in_stride,
                                                              int64_t out_stride, int64_t scales_ld, float scale_ub) {
  // (the buffers hold max_rows rows: an offset beyond that -- a stale or damaged routing tensor -- must not
  // turn into accesses outside them)
  const uint32_t rows_dev = row_offsets[num_offsets - 1];
  const int64_t rows = (int64_t)rows_dev < max_rows ? (int64_t)rows_dev : max_rows;
  const uint32_t groups = (uint32_t)inter >> 7, nxb = (groups + U - 1) / U;
  const uint32_t tiles = (uint32_t)((rows + ROWS - 1) / ROWS) * nxb;  // (an output is 4 bytes of input and more: far below 2^32)
  const int tid = threadIdx.x, sub = tid & 15;
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t rb = tile / nxb, g0 = (tile - rb * nxb) * U;
    const int64_t row = (int64_t)rb * ROWS + (tid >> 4);
    const bool row_ok = row < rows;
    const uint16_t* src = in + row * in_stride + g0 * 128u + sub * 8;
    uint4 gate[U], up[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      gate[u] = up[u] = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);  // (no value: ones, as in the quantiser)
      if (row_ok && g0 + u < groups) {
        gate[u] = *reinterpret_cast<const uint4*>(src + u * 128);
        up[u] = *reinterpret_cast<const uint4*>(src + u * 128 + inter);
      }
    }
    const int64_t at = row * out_stride + g0 * 128u + sub * 8;
    float my_scale = 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool live = row_ok && g0 + u < groups;
      float f[8];
      silu_mul8<ROUND_ACT>(gate[u], up[u], f);
      if constexpr (OUT == kSiluBf16) {
        if (live) *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(out) + at + u * 128) = pack_bf16x8(f);
      } else {
        if constexpr (OUT == kSiluBf16Quant) unpack_bf16x8(pack_bf16x8(f), f);
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(f[j]));
        amax = row16_max(amax);
        float scale, q[8];
        if constexpr (OUT == kSiluQuant) {
          scale = fmaxf(amax, 1e-4f) / 448.0f;
          exact_div8(f, scale, q);
        } else {
          float recip;
          dynamic_scale_f32(amax, scale_ub, scale, recip);
#pragma unroll
          for (int j = 0; j < 8; ++j) q[j] = f[j] * recip;
        }
        if (sub == u) my_scale = scale;
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = clamp448(q[j]);
        if (live) *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(out) + at + u * 128) = pack_e4m3fn8(q);
      }
    }
    if (OUT != kSiluBf16 && row_ok && sub < U && g0 + sub < groups) scales[(int64_t)(g0 + sub) * scales_ld + row] = my_scale;
  }
}

// The same with one scale per row (per-token quantisation of the bf16 product): one block per row, NV 16-byte vectors of
// bf16 products per thread stay in registers between the amax and the convert pass; inter <= THREADS * 8 * NV.
// 2048 x 14336: 45.6 us as two kernels, 28 as one; 32768 x 2048 (256 threads: every one has its vector) 105 and 58.  (As one with expf and
// the IEEE division 38 and 79.)
template <int THREADS, int NV, bool ROUND_ACT>
__global__ __launch_bounds__(THREADS) void fused_silu_row_quant_kernel(uint8_t* __restrict__ out, float* __restrict__ scales,
                                                                               const uint16_t* __restrict__ in,
                                                                               const uint32_t* __restrict__ row_offsets, int num_offsets,
                                                                               int64_t max_rows, int inter, int64_t in_stride,
                                                                               int64_t out_stride, float scale_ub) {
  __shared__ float red[THREADS / 64];
  const uint32_t rows_dev = row_offsets[num_offsets - 1];
  const int64_t rows = (int64_t)rows_dev < max_rows ? (int64_t)rows_dev : max_rows;
  const int64_t m = blockIdx.x;
  if (m >= rows) return;
  const int tid = threadIdx.x, nvec = inter >> 3;
  const uint4* gate_row = reinterpret_cast<const uint4*>(in + m * in_stride);
  const uint4* up_row = reinterpret_cast<const uint4*>(in + m * in_stride + inter);
  uint4 h[NV];
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = tid + i * THREADS;
    h[i] = make_uint4(0, 0, 0, 0);
    if (idx < nvec) {
      float f[8];
      silu_mul8<ROUND_ACT>(gate_row[idx], up_row[idx], f);
      h[i] = pack_bf16x8(f);
      unpack_bf16x8(h[i], f);
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(f[j]));
    }
  }
  amax = wave_max(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < THREADS / 64; ++w) amax = fmaxf(amax, red[w]);
  float scale, recip;
  dynamic_scale_f32(amax, scale_ub, scale, recip);
  if (tid == 0) scales[m] = scale;
  uint2* dst = reinterpret_cast<uint2*>(out + m * out_stride);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = tid + i * THREADS;
    if (idx < nvec) {
      float f[8];
      unpack_bf16x8(h[i], f);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = clamp448(f[j] * recip);
      dst[idx] = pack_e4m3fn8(f);
    }
  }
}

template <bool ROUND_ACT>
static bool launch_silu_row(void* out, float* scales, const void* in, const uint32_t* row_offsets, int64_t num_offsets, int64_t max_rows,
                            int64_t inter, int64_t in_stride, int64_t out_stride, float scale_ub, hipStream_t stream) {
  auto launch = [&](auto kern, int threads) {
    hipLaunchKernelGGL(kern, dim3((unsigned)max_rows), dim3(threads), 0, stream, (uint8_t*)out, scales, (const uint16_t*)in,
                       row_offsets, (int)num_offsets, max_rows, (int)inter, in_stride, out_stride, scale_ub);
    return true;
  };
  if (inter <= 2048) return launch(fused_silu_row_quant_kernel<256, 1, ROUND_ACT>, 256);
  if (inter <= 4096) return launch(fused_silu_row_quant_kernel<512, 1, ROUND_ACT>, 512);
  if (inter <= 8192) return launch(fused_silu_row_quant_kernel<512, 2, ROUND_ACT>, 512);
  if (inter <= 16384) return launch(fused_silu_row_quant_kernel<1024, 2, ROUND_ACT>, 1024);
  if (inter <= 32768) return launch(fused_silu_row_quant_kernel<1024, 4, ROUND_ACT>, 1024);
  return false;
}

// mode: the ABI's `quantize`
int fused_silu_dispatch(void* out, float* scales, const void* in, const uint32_t* row_offsets, int64_t num_offsets,
                        int64_t max_rows, int64_t inter, int64_t in_stride, int64_t out_stride, int64_t scales_ld,
                        int mode, bool row_scales, float scale_ub, hipStream_t stream) {
  if (row_scales) {
    const bool ok = mode == 4
                        ? launch_silu_row<true>(out, scales, in, row_offsets, num_offsets, max_rows, inter, in_stride, out_stride, scale_ub, stream)
                        : launch_silu_row<false>(out, scales, in, row_offsets, num_offsets, max_rows, inter, in_stride, out_stride, scale_ub, stream);
    if (!ok) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused_silu: one scale per row takes rows of at most 32768 outputs");
    return launch_status("fused_silu_quantized (row)");
  }
  // The number of rows in use is only known on the device: the grid is sized for max_rows and walks the tiles in strides.  Tiles of
  // 32 rows x 2 groups, or of 16 x 1 where those would leave half of the CUs without one (rounding twice, from memory, us: 16 x 14336 3.7 and 3.6, 333 x 1408 4.4 and
  // 3.7, 128 x 14336 5.2 and 6.1, 512 x 14336 10.8 and 14.5; from the cache 3.3 and 2.8, 4.0 and 3.4, 5.2 and 6.1).
  const int64_t large = ceil_div(max_rows, 32) * ceil_div(inter / 128, 2);
  auto launch = [&](auto kern, int rows, int64_t tiles) {
    hipLaunchKernelGGL(kern, dim3((unsigned)(tiles < 16384 ? tiles : 16384)), dim3(16 * rows), 0, stream, out, scales, (const uint16_t*)in, row_offsets,
                       (int)num_offsets, max_rows, (int)inter, in_stride, out_stride, scales_ld, scale_ub);
  };
  auto either = [&](auto out_c, auto round_c) {
    constexpr SiluOut OUT = decltype(out_c)::value;
    constexpr bool ROUND_ACT = decltype(round_c)::value;
    if (large >= 128) launch(fused_silu_bf16_kernel<OUT, ROUND_ACT, 32, 2>, 32, large);
    else launch(fused_silu_bf16_kernel<OUT, ROUND_ACT, 16, 1>, 16, ceil_div(max_rows, 16) * (inter / 128));
  };
  constexpr std::integral_constant<SiluOut, kSiluBf16> plain{};
  constexpr std::integral_constant<SiluOut, kSiluQuant> quant{};
  constexpr std::integral_constant<SiluOut, kSiluBf16Quant> bf16_quant{};
  switch (mode) {
    case 1: either(quant, std::false_type{}); break;
    case 2: either(plain, std::true_type{}); break;
    case 3: either(bf16_quant, std::false_type{}); break;
    case 4: either(bf16_quant, std::true_type{}); break;
    default: either(plain, std::false_type{}); break;
  }
  return launch_status(mode == 0 || mode == 2 ? "fused_silu" : "fused_silu_quantized");
}

}  // namespace maxfp8
