// C ABI of the library (include/maxfp8.h): argument checks, kernel selection, error text.
#include <stdarg.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <mutex>

#include "common.h"
#include "gemm_args.h"
#include "tuning.h"

namespace maxfp8 {

static thread_local char g_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

int launch_status(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) MAXFP8_FAIL(MAXFP8_ERR_LAUNCH, "%s: launch failed: %s", what, hipGetErrorString(e));
  return MAXFP8_OK;
}

// kernels (defined in the other translation units)
int quantize_dispatch(void*, void*, const void*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, int,
                      float, int64_t, int64_t, int64_t, int64_t, const uint32_t*, uint32_t, hipStream_t);
int quantize_scatter_dispatch(void*, void*, const void*, int64_t, int64_t, int64_t, int64_t, int64_t, float, const uint32_t*, int64_t,
                              int64_t, hipStream_t);
int rmsnorm_quantize_dispatch(void*, void*, const void*, const void*, int64_t, int64_t, int64_t, int64_t, int, int, float,
                              float, float, hipStream_t);
int quantize_static_dispatch(void*, const void*, int64_t, int64_t, int64_t, int64_t, int, float, hipStream_t);
int quantize_static_for_matmul_dispatch(void*, float*, const void*, int64_t, int64_t, int64_t, int, float, float, hipStream_t);
int quantize_tensor_dispatch(void*, void*, const void*, int64_t, int64_t, int64_t, int64_t, int, int, float, hipStream_t);
int moe_create_indices_dispatch(uint32_t*, uint32_t*, uint32_t*, int32_t*, uint32_t*, const int32_t*, int64_t, int64_t, hipStream_t);
int fused_silu_dispatch(void*, float*, const void*, const uint32_t*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, bool,
                        float, hipStream_t);
int cast_f32_to_e4m3fn_dispatch(void*, const float*, int64_t, hipStream_t);
int cast_e4m3fn_to_f32_dispatch(float*, const void*, int64_t, hipStream_t);
int cast_f32_to_bf16_dispatch(void*, const float*, int64_t, hipStream_t);
int copy_bytes_dispatch(void*, const void*, int64_t, hipStream_t);
int naive_blockwise_dispatch(void*, const void*, const void*, const void*, const void*, int64_t, int64_t, int64_t,
                             int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, int64_t, int64_t,
                             int64_t, int64_t, int64_t, int64_t, hipStream_t);
int naive_rowwise_dispatch(void*, const void*, const void*, const void*, const void*, int64_t, int64_t, int64_t,
                           int64_t, int64_t, int64_t, int64_t, int64_t, int, int, hipStream_t);
int naive_grouped_dispatch(void*, const void*, const void*, const void*, const void*, const uint32_t*,
                           const int32_t*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, hipStream_t);
int gemm_tiled_dispatch(const GemmArgs&, bool, size_t, int64_t, hipStream_t);
size_t gemm_tiled_workspace_bytes(int64_t, int64_t, int64_t);
size_t gemm_tiled_plan_workspace_bytes(int64_t, int64_t, int64_t, bool);
bool gemm_tiled_needs_no_workspace(int64_t, int64_t, int64_t, bool);
int gemm_tiled_describe(int64_t, int64_t, int64_t, bool, bool, char*, size_t);
int gemm_tiled_tall(int64_t, int64_t, int64_t, bool, bool);
int gemm_grouped_dispatch(const GemmArgs&, bool, int64_t, int64_t, hipStream_t);
int gemm_skinny_dispatch(const GemmArgs&, bool, int64_t, hipStream_t);
bool gemm_skinny_quant_ok(int64_t M, int64_t N, int64_t K, bool blockscale);
int gemm_skinny_quant_dispatch(const GemmArgs&, bool, hipStream_t);
int gemm_skinny_max_m();
int compute_units();
bool gemm_short_k_ok(const GemmArgs&, bool, int64_t);
int gemm_short_k_dispatch(const GemmArgs&, int64_t, hipStream_t);
bool gemm_one_slab_ok(const GemmArgs&, bool, int64_t);
int gemm_one_slab_dispatch(const GemmArgs&, int64_t, hipStream_t);
int gemm_mid_dispatch(const GemmArgs&, bool, int, hipStream_t);
bool gemm_mid_ok(int64_t M, int64_t N, int64_t K);
int gemm_mid_shape(int64_t M, int64_t N, int64_t K, bool blockscale, float* us);
int gemm_mid_forced_shape();
float gemm_skinny_cost(int64_t M, int64_t N, int64_t K, bool* alone);
float gemm_tiled_cost(int64_t M, int64_t N, int64_t K, bool blockscale);
float gemm_tiled_qkv_cost(int64_t M, int64_t N, int64_t K, bool blockscale, bool has_workspace);
size_t gemm_tiled_qkv_workspace_bytes(int64_t M, int64_t N, int64_t K, bool blockscale);
bool gemm_skinny_preferred(int64_t M, int64_t N, int64_t K);
int gemm_skinny_read_probe(const void* b, int64_t M, int64_t N, int64_t K, int64_t ldb, hipStream_t stream);
int gemm_persist_probe(const GemmArgs&, bool, int, hipStream_t);
int gemm_w4_probe(const GemmArgs&, bool, int, int, hipStream_t);
bool gemm_w4_ok(const GemmArgs&, bool);
int gemm_w4_gave_up(unsigned int*);
int gemm_streamk_gave_up(unsigned int*);

// v rounded to bf16 / f16 and widened back: how an op parameter of the input's dtype arrives
static float round_to_dtype(float v, int dtype) {
  if (dtype == MAXFP8_BF16) {
    uint32_t u;
    memcpy(&u, &v, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return v;
    u += 0x7fffu + ((u >> 16) & 1u);
    u &= 0xffff0000u;
    memcpy(&v, &u, 4);
    return v;
  }
  if (dtype == MAXFP8_F16) return (float)(_Float16)v;
  return v;
}

static bool is_aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// ---- the library's own scratch memory (maxfp8_matmul_dynamic_scaled_fp8_noalloc) ------------------
// A file-scope device array: every GPU the library runs on holds its own copy, at its own address, from the
// moment the code object is loaded there until the process ends.  In host code the array's NAME is only a handle
// for hipGetSymbolAddress -- it is not a device address and is never passed to a kernel or a memory call.  The
// address is looked up once per device, with that device current, and kept; kernels receive it as an argument,
// exactly like a caller's workspace.
constexpr size_t kScratchBytes = (size_t)48 << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
static void* g_scratch_ptr[64] = {};
static std::mutex g_scratch_mu;

static int scratch_of_current_device(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= 64)
    MAXFP8_FAIL(MAXFP8_ERR_LAUNCH, "matmul (no-alloc): no current device in 0..63: %s", hipGetErrorString(e));
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      (void)hipGetLastError();
      MAXFP8_FAIL(MAXFP8_ERR_LAUNCH, "matmul (no-alloc): cannot resolve the scratch array on device %d: %s", dev, hipGetErrorString(e));
    }
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return MAXFP8_OK;
}

// The MFMA kernels address a tile's operands with 32-bit buffer offsets whose top bit marks lanes that are out of
// range: the rows of the tallest tile (256) times the row stride, and the activation scales of all slabs of a tile
// (ceil(K / 128) rows of a_scales_ld floats), must stay below 2^31 bytes.
static bool offsets_fit(int64_t K, int64_t lda, int64_t ldb, int64_t a_scales_ld, bool block) {
  const int64_t lim = (int64_t)1 << 31;
  if (256 * lda + K >= lim || 256 * ldb + K >= lim) return false;
  return !block || (ceil_div(K, 128) * a_scales_ld + 256) * 4 < lim;
}

// ---- tuning switches: one immutable snapshot of the environment, replaced as a whole by a reload ----
static std::atomic<const Tuning*> g_tuning{nullptr};
static std::mutex g_tuning_mu;

static const Tuning* read_tuning(unsigned generation) {
  Tuning* t = new Tuning();
  auto num = [](const char* name, int dflt) { const char* e = getenv(name); return e ? atoi(e) : dflt; };
  const int tile = num("MAXFP8_TILE", 0);
  t->tile = (tile >= 1 && tile <= 4) ? tile : 0;
  t->splitk = num("MAXFP8_SPLITK", 0);
  t->one_region = getenv("MAXFP8_ONE_REGION") != nullptr;
  t->persist = num("MAXFP8_PERSIST", 1) != 0;
  t->streamk = num("MAXFP8_STREAMK", 1);
  t->big_rows = num("MAXFP8_BIG_ROWS", 1024);
  t->grouped_overlap = num("MAXFP8_GROUPED_OVERLAP", 1) != 0;
  t->grouped_persist = num("MAXFP8_GROUPED_PERSIST", 1) != 0;
  t->grouped_decode = num("MAXFP8_GROUPED_DECODE", t->grouped_decode);
  const int w4 = num("MAXFP8_W4", -1);
  t->w4 = (w4 == 0 || w4 == 4 || w4 == 5 || w4 == 6 || w4 == 8) ? w4 : -1;
  const int w4_split = num("MAXFP8_W4_SPLIT", -1);
  t->w4_split = (w4_split == 0 || w4_split == 1) ? w4_split : -1;
  t->skinny_quant = num("MAXFP8_SKINNY_QUANT", 1) != 0;
  t->skinny_alds = num("MAXFP8_SKINNY_ALDS", 1) != 0;
  const char* sb = getenv("MAXFP8_GROUPED_SHARE");
  t->grouped_share = sb ? (float)atof(sb) : 0.5f;
  t->grouped_w4 = num("MAXFP8_GROUPED_W4", 1) != 0;
  t->grouped_w4_rows = num("MAXFP8_GROUPED_W4_ROWS", 4096);
  const char* sw = getenv("MAXFP8_GROUPED_W4_SHARE");
  t->grouped_w4_share = sw ? (float)atof(sw) : 0.6f;
  t->grouped_w4_hot_rest = num("MAXFP8_GROUPED_W4_HOT_REST", 32);
  t->grouped_w4_cold_rows = num("MAXFP8_GROUPED_W4_COLD_ROWS", 128);
  t->skinny = num("MAXFP8_SKINNY", 0);
  t->mid = num("MAXFP8_MID", -1);
  t->short_k = num("MAXFP8_SHORT_K", 1) != 0;
  t->generation = generation;
  return t;
}

const Tuning& tuning() {
  const Tuning* t = g_tuning.load(std::memory_order_acquire);
  if (t) return *t;
  std::lock_guard<std::mutex> lock(g_tuning_mu);
  t = g_tuning.load(std::memory_order_acquire);
  if (!t) {
    t = read_tuning(0);
    g_tuning.store(t, std::memory_order_release);
  }
  return *t;
}

// (the old snapshot is left in place for threads that still read it: a few dozen bytes per reload)
void tuning_reload() {
  std::lock_guard<std::mutex> lock(g_tuning_mu);
  const Tuning* old = g_tuning.load(std::memory_order_acquire);
  g_tuning.store(read_tuning(old ? old->generation + 1 : 1), std::memory_order_release);
}

}  // namespace maxfp8

using namespace maxfp8;

extern "C" {

const char* maxfp8_last_error(void) { return g_error; }
const char* maxfp8_version(void) { return "maxfp8 0.2 (gfx950)"; }
void maxfp8_tuning_reload(void) { tuning_reload(); }

}  // extern "C"

namespace maxfp8 {
// The kernel for tens to a few hundred tokens (gemm_mid.hip), beside the ABI's algo values.
constexpr int kAlgoMid = 100;
// A kernel, and which of its shapes where it is that one.
struct Choice { int algo, shape; };
static Choice mid_choice(int64_t M, int64_t N, int64_t K, bool block) {
  float us;
  return {kAlgoMid, tuning().mid > 0 ? gemm_mid_forced_shape() : gemm_mid_shape(M, N, K, block, &us)};
}

// What is chosen: for a matmul whose caller brings all the workspace it is asked for, or none for the sums of a K split; for a fused QKV
// matmul with and without that workspace.
enum class Asked : int { kMatmul, kMatmulNoSplit, kQkv, kQkvWorkspace };
static Choice choose_uncached(Asked what, int64_t M, int64_t N, int64_t K, bool block);

// The choice is asked for several times on every call and walks all shapes of the small tiles (1 to 3 us of host time, as much as a
// launch): the answers are kept, keyed by all that they depend on, the generation of the tuning switches included.
static Choice choose(Asked what, int64_t M, int64_t N, int64_t K, bool block) {
  struct Entry { int64_t M, N, K; unsigned generation; Asked what; bool block; Choice choice; };
  static Entry table[256];  // (algo 0: empty)
  static std::mutex mu;
  const unsigned generation = tuning().generation;
  const uint64_t h = ((uint64_t)M * 0x9e3779b97f4a7c15ull) ^ ((uint64_t)N * 0xc2b2ae3d27d4eb4full) ^ ((uint64_t)K * 0x165667b19e3779f9ull) ^
                     ((uint64_t)(2 * (int)what + (block ? 1 : 0)) * 0xd6e8feb86659fd93ull);
  Entry& e = table[(h >> 32) % 256];
  {
    std::lock_guard<std::mutex> lock(mu);
    if (e.choice.algo && e.M == M && e.N == N && e.K == K && e.what == what && e.block == block && e.generation == generation) return e.choice;
  }
  const Choice choice = choose_uncached(what, M, N, K, block);
  std::lock_guard<std::mutex> lock(mu);
  e = Entry{M, N, K, generation, what, block, choice};
  return choice;
}

// Do the small tiles, at `mid` microseconds, stand back behind the decode kernel?  At 17 to 32 rows with row scales and one of its blocks per CU: with its
// whole share of K in flight it is up to 13 per cent ahead with the weights from memory (22 x 5536 x 640 4.3 us against 4.8, 18 x 6144 x 4096 8.5 and 9.1), as a
// model's are, and 5 to 20 behind with them in the memory-side cache (4.9 and 4.5, 8.6 and 8.1).  Block scales cost it more (20 x 6144 x 4096 8.4 and
// 8.6, 8.5 and 7.5), and at up to 16 rows, where it always runs, the two are 3 per cent apart either way.
static bool decode_ahead(int64_t M, int64_t N, int64_t K, bool block, float mid) {
  bool alone;
  return M <= 32 && !block && gemm_skinny_cost(M, N, K, &alone) < 1.02f * mid && alone;
}

// Which kernel MAXFP8_ALGO_AUTO gives a fast-layout matmul whose caller brings all the workspace it is asked for.  At most 16 rows: the decode kernel.  Up to
// 2048: the small tiles or the tiles, by the estimates, or, up to 32, the decode kernel.  Forced shapes keep the other kernels out, and beyond what the small
// tiles take the sizes alone decide.
static int choose_matmul(int64_t M, int64_t N, int64_t K, bool block) {
  const Tuning& t = tuning();
  const int plain = gemm_skinny_preferred(M, N, K) ? MAXFP8_ALGO_SKINNY : MAXFP8_ALGO_TILED;
  if (t.mid > 0) return gemm_mid_ok(M, N, K) ? kAlgoMid : plain;
  if (M <= 16 || !gemm_mid_ok(M, N, K) || t.mid == 0 || t.tile || t.splitk || t.one_region || t.w4 >= 0 || t.w4_split == 1 || t.skinny) return plain;
  float mid;
  gemm_mid_shape(M, N, K, block, &mid);
  if (decode_ahead(M, N, K, block, mid)) return MAXFP8_ALGO_SKINNY;
  const float tiles = gemm_tiled_cost(M, N, K, block);
  const bool large = N * K >= ((int64_t)1 << 26), whole = gemm_tiled_plan_workspace_bytes(M, N, K, block) == 0;
  // The tiles' estimate at up to 64 rows is of weights from memory and the small tiles' is not: the tiles may take more where the small ones need it -- large
  // weights, of long K above all (42 x 8192 x 28672 46 us on tiles, 54 on small ones, estimates 51 and 47), and few slabs in many blocks (45 x 24576 x 1536
  // 11.6 and 13.1, 12.7 and 9.9; 50 x 32768 x 512 7.0 and 8.6, 24 of them 6.7 and 7.0).
  if (M <= 64) {
    const float margin = whole && K <= 512 ? 1.36f : M <= 32 ? 0.95f : large ? (K >= 16384 ? 1.15f : whole ? 1.12f : 1.05f) : whole ? 1.30f : 0.95f;
    return tiles < margin * mid ? MAXFP8_ALGO_TILED : kAlgoMid;
  }
  // Beyond, both by their prices of the chip at work.  (Further from what the estimate was fitted to, or with more of its time spent on memory, or against whole
  // tiles, whose estimate is rough: 1730 x 592 x 5248 19 against 22 us, 79 x 7168 x 16384 35 against 38, 940 x 8320 x 1408 24 against 29.)
  // Up to 512 rows, from 64 slabs on, where the tiles split K: 0.95 of that, as the longest shares of K lose most when the weights come from memory (239 x 4784 x 9984 30 us on
  // tiles, on small ones 31 and from memory 36; 223 x 4096 x 14336 32, 30 and 36; 142 x 4096 x 14336 with row scales 29, 23 and 31; beyond 512 rows level from
  // memory and 6 per cent behind in the cache).
  const float margin = M > 1024 ? 0.80f : whole ? 0.85f : large ? 0.90f : 0.97f;
  return mid < (M <= 512 && !whole && K >= 8192 ? 0.95f * margin : margin) * tiles ? kAlgoMid : MAXFP8_ALGO_TILED;
}
static Choice choose_kernel(int64_t M, int64_t N, int64_t K, bool block) {
  if (M <= 16 && tuning().mid <= 0) return {MAXFP8_ALGO_SKINNY, 0};
  if (M > 2048) return {MAXFP8_ALGO_TILED, 0};
  return choose(Asked::kMatmul, M, N, K, block);
}
// the workspace MAXFP8_ALGO_AUTO uses with this scaling (up to 64 rows the choice of kernel asks whether the plan's is there)
static size_t auto_workspace(int64_t M, int64_t N, int64_t K, bool block) {
  if (choose_kernel(M, N, K, block).algo != MAXFP8_ALGO_TILED) return 0;
  return M > gemm_skinny_max_m() && gemm_tiled_needs_no_workspace(M, N, K, block) ? 0 : gemm_tiled_workspace_bytes(M, N, K);
}

// The same for the fused QKV matmul: decode kernel (at most 16 rows, and up to 32 where it is ahead -- more often than of a plain matmul, since the small tiles' store
// of K and V costs them 1 us with row scales: 18 x 6144 x 4096 9.4 us from memory against 10.5, in the cache 9.5 both --), the small tiles (17 to 64, where the tiles, whole, take 1.7 to 3 times
// as long, and beyond by their estimate) or the tiles, whose plan may cut them along K where the caller brings a workspace.  (348 x 5120 x 2048 15.6 us on tiles, on small ones 15.1 and from memory 16.8;
// 491 x 3072 x 2048 with row scales 16.4 and 17.9, 17.4 and 19.3; 209 x 4608 x 3584 21 and 14, 23 and 16.)
static int choose_qkv_matmul(int64_t T, int64_t N, int64_t K, bool has_workspace, bool block) {
  const Tuning& t = tuning();
  const int plain = T <= gemm_skinny_max_m() ? MAXFP8_ALGO_SKINNY : MAXFP8_ALGO_TILED;
  if (t.mid > 0) return gemm_mid_ok(T, N, K) ? kAlgoMid : plain;
  if (T <= 16 || !gemm_mid_ok(T, N, K) || t.mid == 0 || t.tile || t.skinny) return plain;
  float mid;
  gemm_mid_shape(T, N, K, block, &mid);
  if (plain == MAXFP8_ALGO_SKINNY) return decode_ahead(T, N, K, block, 1.07f * mid) ? MAXFP8_ALGO_SKINNY : kAlgoMid;
  return mid < (T > 256 ? 0.73f : 0.85f) * gemm_tiled_qkv_cost(T, N, K, block, has_workspace) ? kAlgoMid : MAXFP8_ALGO_TILED;
}
static Choice choose_qkv(int64_t T, int64_t N, int64_t K, bool has_workspace, bool block) {
  if (T <= 16 && tuning().mid <= 0) return {MAXFP8_ALGO_SKINNY, 0};
  if (T > 2048) return {MAXFP8_ALGO_TILED, 0};
  return choose(has_workspace ? Asked::kQkvWorkspace : Asked::kQkv, T, N, K, block);
}

// 17 to 64 rows whose tiles would split K, without the workspace for it
static int without_workspace(int64_t M, int64_t N, int64_t K, bool block) {
  const Tuning& t = tuning();
  if (!gemm_mid_ok(M, N, K) || t.skinny || t.mid == 0 || (M <= 16 && t.mid < 0)) return MAXFP8_ALGO_SKINNY;
  if (t.mid > 0) return kAlgoMid;
  float mid;
  gemm_mid_shape(M, N, K, block, &mid);
  return decode_ahead(M, N, K, block, mid) ? MAXFP8_ALGO_SKINNY : kAlgoMid;
}
static Choice choose_uncached(Asked what, int64_t M, int64_t N, int64_t K, bool block) {
  const int algo = what == Asked::kMatmul          ? choose_matmul(M, N, K, block)
                   : what == Asked::kMatmulNoSplit ? without_workspace(M, N, K, block)
                                                   : choose_qkv_matmul(M, N, K, what == Asked::kQkvWorkspace, block);
  return algo == kAlgoMid ? mid_choice(M, N, K, block) : Choice{algo, 0};
}
}  // namespace maxfp8

static int quantize_common(void* out_fp8, void* out_scales, const void* in, const uint32_t* row_index, uint32_t index_div,
                           int64_t M, int64_t K, int64_t in_row_stride, int64_t out_row_stride, int64_t group_size,
                           int64_t scales_ld, int in_dtype, int scales_dtype, float scale_ub, void* stream) {
  if (in_dtype != MAXFP8_BF16 && in_dtype != MAXFP8_F16 && in_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "quantize: input dtype %d is not bf16, f16 or f32", in_dtype);
  if (scales_dtype != MAXFP8_F32 && scales_dtype != MAXFP8_BF16)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "quantize: scales dtype should be bfloat16 or float32 (got %d)", scales_dtype);
  if (M < 0 || K < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize: negative size M=%lld K=%lld", (long long)M, (long long)K);
  if (M == 0 || K == 0) return MAXFP8_OK;  // fp8_quantization.mojo:428-429
  if (group_size == -1) group_size = K;
  if (group_size <= 0 || K % group_size != 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize: group size %lld must divide K = %lld", (long long)group_size, (long long)K);
  if (group_size % 4 != 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize: group size must be multiple of simd size (4), got %lld", (long long)group_size);
  if (in_row_stride < K || out_row_stride < K || scales_ld < M)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize: strides (in %lld, out %lld, scales %lld) smaller than the extents",
                (long long)in_row_stride, (long long)out_row_stride, (long long)scales_ld);
  if (!out_fp8 || !out_scales || !in) MAXFP8_FAIL(MAXFP8_ERR_NULL, "quantize: null pointer");
  return quantize_dispatch(out_fp8, out_scales, in, M, K, in_row_stride, out_row_stride, group_size, scales_ld,
                           in_dtype, scales_dtype, scale_ub, 1, 0, 0, 0, row_index, index_div, (hipStream_t)stream);
}

extern "C" {

int maxfp8_quantize_dynamic_scaled_fp8(void* out_fp8, void* out_scales, const void* in, int64_t M, int64_t K,
                                       int64_t in_row_stride, int64_t out_row_stride, int64_t group_size,
                                       int64_t scales_ld, int in_dtype, int scales_dtype, float scale_ub,
                                       void* stream) {
  return quantize_common(out_fp8, out_scales, in, nullptr, 1, M, K, in_row_stride, out_row_stride, group_size, scales_ld,
                         in_dtype, scales_dtype, scale_ub, stream);
}

int maxfp8_quantize_dynamic_scaled_fp8_gather(void* out_fp8, void* out_scales, const void* in, const uint32_t* row_index,
                                              int64_t index_div, int64_t M, int64_t K, int64_t in_row_stride,
                                              int64_t out_row_stride, int64_t group_size, int64_t scales_ld, int in_dtype,
                                              int scales_dtype, float scale_ub, void* stream) {
  if (M > 0 && K > 0 && !row_index) MAXFP8_FAIL(MAXFP8_ERR_NULL, "quantize (gather): null row index");
  if (index_div < 1 || index_div > 0xffffffffll) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize (gather): index_div must be at least 1");
  return quantize_common(out_fp8, out_scales, in, row_index, (uint32_t)index_div, M, K, in_row_stride, out_row_stride,
                         group_size, scales_ld, in_dtype, scales_dtype, scale_ub, stream);
}

int maxfp8_quantize_dynamic_scaled_fp8_scatter(void* out_fp8, void* out_scales, const void* in, const uint32_t* dst_index,
                                               int64_t copies, int64_t M, int64_t K, int64_t out_rows, int64_t in_row_stride,
                                               int64_t out_row_stride, int64_t group_size, int64_t scales_ld, int in_dtype,
                                               int scales_dtype, float scale_ub, void* stream) {
  if (M < 0 || K < 0 || out_rows < 0 || copies < 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize (scatter): negative size M=%lld K=%lld out_rows=%lld copies=%lld", (long long)M, (long long)K,
                (long long)out_rows, (long long)copies);
  if (M == 0 || K == 0 || copies == 0 || out_rows == 0) return MAXFP8_OK;
  if (in_dtype != MAXFP8_BF16 || scales_dtype != MAXFP8_F32 || group_size != 128)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "quantize (scatter): takes bfloat16 input, float32 scales and groups of 128 (got dtypes %d, %d, group %lld); "
                "the gather form takes the rest", in_dtype, scales_dtype, (long long)group_size);
  if (in_row_stride < K || out_row_stride < K || scales_ld < out_rows)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize (scatter): strides (in %lld, out %lld, scales %lld) smaller than the extents",
                (long long)in_row_stride, (long long)out_row_stride, (long long)scales_ld);
  if (!out_fp8 || !out_scales || !in || !dst_index) MAXFP8_FAIL(MAXFP8_ERR_NULL, "quantize (scatter): null pointer");
  const int rc = quantize_scatter_dispatch(out_fp8, out_scales, in, M, K, in_row_stride, out_row_stride, scales_ld, scale_ub, dst_index,
                                           copies, out_rows, (hipStream_t)stream);
  if (rc == -1)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize (scatter): rows must be 16-byte aligned and K a multiple of 128; the gather form takes the rest");
  return rc;
}

int maxfp8_batched_quantize_dynamic_scaled_fp8(void* out_fp8, void* out_scales, const void* in, int64_t B, int64_t M, int64_t K,
                                               int64_t in_batch_stride, int64_t in_row_stride, int64_t out_batch_stride,
                                               int64_t out_row_stride, int64_t group_size, int64_t scales_batch_stride,
                                               int64_t scales_ld, int in_dtype, int scales_dtype, float scale_ub,
                                               void* stream) {
  if (B < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "batched quantize: negative batch");
  if (B == 0) return MAXFP8_OK;  // fp8_quantization.mojo:826-827
  if (B > 65535) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "batched quantize: batch %lld exceeds 65535", (long long)B);
  if (in_dtype != MAXFP8_BF16 && in_dtype != MAXFP8_F16 && in_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "quantize: input dtype %d is not bf16, f16 or f32", in_dtype);
  if (scales_dtype != MAXFP8_F32 && scales_dtype != MAXFP8_BF16)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "quantize: scales dtype should be bfloat16 or float32 (got %d)", scales_dtype);
  if (M < 0 || K < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize: negative size M=%lld K=%lld", (long long)M, (long long)K);
  if (M == 0 || K == 0) return MAXFP8_OK;
  if (group_size == -1) group_size = K;
  if (group_size <= 0 || K % group_size != 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize: group size %lld must divide K = %lld", (long long)group_size, (long long)K);
  if (group_size % 4 != 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize: group size must be multiple of simd size (4), got %lld", (long long)group_size);
  if (in_row_stride < K || out_row_stride < K || scales_ld < M)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize: strides smaller than the extents");
  if (!out_fp8 || !out_scales || !in) MAXFP8_FAIL(MAXFP8_ERR_NULL, "quantize: null pointer");
  return quantize_dispatch(out_fp8, out_scales, in, M, K, in_row_stride, out_row_stride, group_size, scales_ld, in_dtype,
                           scales_dtype, scale_ub, B, in_batch_stride, out_batch_stride, scales_batch_stride, nullptr, 1,
                           (hipStream_t)stream);
}

int maxfp8_rms_norm_fused_quantize_dynamic_scaled_fp8(void* out_fp8, void* out_scales, const void* in, const void* gamma,
                                                      int64_t rows, int64_t K, int64_t in_row_stride,
                                                      int64_t out_row_stride, int in_dtype, int scales_dtype,
                                                      float epsilon, float weight_offset, float scale_ub, void* stream) {
  if (in_dtype != MAXFP8_BF16 && in_dtype != MAXFP8_F16 && in_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "rms_norm_fused_quantize: input dtype %d is not bf16, f16 or f32", in_dtype);
  if (scales_dtype != MAXFP8_F32 && scales_dtype != MAXFP8_BF16)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "rms_norm_fused_quantize: scales dtype should be bfloat16 or float32 (got %d)", scales_dtype);
  if (rows < 0 || K < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "rms_norm_fused_quantize: negative size");
  if (rows == 0 || K == 0) return MAXFP8_OK;
  if (rows >= ((int64_t)1 << 31) || K >= ((int64_t)1 << 31)) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "rms_norm_fused_quantize: sizes must fit 31 bits");
  if (in_row_stride < K || out_row_stride < K)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "rms_norm_fused_quantize: row strides smaller than the row length");
  if (!out_fp8 || !out_scales || !in || !gamma) MAXFP8_FAIL(MAXFP8_ERR_NULL, "rms_norm_fused_quantize: null pointer");
  return rmsnorm_quantize_dispatch(out_fp8, out_scales, in, gamma, rows, K, in_row_stride, out_row_stride, in_dtype,
                                   scales_dtype, round_to_dtype(epsilon, in_dtype), round_to_dtype(weight_offset, in_dtype),
                                   scale_ub, (hipStream_t)stream);
}

int maxfp8_quantize_static_scaled_fp8(void* out_fp8, const void* in, int64_t M, int64_t K, int64_t in_row_stride,
                                      int64_t out_row_stride, int in_dtype, float scale, void* stream) {
  if (in_dtype != MAXFP8_BF16 && in_dtype != MAXFP8_F16 && in_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "quantize_static: expected input dtype to be float16, bfloat16, or float32 (got %d)", in_dtype);
  if (M < 0 || K < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize_static: negative size");
  if (M == 0 || K == 0) return MAXFP8_OK;
  if (in_row_stride < K || out_row_stride < K) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize_static: row strides smaller than the row length");
  if (!out_fp8 || !in) MAXFP8_FAIL(MAXFP8_ERR_NULL, "quantize_static: null pointer");
  return quantize_static_dispatch(out_fp8, in, M, K, in_row_stride, out_row_stride, in_dtype, scale, (hipStream_t)stream);
}

int maxfp8_quantize_tensor_dynamic_scaled_fp8(void* out_fp8, void* out_scales, const void* in, int64_t M, int64_t K,
                                              int64_t in_row_stride, int64_t out_row_stride, int in_dtype, int scales_dtype,
                                              float scale_ub, void* stream) {
  if (in_dtype != MAXFP8_BF16 && in_dtype != MAXFP8_F16 && in_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "quantize_tensor: input dtype %d is not bf16, f16 or f32", in_dtype);
  if (scales_dtype != MAXFP8_F32 && scales_dtype != MAXFP8_BF16)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "quantize_tensor: scales dtype should be bfloat16 or float32 (got %d)", scales_dtype);
  if (M < 0 || K < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize_tensor: negative size");
  if (M == 0 || K == 0) return MAXFP8_OK;  // fp8_quantization.mojo:296-297
  if (M >= ((int64_t)1 << 31)) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize_tensor: M must fit 31 bits");
  if (K % 4 != 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize_tensor: group size must be multiple of simd size (4), got %lld", (long long)K);
  if (in_row_stride < K || out_row_stride < K) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "quantize_tensor: row strides smaller than the row length");
  if (!out_fp8 || !out_scales || !in) MAXFP8_FAIL(MAXFP8_ERR_NULL, "quantize_tensor: null pointer");
  return quantize_tensor_dispatch(out_fp8, out_scales, in, M, K, in_row_stride, out_row_stride, in_dtype, scales_dtype,
                                  scale_ub, (hipStream_t)stream);
}

int maxfp8_moe_create_indices(uint32_t* token_expert_order, uint32_t* expert_start_indices, uint32_t* restore_token_order,
                              int32_t* expert_ids, uint32_t* expert_usage_stats, const void* topk_ids, int64_t n,
                              int64_t num_experts, void* stream) {
  if (n < 0 || num_experts < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "moe_create_indices: negative size");
  if (n >= ((int64_t)1 << 31) || num_experts > 65535)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "moe_create_indices: %lld assignments / %lld experts exceed the limits", (long long)n,
                (long long)num_experts);
  if (!expert_usage_stats || !expert_start_indices) MAXFP8_FAIL(MAXFP8_ERR_NULL, "moe_create_indices: null pointer");
  if (num_experts == 0) return MAXFP8_OK;
  if (!expert_ids || (n > 0 && (!token_expert_order || !restore_token_order || !topk_ids)))
    MAXFP8_FAIL(MAXFP8_ERR_NULL, "moe_create_indices: null pointer");
  return moe_create_indices_dispatch(token_expert_order, expert_start_indices, restore_token_order, expert_ids,
                                     expert_usage_stats, (const int32_t*)topk_ids, n, num_experts, (hipStream_t)stream);
}

static int fused_silu_common(void* out, void* out_scales, const void* in, const uint32_t* row_offsets, int64_t num_offsets,
                             int64_t max_rows, int64_t inter, int64_t in_row_stride, int64_t out_row_stride, int64_t scales_ld,
                             int in_dtype, int mode, bool row_scales, float scale_ub, void* stream) {
  if (in_dtype != MAXFP8_BF16) MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "fused_silu: input dtype %d is not bf16", in_dtype);
  if (max_rows < 0 || inter < 0 || num_offsets < 1) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused_silu: bad sizes");
  if (max_rows == 0 || inter == 0) return MAXFP8_OK;
  // (max_rows is a bound: only the form with one block per row makes it its grid)
  if (inter >= ((int64_t)1 << 31) || (row_scales && max_rows >= ((int64_t)1 << 31))) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused_silu: sizes must fit 31 bits");
  if (inter % 128 != 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused_silu: the output width %lld must be a multiple of 128", (long long)inter);
  const bool quant = mode != 0 && mode != 2;
  if (in_row_stride < 2 * inter || out_row_stride < inter || (quant && !row_scales && scales_ld < max_rows))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused_silu: strides smaller than the extents");
  if (!out || !in || !row_offsets || (quant && !out_scales)) MAXFP8_FAIL(MAXFP8_ERR_NULL, "fused_silu: null pointer");
  if (!is_aligned(in, 16) || in_row_stride % 8 != 0 || !is_aligned(out, 16) || out_row_stride % 8 != 0)
    MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "fused_silu: rows must be 16-byte aligned");
  return fused_silu_dispatch(out, (float*)out_scales, in, row_offsets, num_offsets, max_rows, inter, in_row_stride,
                             out_row_stride, scales_ld, mode, row_scales, scale_ub, (hipStream_t)stream);
}

int maxfp8_fused_silu(void* out, void* out_scales, const void* in, const uint32_t* row_offsets, int64_t num_offsets,
                      int64_t max_rows, int64_t inter, int64_t in_row_stride, int64_t out_row_stride, int64_t scales_ld,
                      int in_dtype, int quantize, void* stream) {
  if (quantize < 0 || quantize > 2) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused_silu: quantize = %d is not 0, 1 or 2", quantize);
  return fused_silu_common(out, out_scales, in, row_offsets, num_offsets, max_rows, inter, in_row_stride, out_row_stride, scales_ld,
                           in_dtype, quantize, false, 0.0f, stream);
}

int maxfp8_silu_quantize_dynamic_scaled_fp8(void* out_fp8, void* out_scales, const void* in, const uint32_t* row_offsets,
                                            int64_t num_offsets, int64_t max_rows, int64_t inter, int64_t in_row_stride,
                                            int64_t out_row_stride, int64_t group_size, int64_t scales_ld, int in_dtype,
                                            int round_activation, float scale_ub, void* stream) {
  if (group_size != 128 && group_size != inter)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "silu_quantize: group size %lld is not 128 or the row's %lld outputs", (long long)group_size, (long long)inter);
  return fused_silu_common(out_fp8, out_scales, in, row_offsets, num_offsets, max_rows, inter, in_row_stride, out_row_stride, scales_ld,
                           in_dtype, round_activation ? 4 : 3, group_size != 128, scale_ub, stream);
}

size_t maxfp8_matmul_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || (gemm_skinny_preferred(M, N, K) && !auto_workspace(M, N, K, true) && !auto_workspace(M, N, K, false))) return 0;
  return gemm_tiled_workspace_bytes(M, N, K);  // split-K partial sums; 0 when no split would be used
}

size_t maxfp8_matmul_auto_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const size_t block = auto_workspace(M, N, K, true);
  return block ? block : auto_workspace(M, N, K, false);
}

}  // extern "C"

namespace maxfp8 {
struct BatchStrides { int64_t n, a, b, c, a_scales, b_scales; };  // n batches; steps in elements

// A batch of short K and more than 32 rows on the tiles (one slab mostly has a kernel of its own): one slab of K leaves three of the decode
// kernel's four waves idle, and beyond one of its 16-row blocks per CU every block more reads the tokens again.  With one block per CU or less it is ahead from
// two slabs on (decode kernel against tiles, 48 rows, us, cold: 32 x 512 -> 128 5.4 and 6.4, 48 of them 7.8 and 6.5, 128 12.7
// and 6.7; 16 x 256 -> 256 4.8 and 5.3, 24 of them 6.3 and 5.3; 16 x 128 -> 512 5.6 and 4.8, 128 of them 28.7 and 6.7).
static bool batch_on_tiles(int64_t batch, int64_t M, int64_t N, int64_t K) {
  return M > 32 && K <= 512 && (K <= 128 || ceil_div(N, 16) * batch > (int64_t)compute_units());
}

static int matmul_common(void* c, const void* a, const void* b, const void* a_scales, const void* b_scales, int64_t M,
                         int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int input_granularity,
                         int weight_granularity, int64_t gm, int64_t gn, int64_t gk, int64_t a_scales_ld,
                         int64_t b_scales_ld, int c_dtype, int scales_dtype, int algo, void* workspace,
                         size_t workspace_bytes, const BatchStrides& bt, void* stream) {
  if (c_dtype != MAXFP8_BF16 && c_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "matmul: output dtype %d is not bf16 or f32", c_dtype);
  if (M < 0 || N < 0 || K < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "matmul: negative size");
  if (M == 0 || N == 0) return MAXFP8_OK;  // fp8_quantization.mojo:1103-1104
  if (M >= ((int64_t)1 << 31) || N >= ((int64_t)1 << 31) || K >= ((int64_t)1 << 31))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "matmul: sizes must fit 31 bits");
  if (lda < K || ldb < K || ldc < N) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "matmul: leading dimension smaller than the row length");
  if (!c || !a || !b || !a_scales || !b_scales) MAXFP8_FAIL(MAXFP8_ERR_NULL, "matmul: null pointer");

  const bool block = input_granularity == MAXFP8_GRAN_BLOCK && weight_granularity == MAXFP8_GRAN_BLOCK;
  const bool row = input_granularity == MAXFP8_GRAN_COLWISE && weight_granularity == MAXFP8_GRAN_ROWWISE;
  const bool tensor = input_granularity == MAXFP8_GRAN_TENSOR && weight_granularity == MAXFP8_GRAN_TENSOR;
  if (!block && !row && !tensor) MAXFP8_FAIL(MAXFP8_ERR_GRANULARITY, "unsupported FP8 scaling granularity");
  hipStream_t st = (hipStream_t)stream;

  if (block) {
    if (scales_dtype != MAXFP8_F32) MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "a_scales and b_scales dtypes must be float32");
    if (gm <= 0 || gn <= 0 || gk <= 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "matmul: block granularities must be positive");
    if (a_scales_ld < ceil_div(M, gm) || b_scales_ld < ceil_div(K, gk))
      MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "matmul: scale leading dimensions too small");
  } else if (scales_dtype != MAXFP8_F32 && scales_dtype != MAXFP8_BF16 && scales_dtype != MAXFP8_F16) {
    // the three scale dtypes of the reference (fp8_quantization.mojo:996-1018)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "matmul: scales dtype %d is not f32, bf16 or f16", scales_dtype);
  }

  // Fast kernels: 16-byte aligned rows, K a multiple of 16, and for block scaling the
  // (1, 128, 128) granularity.  (Row / tensor scales of any dtype are widened in the epilogue.)
  const bool fast_layout = is_aligned(a, 16) && is_aligned(b, 16) && lda % 16 == 0 && ldb % 16 == 0 && K % 16 == 0 &&
                           K > 0 && (!block || (gm == 1 && gn == 128 && gk == 128)) &&
                           (bt.n == 1 || (bt.a % 16 == 0 && bt.b % 16 == 0)) && offsets_fit(K, lda, ldb, a_scales_ld, block);
  const bool automatic = algo == MAXFP8_ALGO_AUTO;
  int shape = 0;  // of the small tiles
  if (automatic) {
    if (!fast_layout) algo = MAXFP8_ALGO_NAIVE;
    else if (bt.n == 1) { const Choice c = choose_kernel(M, N, K, block); algo = c.algo; shape = c.shape; }
    else if (gemm_skinny_preferred(M, N, K) && !batch_on_tiles(bt.n, M, N, K)) algo = MAXFP8_ALGO_SKINNY;
    else algo = MAXFP8_ALGO_TILED;
    // 33 to 64 rows: the tiles win through their K split.  Without the workspace the split needs, a narrow weight
    // matrix would run on a fraction of the chip: the streaming kernel then.  (What this shape's own plan needs, not the
    // worst case over all tile shapes: a plan that does not split runs the same with and without a workspace.)
    if (algo == MAXFP8_ALGO_TILED && M <= gemm_skinny_max_m() && bt.n == 1 &&
        gemm_tiled_plan_workspace_bytes(M, N, K, block) > (workspace ? workspace_bytes : 0)) {
      const Choice c = choose(Asked::kMatmulNoSplit, M, N, K, block);
      algo = c.algo;
      shape = c.shape;
    }
  }
  if (algo == MAXFP8_ALGO_NAIVE) {
    if (block)
      return naive_blockwise_dispatch(c, a, b, a_scales, b_scales, M, N, K, lda, ldb, ldc, gm, gn, gk, a_scales_ld,
                                      b_scales_ld, c_dtype, bt.n, bt.a, bt.b, bt.c, bt.a_scales, bt.b_scales, st);
    if (bt.n != 1) MAXFP8_FAIL(MAXFP8_ERR_GRANULARITY, "batched matmul: only block scaling is supported");
    return naive_rowwise_dispatch(c, a, b, a_scales, b_scales, M, N, K, lda, ldb, ldc, tensor ? 0 : 1,
                                  tensor ? 0 : b_scales_ld, c_dtype, scales_dtype, st);
  }
  if (algo != MAXFP8_ALGO_TILED && algo != MAXFP8_ALGO_SKINNY && !(automatic && algo == kAlgoMid))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "matmul: unknown algo %d", algo);
  if (!fast_layout)
    MAXFP8_FAIL(MAXFP8_ERR_ALIGN,
                "matmul: the MFMA kernels need 16-byte aligned rows, K %% 16 == 0, (1,128,128) blocks and "
                "row strides below 2^31 / 256 bytes");

  GemmArgs p;
  memset(&p, 0, sizeof(p));
  p.a = (const uint8_t*)a;
  p.b = (const uint8_t*)b;
  p.c = c;
  p.a_scales = (const float*)a_scales;
  p.b_scales = (const float*)b_scales;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.a_scales_ld = a_scales_ld;
  p.b_scales_ld = b_scales_ld;
  p.a_scale_stride = tensor ? 0 : 1;
  p.b_scale_stride = tensor ? 0 : b_scales_ld;
  p.c_dtype = c_dtype;
  p.scales_dtype = scales_dtype;  // (f32 for block scaling, checked above)
  p.c_vec_ok = (ldc % 4 == 0) && is_aligned(c, c_dtype == MAXFP8_BF16 ? 8 : 16);
  p.c_vec8_ok = (ldc % 8 == 0) && is_aligned(c, 16);
  if (bt.n != 1) {  // every batch's C must keep the alignment the vector stores assume
    p.c_vec_ok = p.c_vec_ok && bt.c % 4 == 0;
    p.c_vec8_ok = p.c_vec8_ok && bt.c % 8 == 0;
  }
  p.a_batch = bt.a; p.b_batch = bt.b; p.c_batch = bt.c;
  p.a_scales_batch = bt.a_scales; p.b_scales_batch = bt.b_scales;
  if (algo == kAlgoMid) return gemm_mid_dispatch(p, block, shape, st);
  if (automatic && gemm_one_slab_ok(p, block, bt.n)) return gemm_one_slab_dispatch(p, bt.n, st);
  if (automatic && gemm_short_k_ok(p, block, bt.n)) return gemm_short_k_dispatch(p, bt.n, st);
  if (algo == MAXFP8_ALGO_SKINNY) return gemm_skinny_dispatch(p, block, bt.n, st);
  if (workspace && !is_aligned(workspace, 16)) MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "matmul: workspace must be 16-byte aligned");
  p.workspace = (float*)workspace;
  return gemm_tiled_dispatch(p, block, workspace_bytes, bt.n, st);
}
}  // namespace maxfp8

extern "C" {

int maxfp8_matmul_tall(int64_t M, int64_t N, int64_t K, int block_scaling, int with_workspace) {
  if (M <= 0 || N <= 0 || K <= 0 || choose_kernel(M, N, K, block_scaling != 0).algo != MAXFP8_ALGO_TILED) return 0;
  return gemm_tiled_tall(M, N, K, block_scaling != 0, with_workspace != 0);
}

int maxfp8_matmul_describe(int64_t M, int64_t N, int64_t K, int block_scaling, int with_workspace, char* buf, size_t len) {
  if (!buf || len == 0) return 0;
  if (M <= 0 || N <= 0 || K <= 0) return snprintf(buf, len, "nothing to do");
  Choice c = choose_kernel(M, N, K, block_scaling != 0);
  if (c.algo == MAXFP8_ALGO_TILED && M <= gemm_skinny_max_m() && !with_workspace && gemm_tiled_plan_workspace_bytes(M, N, K, block_scaling != 0) > 0)
    c = choose(Asked::kMatmulNoSplit, M, N, K, block_scaling != 0);
  if (c.algo == MAXFP8_ALGO_SKINNY) return snprintf(buf, len, "skinny");
  if (c.algo == kAlgoMid) {
    const int sel = c.shape;
    const int bm = 16 * (sel / 10 % 10), bn = 16 * (sel % 10);
    return snprintf(buf, len, "%dx%d x%lld, %d per CU, K split over the block's waves", bm, bn, (long long)(ceil_div(M, bm) * ceil_div(N, bn)), sel / 100);
  }
  return gemm_tiled_describe(M, N, K, block_scaling != 0, with_workspace != 0, buf, len);
}

int maxfp8_matmul_dynamic_scaled_fp8(void* c, const void* a, const void* b, const void* a_scales,
                                     const void* b_scales, int64_t M, int64_t N, int64_t K, int64_t lda,
                                     int64_t ldb, int64_t ldc, int input_granularity, int weight_granularity,
                                     int64_t gm, int64_t gn, int64_t gk, int64_t a_scales_ld, int64_t b_scales_ld,
                                     int c_dtype, int scales_dtype, int algo, void* workspace,
                                     size_t workspace_bytes, void* stream) {
  const BatchStrides one = {1, 0, 0, 0, 0, 0};
  return matmul_common(c, a, b, a_scales, b_scales, M, N, K, lda, ldb, ldc, input_granularity, weight_granularity, gm, gn,
                       gk, a_scales_ld, b_scales_ld, c_dtype, scales_dtype, algo, workspace, workspace_bytes, one, stream);
}

size_t maxfp8_matmul_noalloc_max_scratch_bytes(void) { return kScratchBytes; }

int maxfp8_matmul_dynamic_scaled_fp8_noalloc(void* c, const void* a, const void* b, const void* a_scales,
                                             const void* b_scales, int64_t M, int64_t N, int64_t K, int64_t lda,
                                             int64_t ldb, int64_t ldc, int input_granularity, int weight_granularity,
                                             int64_t gm, int64_t gn, int64_t gk, int64_t a_scales_ld, int64_t b_scales_ld,
                                             int c_dtype, int scales_dtype, int algo, void* stream) {
  // The scratch of the K split this shape gets when its caller brings all the workspace
  // maxfp8_matmul_workspace_bytes asks for: with exactly that much the planner lands on the same plan, so both
  // entry points add the same partial sums in the same order.
  const bool block = input_granularity == MAXFP8_GRAN_BLOCK && weight_granularity == MAXFP8_GRAN_BLOCK;
  size_t need = 0;
  if (M > 0 && N > 0 && K > 0 && (algo == MAXFP8_ALGO_AUTO ? auto_workspace(M, N, K, block) : maxfp8_matmul_workspace_bytes(M, N, K)) > 0) need = gemm_tiled_plan_workspace_bytes(M, N, K, block);
  if (need > kScratchBytes)
    MAXFP8_FAIL(MAXFP8_ERR_WORKSPACE,
                "matmul (no-alloc): the split of %lld x %lld x %lld uses %zu bytes of scratch, the library's static buffer holds "
                "%zu; call maxfp8_matmul_dynamic_scaled_fp8 with workspace = NULL (no split, no allocation) or with a workspace",
                (long long)M, (long long)N, (long long)K, need, kScratchBytes);
  void* ws = nullptr;
  if (need > 0 && M > 0 && N > 0) {
    const int rc = scratch_of_current_device(&ws);
    if (rc != MAXFP8_OK) return rc;
  }
  // (Nothing in the scratch has to start at zero: every partial tile a split writes is written in full before the
  // reduction reads it.  Its contents after the call are the last call's partial sums.)
  const BatchStrides one = {1, 0, 0, 0, 0, 0};
  return matmul_common(c, a, b, a_scales, b_scales, M, N, K, lda, ldb, ldc, input_granularity, weight_granularity, gm, gn,
                       gk, a_scales_ld, b_scales_ld, c_dtype, scales_dtype, algo, ws, ws ? need : 0, one, stream);
}

// ---- a whole linear: quantise bf16 activations, then the scaled matmul --------------------------------------------
// What the two launches of a linear keep in the caller's workspace: fp8 activations, their scales, the matmul's partial sums.
}  // extern "C"
namespace maxfp8 {
struct LinearLayout { size_t scales, partial, partial_bytes, total; int64_t scales_ld; };
// (plain: the matmul behind it is the plain one, whose workspace comes last)
static LinearLayout linear_layout(int64_t M, int64_t N, int64_t K, bool block, bool fixed, bool plain = true) {
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  LinearLayout l;
  l.scales_ld = block ? ceil_div(M, 4) * 4 : M;
  l.scales = up((size_t)M * (size_t)K);
  l.partial = l.scales + up((fixed ? 2 : block ? (size_t)(K / 128) * l.scales_ld : (size_t)M) * 4);
  l.partial_bytes = plain && M > 0 && N > 0 && K > 0 ? auto_workspace(M, N, K, block) : 0;
  l.total = l.partial + l.partial_bytes;
  return l;
}
// does the decode kernel quantise by itself? (the layout as far as it is the operands': see linear_common)
static bool linear_in_one(int64_t M, int64_t N, int64_t K, bool block) {
  return M > 0 && N > 0 && K > 0 && choose_kernel(M, N, K, block).algo == MAXFP8_ALGO_SKINNY && gemm_skinny_quant_ok(M, N, K, block);
}

static int linear_common(void* y, const void* x, const void* w, const void* w_scales, int64_t M, int64_t N, int64_t K, int64_t ldx,
                         int64_t ldw, int64_t ldy, bool block, int64_t w_scales_ld, bool fixed, float input_scale, float weight_scale,
                         float scale_ub, void* workspace, size_t workspace_bytes, void* stream) {
  if (M < 0 || N < 0 || K < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "linear: negative size");
  if (M == 0 || N == 0) return MAXFP8_OK;
  if (M >= ((int64_t)1 << 31) || N >= ((int64_t)1 << 31) || K >= ((int64_t)1 << 31)) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "linear: sizes must fit 31 bits");
  if (ldx < K || ldw < K || ldy < N) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "linear: row strides smaller than the rows");
  if (K <= 0 || K % (block ? 128 : 4) != 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "linear: K = %lld is not a positive multiple of %d", (long long)K, block ? 128 : 4);
  if (block && w_scales_ld < K / 128) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "linear: scale leading dimension too small");
  if (!y || !x || !w || (!fixed && !w_scales)) MAXFP8_FAIL(MAXFP8_ERR_NULL, "linear: null pointer");
  hipStream_t st = (hipStream_t)stream;
  if (linear_in_one(M, N, K, block) && is_aligned(x, 16) && ldx % 8 == 0 && is_aligned(w, 16) && ldw % 16 == 0 && K % 16 == 0 &&
      offsets_fit(K, ldw, ldw, 0, false) && 32 * ldx < ((int64_t)1 << 31)) {
    GemmArgs p;
    memset(&p, 0, sizeof(p));
    p.b = (const uint8_t*)w;
    p.c = y;
    p.b_scales = (const float*)w_scales;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    p.ldb = ldw; p.ldc = ldy;
    p.b_scales_ld = w_scales_ld;
    p.b_scale_stride = w_scales_ld;
    p.c_dtype = MAXFP8_BF16;
    p.scales_dtype = MAXFP8_F32;
    p.c_vec_ok = (ldy % 4 == 0) && is_aligned(y, 8);
    p.x = (const uint16_t*)x;
    p.ldx = ldx;
    p.x_static = fixed ? 1 : 0;
    p.x_scale_ub = scale_ub;
    p.x_recip = fixed ? 1.0f / input_scale : 0.f;
    p.x_scale = input_scale * weight_scale;
    return gemm_skinny_quant_dispatch(p, block, st);
  }
  const LinearLayout l = linear_layout(M, N, K, block, fixed);
  if (!workspace || workspace_bytes < l.total)
    MAXFP8_FAIL(MAXFP8_ERR_WORKSPACE, "linear: %lld x %lld x %lld needs %zu bytes of workspace (maxfp8_linear_workspace_bytes), got %zu", (long long)M,
                (long long)N, (long long)K, l.total, workspace ? workspace_bytes : (size_t)0);
  if (!is_aligned(workspace, 16)) MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "linear: workspace must be 16-byte aligned");
  uint8_t* q = (uint8_t*)workspace;
  float* scales = (float*)(q + l.scales);
  int rc;
  if (fixed) rc = quantize_static_for_matmul_dispatch(q, scales, x, M, K, ldx, MAXFP8_BF16, input_scale, weight_scale, st);
  else rc = quantize_dispatch(q, scales, x, M, K, ldx, K, block ? 128 : K, l.scales_ld, MAXFP8_BF16, MAXFP8_F32, scale_ub, 1, 0, 0, 0, nullptr, 1, st);
  if (rc != MAXFP8_OK) return rc;
  const int gran_in = fixed ? MAXFP8_GRAN_TENSOR : block ? MAXFP8_GRAN_BLOCK : MAXFP8_GRAN_COLWISE;
  const int gran_w = fixed ? MAXFP8_GRAN_TENSOR : block ? MAXFP8_GRAN_BLOCK : MAXFP8_GRAN_ROWWISE;
  const BatchStrides one = {1, 0, 0, 0, 0, 0};
  return matmul_common(y, q, w, scales, fixed ? scales + 1 : w_scales, M, N, K, K, ldw, ldy, gran_in, gran_w, block ? 1 : -1, block ? 128 : -1,
                       block ? 128 : -1, l.scales_ld, fixed ? 1 : w_scales_ld, MAXFP8_BF16, MAXFP8_F32, MAXFP8_ALGO_AUTO,
                       l.partial_bytes ? q + l.partial : nullptr, l.partial_bytes, one, st);
}
}  // namespace maxfp8
extern "C" {

size_t maxfp8_linear_workspace_bytes(int64_t M, int64_t N, int64_t K, int weight_granularity) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const bool block = weight_granularity == MAXFP8_GRAN_BLOCK;
  return linear_in_one(M, N, K, block) ? 0 : linear_layout(M, N, K, block, weight_granularity == MAXFP8_GRAN_TENSOR).total;
}

int maxfp8_linear_dynamic_scaled_fp8(void* y, const void* x, const void* w, const void* w_scales, int64_t M, int64_t N, int64_t K,
                                     int64_t x_row_stride, int64_t ldw, int64_t ldy, int weight_granularity, int64_t w_scales_ld,
                                     float scale_ub, void* workspace, size_t workspace_bytes, void* stream) {
  if (weight_granularity != MAXFP8_GRAN_BLOCK && weight_granularity != MAXFP8_GRAN_ROWWISE)
    MAXFP8_FAIL(MAXFP8_ERR_GRANULARITY, "linear: weight granularity %d is not block or rowwise", weight_granularity);
  return linear_common(y, x, w, w_scales, M, N, K, x_row_stride, ldw, ldy, weight_granularity == MAXFP8_GRAN_BLOCK, w_scales_ld, false, 1.f, 1.f,
                       scale_ub, workspace, workspace_bytes, stream);
}

int maxfp8_linear_static_scaled_fp8(void* y, const void* x, const void* w, int64_t M, int64_t N, int64_t K, int64_t x_row_stride,
                                    int64_t ldw, int64_t ldy, float input_scale, float weight_scale, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  return linear_common(y, x, w, nullptr, M, N, K, x_row_stride, ldw, ldy, false, 1, true, input_scale, weight_scale, 0.f, workspace,
                       workspace_bytes, stream);
}

int maxfp8_batched_matmul_dynamic_scaled_fp8(void* c, const void* a, const void* b, const void* a_scales,
                                             const void* b_scales, int64_t B, int64_t M, int64_t N, int64_t K,
                                             int64_t a_batch_stride, int64_t lda, int64_t b_batch_stride, int64_t ldb,
                                             int64_t c_batch_stride, int64_t ldc, int64_t gm, int64_t gn, int64_t gk,
                                             int64_t a_scales_batch_stride, int64_t a_scales_ld,
                                             int64_t b_scales_batch_stride, int64_t b_scales_ld, int c_dtype,
                                             int scales_dtype, int algo, void* stream) {
  if (B < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "batched matmul: negative batch");
  if (B == 0) return MAXFP8_OK;
  if (B > 65535) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "batched matmul: batch %lld exceeds 65535", (long long)B);
  const BatchStrides bt = {B, a_batch_stride, b_batch_stride, c_batch_stride, a_scales_batch_stride, b_scales_batch_stride};
  return matmul_common(c, a, b, a_scales, b_scales, M, N, K, lda, ldb, ldc, MAXFP8_GRAN_BLOCK, MAXFP8_GRAN_BLOCK, gm, gn, gk,
                       a_scales_ld, b_scales_ld, c_dtype, scales_dtype, algo, nullptr, 0, bt, stream);
}

}  // extern "C"

// x != nullptr: the decode kernel quantises x (bf16 rows of ldx elements) by itself; input and input_scale are not used.
// chosen: what the caller has found for MAXFP8_ALGO_AUTO, with the workspace that takes; nullptr: it is chosen here, without any.
static int qkv_common(void* output, const void* input, const void* x, int64_t ldx, float scale_ub, const uint32_t* input_row_offsets,
                                               const void* wqkv, const void* input_scale, const void* weight_scale,
                                               void* kv_blocks, const uint32_t* cache_lengths, const uint32_t* lookup_table,
                                               const void* bias, int64_t T, int64_t N, int64_t K, int64_t q_dim,
                                               int64_t batch_size, int64_t num_blocks, int64_t kv_dim, int64_t num_layers,
                                               int64_t layer_idx, int64_t page_size, int64_t num_kv_heads, int64_t head_dim,
                                               int64_t lut_ld, int64_t gm, int64_t gn, int64_t gk, int64_t input_scale_ld,
                                               int64_t weight_scale_ld, int scales_dtype, int algo, const Choice* chosen, void* workspace,
                                               size_t workspace_bytes, void* stream) {
  if (T < 0 || N < 0 || K < 0 || q_dim < 0 || batch_size < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused qkv matmul: negative size");
  if (batch_size == 0 || T == 0 || N == 0) return MAXFP8_OK;  // kv_cache_ragged.mojo:1193-1194
  if (T >= ((int64_t)1 << 31) || N >= ((int64_t)1 << 31) || K >= ((int64_t)1 << 31) || batch_size >= ((int64_t)1 << 31))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused qkv matmul: sizes must fit 31 bits");
  if (kv_dim != 1 && kv_dim != 2) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused qkv matmul: the cache holds 2 (K, V) or 1 (MLA) planes, got %lld", (long long)kv_dim);
  if (num_blocks <= 0 || num_layers <= 0 || layer_idx < 0 || layer_idx >= num_layers || page_size <= 0 || num_kv_heads <= 0 ||
      head_dim <= 0 || lut_ld <= 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused qkv matmul: bad cache geometry");
  const int64_t k_dim = num_kv_heads * head_dim;
  const int64_t rest = N - q_dim;
  if (rest != k_dim && !(rest == 2 * k_dim && kv_dim == 2))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused qkv matmul: N = %lld is not q_dim %lld plus one or two times kv_heads * head_dim = %lld",
                (long long)N, (long long)q_dim, (long long)k_dim);
  if ((!x && (!input || !input_scale)) || !wqkv || !weight_scale || !kv_blocks || !cache_lengths || !lookup_table || !input_row_offsets ||
      (q_dim > 0 && !output))
    MAXFP8_FAIL(MAXFP8_ERR_NULL, "fused qkv matmul: null pointer");
  if (scales_dtype != MAXFP8_F32) MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "fused qkv matmul: scales must be float32");
  const bool per_tensor = gm == -1 && gn == -1 && gk == -1;
  const bool per_channel = gm == 1 && gn == 1 && gk == -1;
  const bool block = !per_tensor && !per_channel;
  if (block && !(gm == 1 && gn == 128 && gk == 128))
    MAXFP8_FAIL(MAXFP8_ERR_GRANULARITY, "fused qkv matmul: block scaling needs the (1, 128, 128) granularity");
  if (block && ((!x && input_scale_ld < T) || weight_scale_ld < ceil_div(K, 128)))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused qkv matmul: scale leading dimensions too small");
  // the MFMA kernels' layout, and 8-element chunks that stay inside one of Q / K / V and one cache row
  if (!is_aligned(input, 16) || !is_aligned(wqkv, 16) || K % 16 != 0 || K <= 0)
    MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "fused qkv matmul: needs 16-byte aligned rows and K %% 16 == 0");
  if (!offsets_fit(K, K, K, input_scale_ld, block))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused qkv matmul: K = %lld is too long for the kernels' 32-bit tile offsets", (long long)K);
  if (q_dim % 8 != 0 || k_dim % 8 != 0 || !is_aligned(kv_blocks, 16) || (q_dim > 0 && !is_aligned(output, 16)))
    MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "fused qkv matmul: q_dim and kv_heads * head_dim must be multiples of 8, buffers 16-byte aligned");

  GemmArgs p;
  memset(&p, 0, sizeof(p));
  p.a = (const uint8_t*)input;
  p.b = (const uint8_t*)wqkv;
  p.c = output;
  p.a_scales = (const float*)input_scale;
  p.b_scales = (const float*)weight_scale;
  p.M = (int)T; p.N = (int)N; p.K = (int)K;
  p.lda = K; p.ldb = K; p.ldc = q_dim;
  p.a_scales_ld = input_scale_ld;
  p.b_scales_ld = weight_scale_ld;
  p.a_scale_stride = per_tensor ? 0 : 1;
  p.b_scale_stride = per_tensor ? 0 : weight_scale_ld;
  p.c_dtype = MAXFP8_BF16;
  p.scales_dtype = MAXFP8_F32;
  p.c_vec_ok = 1;
  p.c_vec8_ok = 1;
  p.kv_on = 1;
  const int64_t plane = page_size * k_dim;  // one (block, K|V, layer) plane
  uint16_t* blocks = (uint16_t*)kv_blocks;
  p.kv.k_base = blocks + layer_idx * plane;
  p.kv.v_base = kv_dim == 2 ? blocks + (num_layers + layer_idx) * plane : nullptr;
  p.kv.lookup_table = lookup_table;
  p.kv.cache_lengths = cache_lengths;
  p.kv.row_offsets = input_row_offsets;
  p.kv.bias = (const uint16_t*)bias;
  p.kv.block_stride = kv_dim * num_layers * plane;
  p.kv.lut_ld = lut_ld;
  p.kv.num_blocks = num_blocks;
  p.kv.q_dim = (int)q_dim;
  p.kv.k_dim = (int)k_dim;
  p.kv.row_elems = (int)k_dim;
  p.kv.page_size = (int)page_size;
  p.kv.batch = (int)batch_size;
  p.kv.bf16_scaling = block ? 0 : 1;
  hipStream_t st = (hipStream_t)stream;
  if (x) {
    p.a = nullptr;
    p.x = (const uint16_t*)x;
    p.ldx = ldx;
    p.x_scale_ub = scale_ub;
    return gemm_skinny_quant_dispatch(p, block, st);
  }
  const bool automatic = algo == MAXFP8_ALGO_AUTO;
  const Choice choice = !automatic ? Choice{algo, 0} : chosen ? *chosen : choose_qkv(T, N, K, false, block);
  if (automatic) algo = choice.algo;
  if (automatic && algo == kAlgoMid) return gemm_mid_dispatch(p, block, choice.shape, st);
  if (algo == MAXFP8_ALGO_SKINNY) return gemm_skinny_dispatch(p, block, 1, st);
  if (algo != MAXFP8_ALGO_TILED) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "fused qkv matmul: algo %d is not available", algo);
  p.workspace = (float*)workspace;
  return gemm_tiled_dispatch(p, block, workspace_bytes, 1, st);
}

extern "C" {

int maxfp8_fused_qkv_matmul_ragged_paged_scale(void* output, const void* input, const uint32_t* input_row_offsets,
                                               const void* wqkv, const void* input_scale, const void* weight_scale,
                                               void* kv_blocks, const uint32_t* cache_lengths, const uint32_t* lookup_table,
                                               const void* bias, int64_t T, int64_t N, int64_t K, int64_t q_dim,
                                               int64_t batch_size, int64_t num_blocks, int64_t kv_dim, int64_t num_layers,
                                               int64_t layer_idx, int64_t page_size, int64_t num_kv_heads, int64_t head_dim,
                                               int64_t lut_ld, int64_t gm, int64_t gn, int64_t gk, int64_t input_scale_ld,
                                               int64_t weight_scale_ld, int scales_dtype, int algo, void* stream) {
  return qkv_common(output, input, nullptr, 0, 0.f, input_row_offsets, wqkv, input_scale, weight_scale, kv_blocks, cache_lengths, lookup_table,
                    bias, T, N, K, q_dim, batch_size, num_blocks, kv_dim, num_layers, layer_idx, page_size, num_kv_heads, head_dim, lut_ld, gm,
                    gn, gk, input_scale_ld, weight_scale_ld, scales_dtype, algo, nullptr, nullptr, 0, stream);
}

// does the decode kernel quantise by itself?
static bool qkv_in_one(const Choice& choice, int64_t T, int64_t N, int64_t K, bool block) {
  return choice.algo == MAXFP8_ALGO_SKINNY && gemm_skinny_quant_ok(T, N, K, block);
}
// what follows the quantised activations and their scales: the sums of cut tiles
static size_t qkv_partial_bytes(const Choice& choice, int64_t T, int64_t N, int64_t K, bool block) {
  return choice.algo == MAXFP8_ALGO_TILED ? gemm_tiled_qkv_workspace_bytes(T, N, K, block) : 0;
}

size_t maxfp8_fused_qkv_matmul_workspace_bytes(int64_t T, int64_t N, int64_t K, int block_scaling) {
  const bool block = block_scaling != 0;
  return T > 0 && N > 0 && K > 0 ? qkv_partial_bytes(choose_qkv(T, N, K, true, block), T, N, K, block) : 0;
}

int maxfp8_fused_qkv_matmul_ragged_paged_scale_workspace(
    void* output, const void* input, const uint32_t* input_row_offsets, const void* wqkv, const void* input_scale, const void* weight_scale,
    void* kv_blocks, const uint32_t* cache_lengths, const uint32_t* lookup_table, const void* bias, int64_t T, int64_t N, int64_t K,
    int64_t q_dim, int64_t batch_size, int64_t num_blocks, int64_t kv_dim, int64_t num_layers, int64_t layer_idx, int64_t page_size,
    int64_t num_kv_heads, int64_t head_dim, int64_t lut_ld, int64_t gm, int64_t gn, int64_t gk, int64_t input_scale_ld,
    int64_t weight_scale_ld, int scales_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const bool block = !(gk == -1 && gm == gn && (gm == -1 || gm == 1));
  Choice choice = {MAXFP8_ALGO_AUTO, 0};
  size_t need = 0;
  if (T > 0 && N > 0 && K > 0) {
    choice = choose_qkv(T, N, K, true, block);
    need = qkv_partial_bytes(choice, T, N, K, block);
  }
  if (need > 0 && (!workspace || workspace_bytes < need))
    MAXFP8_FAIL(MAXFP8_ERR_WORKSPACE, "fused qkv matmul: needs %zu bytes of workspace, got %zu", need, workspace ? workspace_bytes : (size_t)0);
  if (need > 0 && !is_aligned(workspace, 16)) MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "fused qkv matmul: workspace must be 16-byte aligned");
  return qkv_common(output, input, nullptr, 0, 0.f, input_row_offsets, wqkv, input_scale, weight_scale, kv_blocks, cache_lengths, lookup_table,
                    bias, T, N, K, q_dim, batch_size, num_blocks, kv_dim, num_layers, layer_idx, page_size, num_kv_heads, head_dim, lut_ld, gm,
                    gn, gk, input_scale_ld, weight_scale_ld, scales_dtype, MAXFP8_ALGO_AUTO, &choice, need ? workspace : nullptr, need, stream);
}

size_t maxfp8_linear_qkv_workspace_bytes(int64_t T, int64_t N, int64_t K, int weight_granularity) {
  if (T <= 0 || N <= 0 || K <= 0) return 0;
  const bool block = weight_granularity == MAXFP8_GRAN_BLOCK;
  const Choice choice = choose_qkv(T, N, K, true, block);
  return qkv_in_one(choice, T, N, K, block) ? 0 : linear_layout(T, N, K, block, false, false).partial + qkv_partial_bytes(choice, T, N, K, block);
}

int maxfp8_linear_qkv_ragged_paged_scale(void* output, const void* x, int64_t x_row_stride, const uint32_t* input_row_offsets,
                                         const void* wqkv, const void* weight_scale, void* kv_blocks, const uint32_t* cache_lengths,
                                         const uint32_t* lookup_table, const void* bias, int64_t T, int64_t N, int64_t K, int64_t q_dim,
                                         int64_t batch_size, int64_t num_blocks, int64_t kv_dim, int64_t num_layers, int64_t layer_idx,
                                         int64_t page_size, int64_t num_kv_heads, int64_t head_dim, int64_t lut_ld, int weight_granularity,
                                         int64_t weight_scale_ld, float scale_ub, void* workspace, size_t workspace_bytes, void* stream) {
  if (weight_granularity != MAXFP8_GRAN_BLOCK && weight_granularity != MAXFP8_GRAN_ROWWISE)
    MAXFP8_FAIL(MAXFP8_ERR_GRANULARITY, "qkv linear: weight granularity %d is not block or rowwise", weight_granularity);
  const bool block = weight_granularity == MAXFP8_GRAN_BLOCK;
  const int64_t gm = 1, gn = block ? 128 : 1, gk = block ? 128 : -1;
  if (T < 0 || N < 0 || K < 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "qkv linear: negative size");
  if (batch_size == 0 || T == 0 || N == 0) return MAXFP8_OK;
  if (!x) MAXFP8_FAIL(MAXFP8_ERR_NULL, "qkv linear: null pointer");
  if (x_row_stride < K || K <= 0 || K % (block ? 128 : 16) != 0) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "qkv linear: K = %lld does not suit the scaling", (long long)K);
  const Choice choice = choose_qkv(T, N, K, true, block);
  if (qkv_in_one(choice, T, N, K, block) && is_aligned(x, 16) && x_row_stride % 8 == 0 && 32 * x_row_stride < ((int64_t)1 << 31))
    return qkv_common(output, nullptr, x, x_row_stride, scale_ub, input_row_offsets, wqkv, nullptr, weight_scale, kv_blocks, cache_lengths,
                      lookup_table, bias, T, N, K, q_dim, batch_size, num_blocks, kv_dim, num_layers, layer_idx, page_size, num_kv_heads,
                      head_dim, lut_ld, gm, gn, gk, 0, weight_scale_ld, MAXFP8_F32, MAXFP8_ALGO_SKINNY, nullptr, nullptr, 0, stream);
  const LinearLayout l = linear_layout(T, N, K, block, false, false);
  const size_t partial = qkv_partial_bytes(choice, T, N, K, block), total = l.partial + partial;
  if (!workspace || workspace_bytes < total)
    MAXFP8_FAIL(MAXFP8_ERR_WORKSPACE, "qkv linear: needs %zu bytes of workspace, got %zu", total, workspace ? workspace_bytes : (size_t)0);
  if (!is_aligned(workspace, 16)) MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "qkv linear: workspace must be 16-byte aligned");
  uint8_t* q = (uint8_t*)workspace;
  float* scales = (float*)(q + l.scales);
  const int rc = quantize_dispatch(q, scales, x, T, K, x_row_stride, K, block ? 128 : K, l.scales_ld, MAXFP8_BF16, MAXFP8_F32, scale_ub, 1, 0, 0, 0,
                                   nullptr, 1, (hipStream_t)stream);
  if (rc != MAXFP8_OK) return rc;
  return qkv_common(output, q, nullptr, 0, 0.f, input_row_offsets, wqkv, scales, weight_scale, kv_blocks, cache_lengths, lookup_table, bias, T, N,
                    K, q_dim, batch_size, num_blocks, kv_dim, num_layers, layer_idx, page_size, num_kv_heads, head_dim, lut_ld, gm, gn, gk,
                    block ? l.scales_ld : T, weight_scale_ld, MAXFP8_F32, MAXFP8_ALGO_AUTO, &choice, partial ? q + l.partial : nullptr, partial, stream);
}

}  // extern "C"

static int grouped_block_common(void* c, const uint32_t* c_row_index, const void* a, const void* b, const void* a_scales,
                                const void* b_scales, const uint32_t* expert_start_indices, const int32_t* expert_ids,
                                int64_t T, int64_t N, int64_t K, int64_t num_experts, int64_t max_num_tokens_per_expert,
                                int64_t num_active_experts, int64_t a_scales_ld, int c_dtype, int scales_dtype, int algo,
                                void* stream) {
  if (c_dtype != MAXFP8_BF16 && c_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "grouped matmul: output dtype %d is not bf16 or f32", c_dtype);
  if (scales_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "grouped matmul: scales must be float32");
  if (T < 0 || N < 0 || K < 0 || num_experts < 0 || max_num_tokens_per_expert < 0 || num_active_experts < 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped matmul: negative size");
  // grouped_matmul_sm100_blockwise_fp8.mojo:3016-3017
  if (max_num_tokens_per_expert == 0 || num_active_experts == 0 || T == 0 || N == 0) return MAXFP8_OK;
  if (num_active_experts > num_experts)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped matmul: %lld active slots but expert_ids holds %lld", (long long)num_active_experts,
                (long long)num_experts);
  if (T >= ((int64_t)1 << 31) || N >= ((int64_t)1 << 31) || K >= ((int64_t)1 << 31))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped matmul: sizes must fit 31 bits");
  if (a_scales_ld < T) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped matmul: a_scales leading dimension %lld < T = %lld",
                                   (long long)a_scales_ld, (long long)T);
  if (!c || !a || !b || !a_scales || !b_scales || !expert_start_indices || !expert_ids)
    MAXFP8_FAIL(MAXFP8_ERR_NULL, "grouped matmul: null pointer");
  hipStream_t st = (hipStream_t)stream;
  const bool fast_layout = is_aligned(a, 16) && is_aligned(b, 16) && K % 16 == 0 && K > 0 && offsets_fit(K, K, K, a_scales_ld, true);
  if (algo == MAXFP8_ALGO_AUTO) algo = fast_layout ? MAXFP8_ALGO_TILED : MAXFP8_ALGO_NAIVE;
  if (algo == MAXFP8_ALGO_NAIVE && c_row_index)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped matmul: the row scatter needs the MFMA kernel (16-byte aligned rows, K %% 16 == 0)");
  if (algo == MAXFP8_ALGO_NAIVE)
    return naive_grouped_dispatch(c, a, b, a_scales, b_scales, expert_start_indices, expert_ids, T, N, K,
                                  max_num_tokens_per_expert, num_active_experts, a_scales_ld, c_dtype, st);
  if (algo != MAXFP8_ALGO_TILED) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped matmul: unknown algo %d", algo);
  if (!fast_layout) MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "grouped matmul: the MFMA kernel needs 16-byte aligned rows and K %% 16 == 0");

  GemmArgs p;
  memset(&p, 0, sizeof(p));
  p.a = (const uint8_t*)a;
  p.b = (const uint8_t*)b;
  p.c = c;
  p.a_scales = (const float*)a_scales;
  p.b_scales = (const float*)b_scales;
  p.M = (int)T; p.N = (int)N; p.K = (int)K;
  p.lda = K; p.ldb = K; p.ldc = N;
  p.a_scales_ld = a_scales_ld;
  p.b_scales_ld = ceil_div(K, 128);
  p.c_dtype = c_dtype;
  p.scales_dtype = MAXFP8_F32;
  p.c_vec_ok = (N % 4 == 0) && is_aligned(c, c_dtype == MAXFP8_BF16 ? 8 : 16);
  p.c_vec8_ok = (N % 8 == 0) && is_aligned(c, 16);
  p.offsets = expert_start_indices;
  p.expert_ids = expert_ids;
  p.num_active = (int)num_active_experts;
  p.b_expert_stride = N * K;
  p.bs_expert_stride = ceil_div(N, 128) * ceil_div(K, 128);
  p.c_row_index = c_row_index;
  return gemm_grouped_dispatch(p, true, T, max_num_tokens_per_expert, st);
}

extern "C" {

int maxfp8_grouped_matmul_dynamic_scaled_fp8(void* c, const void* a, const void* b, const void* a_scales,
                                             const void* b_scales, const uint32_t* expert_start_indices,
                                             const int32_t* expert_ids, int64_t T, int64_t N, int64_t K,
                                             int64_t num_experts, int64_t max_num_tokens_per_expert,
                                             int64_t num_active_experts, int64_t a_scales_ld, int c_dtype,
                                             int scales_dtype, int algo, void* stream) {
  return grouped_block_common(c, nullptr, a, b, a_scales, b_scales, expert_start_indices, expert_ids, T, N, K, num_experts,
                              max_num_tokens_per_expert, num_active_experts, a_scales_ld, c_dtype, scales_dtype, algo, stream);
}

int maxfp8_grouped_matmul_dynamic_scaled_fp8_scatter(void* c, const uint32_t* c_row_index, const void* a, const void* b,
                                                     const void* a_scales, const void* b_scales,
                                                     const uint32_t* expert_start_indices, const int32_t* expert_ids,
                                                     int64_t T, int64_t N, int64_t K, int64_t num_experts,
                                                     int64_t max_num_tokens_per_expert, int64_t num_active_experts,
                                                     int64_t a_scales_ld, int c_dtype, int scales_dtype, int algo,
                                                     void* stream) {
  if (T > 0 && N > 0 && !c_row_index) MAXFP8_FAIL(MAXFP8_ERR_NULL, "grouped matmul (scatter): null row index");
  return grouped_block_common(c, c_row_index, a, b, a_scales, b_scales, expert_start_indices, expert_ids, T, N, K, num_experts,
                              max_num_tokens_per_expert, num_active_experts, a_scales_ld, c_dtype, scales_dtype, algo, stream);
}

int maxfp8_grouped_matmul_rowwise_dynamic_scaled_fp8(void* c, const void* a, const void* b, const void* a_scales,
                                                     const void* b_scales, const uint32_t* expert_start_indices,
                                                     const int32_t* expert_ids, int64_t T, int64_t N, int64_t K,
                                                     int64_t num_experts, int64_t max_num_tokens_per_expert,
                                                     int64_t num_active_experts, int c_dtype, int scales_dtype, void* stream) {
  if (c_dtype != MAXFP8_BF16 && c_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "grouped rowwise matmul: output dtype %d is not bf16 or f32", c_dtype);
  if (scales_dtype != MAXFP8_F32)
    MAXFP8_FAIL(MAXFP8_ERR_DTYPE, "grouped rowwise matmul: A and B scales must be float32 for rowwise/per-token granularity");
  if (T < 0 || N < 0 || K < 0 || num_experts < 0 || max_num_tokens_per_expert < 0 || num_active_experts < 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped rowwise matmul: negative size");
  // grouped_matmul.mojo:1675-1676
  if (max_num_tokens_per_expert == 0 || num_active_experts == 0 || T == 0 || N == 0) return MAXFP8_OK;
  if (num_active_experts > num_experts)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped rowwise matmul: %lld active slots but expert_ids holds %lld",
                (long long)num_active_experts, (long long)num_experts);
  if (T >= ((int64_t)1 << 31) || N >= ((int64_t)1 << 31) || K >= ((int64_t)1 << 31))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped rowwise matmul: sizes must fit 31 bits");
  if (!c || !a || !b || !a_scales || !b_scales || !expert_start_indices || !expert_ids)
    MAXFP8_FAIL(MAXFP8_ERR_NULL, "grouped rowwise matmul: null pointer");
  if (!(is_aligned(a, 16) && is_aligned(b, 16) && K % 16 == 0 && K > 0))
    MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "grouped rowwise matmul: needs 16-byte aligned rows and K %% 16 == 0");
  if (!offsets_fit(K, K, K, 0, false))
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "grouped rowwise matmul: K = %lld is too long for the kernels' 32-bit tile offsets", (long long)K);
  GemmArgs p;
  memset(&p, 0, sizeof(p));
  p.a = (const uint8_t*)a;
  p.b = (const uint8_t*)b;
  p.c = c;
  p.a_scales = (const float*)a_scales;  // [T, 1]
  p.b_scales = (const float*)b_scales;  // [E, N, 1]
  p.M = (int)T; p.N = (int)N; p.K = (int)K;
  p.lda = K; p.ldb = K; p.ldc = N;
  p.a_scale_stride = 1;
  p.b_scale_stride = 1;
  p.c_dtype = c_dtype;
  p.scales_dtype = MAXFP8_F32;
  p.c_vec_ok = (N % 4 == 0) && is_aligned(c, c_dtype == MAXFP8_BF16 ? 8 : 16);
  p.c_vec8_ok = (N % 8 == 0) && is_aligned(c, 16);
  p.offsets = expert_start_indices;
  p.expert_ids = expert_ids;
  p.num_active = (int)num_active_experts;
  p.b_expert_stride = N * K;
  p.bs_expert_stride = N;
  return gemm_grouped_dispatch(p, false, T, max_num_tokens_per_expert, (hipStream_t)stream);
}

int maxfp8_cast_f32_to_e4m3fn(void* out_fp8, const float* in, int64_t n, void* stream) {
  if (n <= 0) return MAXFP8_OK;
  if (!out_fp8 || !in) MAXFP8_FAIL(MAXFP8_ERR_NULL, "cast: null pointer");
  return cast_f32_to_e4m3fn_dispatch(out_fp8, in, n, (hipStream_t)stream);
}

int maxfp8_cast_e4m3fn_to_f32(float* out, const void* in_fp8, int64_t n, void* stream) {
  if (n <= 0) return MAXFP8_OK;
  if (!out || !in_fp8) MAXFP8_FAIL(MAXFP8_ERR_NULL, "cast: null pointer");
  return cast_e4m3fn_to_f32_dispatch(out, in_fp8, n, (hipStream_t)stream);
}

int maxfp8_cast_f32_to_bf16(void* out_bf16, const float* in, int64_t n, void* stream) {
  if (n <= 0) return MAXFP8_OK;
  if (!out_bf16 || !in) MAXFP8_FAIL(MAXFP8_ERR_NULL, "cast: null pointer");
  return cast_f32_to_bf16_dispatch(out_bf16, in, n, (hipStream_t)stream);
}

int maxfp8_copy_bytes(void* dst, const void* src, int64_t n, void* stream) {
  if (n <= 0) return MAXFP8_OK;
  if (!dst || !src) MAXFP8_FAIL(MAXFP8_ERR_NULL, "copy: null pointer");
  if (n % 16 != 0 || !is_aligned(dst, 16) || !is_aligned(src, 16))
    MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "copy: size and pointers must be multiples of 16 bytes");
  return copy_bytes_dispatch(dst, src, n, (hipStream_t)stream);
}

int maxfp8_decode_weight_read_probe(const void* b, int64_t M, int64_t N, int64_t K, int64_t ldb, void* stream) {
  if (!b) MAXFP8_FAIL(MAXFP8_ERR_NULL, "read probe: null pointer");
  if (M <= 0 || M > 16 || N <= 0 || K <= 0 || ldb < K)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "read probe: needs 1 <= M <= 16, N > 0, 0 < K <= ldb (got M %lld, N %lld, K %lld, ldb %lld)",
                (long long)M, (long long)N, (long long)K, (long long)ldb);
  if (!is_aligned(b, 16) || K % 16 != 0 || ldb % 16 != 0) MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "read probe: needs 16-byte aligned rows and K %% 16 == 0");
  if (!offsets_fit(K, ldb, ldb, 0, false)) MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "read probe: rows too long for 32-bit tile offsets");
  return gemm_skinny_read_probe(b, M, N, K, ldb, (hipStream_t)stream);
}

long long maxfp8_handovers_given_up(void) {
  unsigned int pieces = 0, shares = 0;
  int rc = gemm_w4_gave_up(&pieces);
  if (rc == MAXFP8_OK) rc = gemm_streamk_gave_up(&shares);
  return rc == MAXFP8_OK ? (long long)pieces + (long long)shares : (long long)rc;
}

int maxfp8_mfma_issue_probe(int kernel, int blockscale, int level, int64_t slabs, const void* a, const void* b, const float* a_scales,
                            const float* b_scales, void* c, uint64_t* clocks, void* stream) {
  if (!a || !b || !c || !a_scales || !b_scales) MAXFP8_FAIL(MAXFP8_ERR_NULL, "issue probe: null pointer");
  if (clocks && !is_aligned(clocks, 8)) MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "issue probe: clocks must be 8-byte aligned");
  if ((kernel != 0 && kernel != 4 && kernel != 5 && kernel != 6) || (level != 1 && level != 2) || slabs < 8 || slabs > (1 << 22) || slabs % 2 != 0)
    MAXFP8_FAIL(MAXFP8_ERR_SHAPE, "issue probe: kernel 0 / 4 / 5 / 6, level 1 / 2, an even number of slabs in [8, 2^22]");
  if (!is_aligned(a, 16) || !is_aligned(b, 16) || !is_aligned(c, 16)) MAXFP8_FAIL(MAXFP8_ERR_ALIGN, "issue probe: 16-byte aligned buffers");
  GemmArgs p;
  memset(&p, 0, sizeof(p));
  p.a = (const uint8_t*)a;
  p.b = (const uint8_t*)b;
  p.c = c;
  p.a_scales = a_scales;
  p.b_scales = b_scales;
  p.M = 256; p.N = 256; p.K = (int)(slabs * 128);
  p.lda = 1024; p.ldb = 1024; p.ldc = 256;
  p.a_scales_ld = 256; p.b_scales_ld = 8;
  p.a_scale_stride = 0; p.b_scale_stride = 0;  // (row mode: element 0 of each scale vector, in the epilogue)
  p.c_dtype = MAXFP8_BF16;
  p.scales_dtype = MAXFP8_F32;
  p.c_vec_ok = 1; p.c_vec8_ok = 1;
  p.splits = 1;
  p.workspace = reinterpret_cast<float*>(clocks);
  return kernel == 0 ? gemm_persist_probe(p, blockscale != 0, level, (hipStream_t)stream) : gemm_w4_probe(p, blockscale != 0, level, kernel, (hipStream_t)stream);
}

}  // extern "C"
