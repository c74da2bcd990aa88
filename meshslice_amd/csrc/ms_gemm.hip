// libmeshslice_hip.so — C ABI over the gfx950 GEMM kernels (declarations: include/meshslice_hip.h).
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "ms_common.hip.inc"

#include "ms_gemm_bf16.hip.inc"
#include "ms_gemm_bf16_big.hip.inc"
#include "ms_gemm_bf16_x16.hip.inc"
#include "ms_gemm_f32.hip.inc"
#include "ms_gemm_f32_waves.hip.inc"

// Every kernel variant is instantiated explicitly: with implicit instantiation alone the host
// compiler leaves some of the launch stubs undefined.
#define MS_INSTANTIATE_RING(BM, BN, BK, NS, WGM, WGN)                                                                         \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, true, false, true, false>(const msk::GemmArgs);   \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, true, false, false, false>(const msk::GemmArgs);  \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, true, false, true, true>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, true, false, false, true>(const msk::GemmArgs);   \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, true, true, false, false>(const msk::GemmArgs);   \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, true, true, true, false>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, false, false, false, false>(const msk::GemmArgs); \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, false, false, true, false>(const msk::GemmArgs);
// output-stationary products with their contraction split (all but the four-wave 256x256 tile)
#define MS_INSTANTIATE_RING_SPLIT(BM, BN, BK, NS, WGM, WGN)                                                                                \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, true, false, true, false, false, true>(const msk::GemmArgs); \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, NS, WGM, WGN, true, false, false, false, false, true>(const msk::GemmArgs);
MS_INSTANTIATE_RING_SPLIT(192, 192, 64, 3, 2, 2)
MS_INSTANTIATE_RING_SPLIT(128, 128, 64, 2, 2, 2)
MS_INSTANTIATE_RING_SPLIT(128, 192, 64, 3, 2, 2)
MS_INSTANTIATE_RING_SPLIT(256, 192, 32, 4, 2, 2)
MS_INSTANTIATE_RING_SPLIT(192, 256, 32, 4, 2, 2)
MS_INSTANTIATE_RING_SPLIT(256, 256, 64, 2, 2, 4)
MS_INSTANTIATE_RING_SPLIT(256, 192, 64, 2, 2, 2)
MS_INSTANTIATE_RING_SPLIT(192, 256, 64, 2, 2, 2)
MS_INSTANTIATE_RING_SPLIT(128, 128, 64, 3, 2, 2)
MS_INSTANTIATE_RING_SPLIT(64, 64, 128, 3, 2, 2)
MS_INSTANTIATE_RING_SPLIT(64, 128, 64, 3, 2, 2)
#undef MS_INSTANTIATE_RING_SPLIT
// and those with a fused epilogue too
#define MS_INSTANTIATE_FUSED_SPLIT(BM, BN, BK)                                                                                        \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, 3, 2, 2, true, false, true, true, false, true>(const msk::GemmArgs); \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, BK, 3, 2, 2, true, false, false, true, false, true>(const msk::GemmArgs);
MS_INSTANTIATE_FUSED_SPLIT(64, 64, 128)
MS_INSTANTIATE_FUSED_SPLIT(128, 128, 64)
#undef MS_INSTANTIATE_FUSED_SPLIT
MS_INSTANTIATE_RING(256, 256, 64, 2, 2, 2)
MS_INSTANTIATE_RING(192, 192, 64, 3, 2, 2)
MS_INSTANTIATE_RING(128, 128, 64, 2, 2, 2)
MS_INSTANTIATE_RING(128, 192, 64, 3, 2, 2)
MS_INSTANTIATE_RING(64, 64, 128, 3, 2, 2)
MS_INSTANTIATE_RING(64, 128, 64, 3, 2, 2)
MS_INSTANTIATE_RING(256, 192, 32, 4, 2, 2)
MS_INSTANTIATE_RING(192, 256, 32, 4, 2, 2)
MS_INSTANTIATE_RING(256, 256, 64, 2, 2, 4)
MS_INSTANTIATE_RING(256, 192, 64, 2, 2, 2)
MS_INSTANTIATE_RING(192, 256, 64, 2, 2, 2)
MS_INSTANTIATE_RING(128, 128, 64, 3, 2, 2)
#undef MS_INSTANTIATE_RING
// several devices' partial sums in one product (Problem::sum): the tiles on three stages, whose waves have room for the totals
#define MS_INSTANTIATE_SUM(BM, BN)                                                                                           \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, 64, 3, 2, 2, true, true, true, false, true>(const msk::GemmArgs); \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, 64, 3, 2, 2, false, false, true, false, true>(const msk::GemmArgs); \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, 64, 3, 2, 2, true, true, true, false, true, true>(const msk::GemmArgs); \
  template __global__ void msk::gemm_bf16_ring_kernel<BM, BN, 64, 3, 2, 2, false, false, true, false, true, true>(const msk::GemmArgs);
MS_INSTANTIATE_SUM(128, 128)
MS_INSTANTIATE_SUM(128, 192)
MS_INSTANTIATE_SUM(192, 192)
#undef MS_INSTANTIATE_SUM
// operands whose rows along the contraction are too far apart for the other kernels' offsets (Operand's FAR, reaches): one tile of each type
#define MS_INSTANTIATE_FAR(AK, OBF, EPI, FOLD) \
  template __global__ void msk::gemm_bf16_ring_kernel<128, 128, 64, 3, 2, 2, AK, false, OBF, EPI, FOLD, false, true>(const msk::GemmArgs);
MS_INSTANTIATE_FAR(true, true, false, false)
MS_INSTANTIATE_FAR(true, false, false, false)
MS_INSTANTIATE_FAR(true, true, true, false)
MS_INSTANTIATE_FAR(true, false, true, false)
MS_INSTANTIATE_FAR(false, true, false, false)
MS_INSTANTIATE_FAR(false, false, false, false)
MS_INSTANTIATE_FAR(false, true, false, true)
#undef MS_INSTANTIATE_FAR
template __global__ void msk::gemm_f32_tile_kernel<2, 2, 1, 1, true, false, true, false, true>(const msk::GemmArgs);
template __global__ void msk::gemm_f32_tile_kernel<2, 2, 1, 1, true, false, false, false, true>(const msk::GemmArgs);
template __global__ void msk::gemm_f32_tile_kernel<2, 2, 1, 1, false, false, true, false, true>(const msk::GemmArgs);
template __global__ void msk::gemm_f32_tile_kernel<2, 2, 1, 1, false, false, false, false, true>(const msk::GemmArgs);
#define MS_INSTANTIATE_BIG(TM, TN)                                                                             \
  template __global__ void msk::gemm_bf16_big_kernel<TM, TN, true, false, true, false>(const msk::GemmArgs);   \
  template __global__ void msk::gemm_bf16_big_kernel<TM, TN, true, false, false, false>(const msk::GemmArgs);  \
  template __global__ void msk::gemm_bf16_big_kernel<TM, TN, true, false, true, true>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_bf16_big_kernel<TM, TN, true, false, false, true>(const msk::GemmArgs);   \
  template __global__ void msk::gemm_bf16_big_kernel<TM, TN, true, true, false, false>(const msk::GemmArgs);   \
  template __global__ void msk::gemm_bf16_big_kernel<TM, TN, true, true, true, false>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_bf16_big_kernel<TM, TN, false, false, false, false>(const msk::GemmArgs); \
  template __global__ void msk::gemm_bf16_big_kernel<TM, TN, false, false, true, false>(const msk::GemmArgs);
MS_INSTANTIATE_BIG(4, 6)
MS_INSTANTIATE_BIG(6, 3)
#undef MS_INSTANTIATE_BIG
#define MS_INSTANTIATE_X16(BN)                                                                                  \
  template __global__ void msk::gemm_bf16_x16_kernel<true, false, true, false, 0, BN>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_bf16_x16_kernel<true, false, false, false, 0, BN>(const msk::GemmArgs);   \
  template __global__ void msk::gemm_bf16_x16_kernel<true, false, true, true, 0, BN>(const msk::GemmArgs);     \
  template __global__ void msk::gemm_bf16_x16_kernel<true, false, false, true, 0, BN>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_bf16_x16_kernel<true, true, false, false, 0, BN>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_bf16_x16_kernel<true, true, true, false, 0, BN>(const msk::GemmArgs);     \
  template __global__ void msk::gemm_bf16_x16_kernel<false, false, false, false, 0, BN>(const msk::GemmArgs);  \
  template __global__ void msk::gemm_bf16_x16_kernel<false, false, true, false, 0, BN>(const msk::GemmArgs);
MS_INSTANTIATE_X16(384)
MS_INSTANTIATE_X16(256)
#undef MS_INSTANTIATE_X16
#define MS_INSTANTIATE_F32(WGM, WGN, TM, TN)                                                                          \
  template __global__ void msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, true>(const msk::GemmArgs);     \
  template __global__ void msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, false>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, true, true>(const msk::GemmArgs);  \
  template __global__ void msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, false, true>(const msk::GemmArgs); \
  template __global__ void msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, true, true>(const msk::GemmArgs);      \
  template __global__ void msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, true, false>(const msk::GemmArgs);     \
  template __global__ void msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, false, false, true>(const msk::GemmArgs);    \
  template __global__ void msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, false, false, false>(const msk::GemmArgs);
MS_INSTANTIATE_F32(4, 2, 2, 2)
MS_INSTANTIATE_F32(4, 2, 1, 3)
MS_INSTANTIATE_F32(2, 2, 2, 2)
MS_INSTANTIATE_F32(2, 2, 1, 1)
MS_INSTANTIATE_F32(2, 2, 3, 3)
MS_INSTANTIATE_F32(2, 2, 1, 3)
MS_INSTANTIATE_F32(2, 2, 1, 2)
#undef MS_INSTANTIATE_F32
template __global__ void msk::gemm_f32_waves_kernel<true, false, true>(const msk::GemmArgs);
template __global__ void msk::gemm_f32_waves_kernel<true, false, false>(const msk::GemmArgs);
template __global__ void msk::gemm_f32_waves_kernel<true, true, true>(const msk::GemmArgs);
template __global__ void msk::gemm_f32_waves_kernel<true, true, false>(const msk::GemmArgs);
template __global__ void msk::gemm_f32_waves_kernel<false, false, true>(const msk::GemmArgs);
template __global__ void msk::gemm_f32_waves_kernel<false, false, false>(const msk::GemmArgs);

namespace {
thread_local char g_err[512] = "";
}

int msi::fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

namespace {

thread_local int g_variant = 0;
thread_local int g_splits = 0;    // forced split count of the contraction (0 = library default)
thread_local int g_launches = 0;   // kernels launched by the last GEMM call of this thread
thread_local int g_last_variant = 0;   // kernel variant of that call's first launch (bf16 tiles 1..VARIANTS, fp32 tiles F32_FIRST..F32_WAVES)
thread_local int g_last_splits = 1;    // and the number of ways it split the contraction
thread_local int g_last_grid = 0;      // and its workgroup count
thread_local int g_reserved_cus = 0;   // compute units the GEMM launches of this thread leave free (ms_set_reserved_cus)
thread_local int g_last_tiles_per_chunk = 0;   // output tiles per chunk (per output, for OS) of that call's last launch

using msi::fail;

struct DevFacts {
  int cus = 0, clock_khz = 0, gfx950 = 0, lds = 0;
};
struct DevInfo : DevFacts {
  std::once_flag once;
  hipError_t err = hipSuccess;
};
DevInfo g_dev[64];

// Facts about the calling thread's current device, read from the runtime once per ordinal (call_once: concurrent
// first calls from several host threads wait for the one that fills the entry).
int dev_info(DevInfo **out) {
  int d = 0;
  MS_HIP(hipGetDevice(&d));
  if (d < 0 || d >= 64) return fail(MS_ERR_HIP, "device ordinal %d out of range", d);
  DevInfo &di = g_dev[d];
  std::call_once(di.once, [&di, d]() {
    hipDeviceProp_t p;
    di.err = hipGetDeviceProperties(&p, d);
    if (di.err != hipSuccess) return;
    di.cus = p.multiProcessorCount;
    di.clock_khz = p.clockRate;
    di.gfx950 = strncmp(p.gcnArchName, "gfx950", 6) == 0;
    di.lds = (int)p.sharedMemPerBlock;
  });
  if (di.err != hipSuccess) return fail(MS_ERR_HIP, "hipGetDeviceProperties failed: %s", hipGetErrorString(di.err));
  *out = &di;
  return MS_OK;
}

enum Flow { OS = 0, LS = 1, RS = 2 };

// One local contraction, in kernel terms.
struct Problem {
  Flow flow;
  const void *const *a;  // nkslices (OS), nchunks (the operand cut into chunks, and both in several devices' calls) or 1 pointers
  const void *const *b;
  void *const *c;
  int na, nb, nc;
  int S;
  int M, N, K;           // per-chunk rows/cols, per-slice contraction
  int lda, ldb, ldc;
  int b_blk = 0;         // OS, LS: bytes from one block of eight rows of a B slice to its next (0: they follow each other)
  int in_dtype, out_dtype;
  // LS / RS: C = sum over the S entries of both tables, each entry's partial sum by itself, added up in fp32 in their order
  bool sum = false;
  // fused OS epilogue (all zero / null = plain product)
  int act = 0;
  const void *res = nullptr;
  int ldr = 0;
  float *row_sum = nullptr;
  float *row_sumsq = nullptr;
  // workspace for split contractions (null / 0: none, the contraction is never split)
  void *ws = nullptr;
  size_t ws_bytes = 0;
  // LS / RS: per-chunk completion counters (null: none)
  unsigned *chunk_done = nullptr;
  // OS: per-slice input gate (null: none) and the longest wait for one slice, in ticks of the 100 MHz wall clock
  unsigned *slice_ready = nullptr;
  unsigned long long gate_ticks = 0;
};

// Layout of a split-contraction workspace: SPLIT_MAX_BANDS words of arrival counts per output tile, then one fp32 partial tile
// per work item.
constexpr size_t WS_HEADER_BYTES = 4096;
constexpr int WS_COUNTERS = (int)(WS_HEADER_BYTES / sizeof(int));
constexpr int WS_MAX_TILES = WS_COUNTERS / msk::SPLIT_MAX_BANDS;     // output tiles of a split product

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int validate(const Problem &p) {
  static const char *names[] = {"ms_gemm_os", "ms_gemm_ls", "ms_gemm_rs"};
  const char *fn = names[p.flow];
  if (p.S < 1 || p.S > MS_MAX_SLICES) return fail(MS_ERR_ARG, "%s: S = %d outside [1, %d]", fn, p.S, MS_MAX_SLICES);
  if (p.M <= 0 || p.N <= 0 || p.K <= 0) return fail(MS_ERR_ARG, "%s: non-positive extent (m=%d n=%d k=%d)", fn, p.M, p.N, p.K);
  if (p.in_dtype != MS_DTYPE_F32 && p.in_dtype != MS_DTYPE_BF16) return fail(MS_ERR_UNSUPPORTED, "%s: unknown in_dtype %d", fn, p.in_dtype);
  if (p.out_dtype != MS_DTYPE_F32 && p.out_dtype != MS_DTYPE_BF16) return fail(MS_ERR_UNSUPPORTED, "%s: unknown out_dtype %d", fn, p.out_dtype);
  if (!p.a || !p.b || !p.c) return fail(MS_ERR_ARG, "%s: null pointer table", fn);
  const int q = p.in_dtype == MS_DTYPE_BF16 ? 8 : 4;  // elements per 16 bytes
  // contiguous extent of each operand, and minimum leading dimension
  const int a_cont = p.flow == RS ? p.M : p.K;
  const int b_cont = p.flow == LS ? p.K : p.N;
  if (a_cont % q || b_cont % q) return fail(MS_ERR_ARG, "%s: contiguous extents (%d, %d) must be multiples of %d", fn, a_cont, b_cont, q);
  if (p.lda < a_cont || p.ldb < b_cont || p.ldc < p.N) return fail(MS_ERR_ARG, "%s: leading dimension smaller than the row length", fn);
  if (p.lda % q || p.ldb % q) return fail(MS_ERR_ARG, "%s: operand leading dimensions must be multiples of %d", fn, q);
  {
    // the kernels address an operand slice with 32-bit byte offsets, the upper half reserved for "out of range"
    const long long a_rows = p.flow == RS ? p.K : p.M, b_rows = p.flow == LS ? p.N : p.K;
    const long long es = p.in_dtype == MS_DTYPE_BF16 ? 2 : 4;
    if (a_rows * p.lda * es > 0x7FFFFFFFLL || b_rows * p.ldb * es > 0x7FFFFFFFLL)
      return fail(MS_ERR_UNSUPPORTED, "%s: an operand slice spans 2 GiB or more", fn);
  }
  const int qo = p.out_dtype == MS_DTYPE_BF16 ? 8 : 4;
  if (p.N % qo || p.ldc % qo) return fail(MS_ERR_ARG, "%s: output columns / leading dimension must be multiples of %d", fn, qo);
  if (p.act != MS_ACT_NONE && p.act != MS_ACT_GELU) return fail(MS_ERR_ARG, "%s: unknown activation %d", fn, p.act);
  if (p.res) {
    if (!aligned16(p.res)) return fail(MS_ERR_ARG, "%s: residual pointer not 16-byte aligned", fn);
    if (p.ldr < p.N || p.ldr % qo) return fail(MS_ERR_ARG, "%s: residual leading dimension %d must be >= n and a multiple of %d", fn, p.ldr, qo);
  }
  if (p.ws && ((reinterpret_cast<uintptr_t>(p.ws) & 255) || p.ws_bytes < WS_HEADER_BYTES))
    return fail(MS_ERR_ARG, "%s: a workspace must be 256-byte aligned and hold at least %zu bytes", fn, WS_HEADER_BYTES);
  if ((reinterpret_cast<uintptr_t>(p.row_sum) | reinterpret_cast<uintptr_t>(p.row_sumsq)) & 3) return fail(MS_ERR_ARG, "%s: row-moment pointers must be 4-byte aligned", fn);
  if ((p.act || p.res || p.row_sum || p.row_sumsq) && (p.flow != OS || p.in_dtype != MS_DTYPE_BF16))
    return fail(MS_ERR_UNSUPPORTED, "%s: the fused epilogue exists for the output-stationary bf16 kernel only", fn);
  for (int i = 0; i < p.na; i++) if (!p.a[i] || !aligned16(p.a[i])) return fail(MS_ERR_ARG, "%s: operand pointer %d null or not 16-byte aligned", fn, i);
  for (int i = 0; i < p.nb; i++) if (!p.b[i] || !aligned16(p.b[i])) return fail(MS_ERR_ARG, "%s: operand pointer %d null or not 16-byte aligned", fn, i);
  for (int i = 0; i < p.nc; i++) if (!p.c[i] || !aligned16(p.c[i])) return fail(MS_ERR_ARG, "%s: output pointer %d null or not 16-byte aligned", fn, i);
  return MS_OK;
}

// KIND 0: gemm_bf16_ring_kernel<BM, BN, ...>; 1: gemm_bf16_big_kernel (32x32x16 MFMA, 2x2 waves, two 64-deep stages);
// 2: gemm_bf16_x16_kernel (256x384x64 or 256x256x64 on the 16x16x32 MFMA)
template <int KIND, int BM, int BN, int BK_, int NS, int WGM, int WGN, bool AK, bool BKM, bool OBF, bool EPI>
void launch_one(dim3 gd, dim3 bd, hipStream_t stream, const msk::GemmArgs &g) {
  if constexpr (KIND == 0) {
    msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, AK, BKM, OBF, EPI><<<gd, bd, 0, stream>>>(g);
  } else if constexpr (KIND == 1) {
    static_assert(BM % 64 == 0 && BN % 64 == 0 && BK_ == 64 && NS == 2 && WGM == 2 && WGN == 2, "the big-tile kernels are 2 x 2 waves on two 64-deep stages");
    msk::gemm_bf16_big_kernel<BM / 64, BN / 64, AK, BKM, OBF, EPI><<<gd, bd, 0, stream>>>(g);
  } else {
    static_assert(BM == 256 && (BN == 384 || BN == 256) && BK_ == 64 && NS == 2 && WGM == 2 && WGN == 2, "the 16x16x32 kernel has two shapes");
    msk::gemm_bf16_x16_kernel<AK, BKM, OBF, EPI, 0, BN><<<gd, bd, 0, stream>>>(g);
  }
}

using msi::balanced_grid;

constexpr int ROWS_WALKED = 8;             // tile rows walked together
constexpr double RUNS_MIN_GAIN = 0.9;      // operand panels that runs may need, of those that taking turns does
constexpr long RUNS_MIN_SPLIT_K = 700;     // contraction elements per part, at least

// Whether the eight XCDs take runs of neighbouring items (xcd_slot) or turns, item i on XCD i % 8.  A grid that is a multiple of eight takes runs.
// Another one takes them where that lets the XCDs' L2s fetch at least a tenth fewer operand panels, counted here: on 1265 unsplit grids of that
// kind (230 drawn products, every tile) runs take 0.89 of the time where they fetch less than half, 0.95 at 0.5 to 0.7, 0.98 at 0.8 to 0.9, and
// 1.02 where they fetch more (tall outputs, whose eight tile rows a walk puts on eight XCDs by turns).  268 x 10288 x 3120 on 243 tiles of 128x128 45.7 -> 31.7 us,
// 552 x 7144 x 6112 on 190 of 128x192 90 -> 64.  The parts of a split product take them from some 700 contraction elements a part (0.92
// at 1000 to 1500); shorter ones are all exchange, which runs slow down (1.06 below 300).
bool xcds_take_runs(const msk::GemmArgs &g, int grid, int bm, int bn, bool a_by_chunk, bool b_by_chunk) {
  if (grid % 8 == 0) return true;
  const long k_part = (long)g.K * g.nkslices / g.splits;
  if (grid > 1024 || (g.splits > 1 && k_part < RUNS_MIN_SPLIT_K)) return false;
  // (the count takes the host 0.8 to 1 us, a fifth of a small product's call: a thread keeps the last answers, by the grid alone)
  struct Answer { int grid, tiles_m, tiles_n, nchunks, splits, bm, bn, by_chunk; bool runs; };
  thread_local Answer answers[16] = {};
  const int by_chunk = a_by_chunk + 2 * b_by_chunk;
  Answer &kept = answers[(unsigned)(grid + 3 * g.tiles_m + 5 * g.tiles_n + 7 * g.nchunks + g.splits) % 16];
  if (kept.grid == grid && kept.tiles_m == g.tiles_m && kept.tiles_n == g.tiles_n && kept.nchunks == g.nchunks && kept.splits == g.splits && kept.bm == bm &&
      kept.bn == bn && kept.by_chunk == by_chunk) return kept.runs;
  // panel numbers of the first round's items, in the order of the kernels' walk
  short a[1024], b[1024];
  int n = 0, na = 0, nb = 0;      // panels of the parts and chunks before this one
  for (int s = 0; s < g.splits && n < grid; s++, na += g.tiles_m, nb += g.tiles_n) {
    for (int c = 0; c < g.nchunks && n < grid; c++) {
      if (c && a_by_chunk) na += g.tiles_m;
      if (c && b_by_chunk) nb += g.tiles_n;
      for (int m0 = 0; m0 < g.tiles_m && n < grid; m0 += ROWS_WALKED)
        for (int j = 0; j < g.tiles_n && n < grid; j++)
          for (int i = m0; i < g.tiles_m && i < m0 + ROWS_WALKED && n < grid; i++, n++) { a[n] = (short)((na + i) & 2047); b[n] = (short)((nb + j) & 2047); }
    }
  }
  long fetched[2];
  for (int runs = 0; runs < 2; runs++) {
    signed char seen_a[2048], seen_b[2048];
    memset(seen_a, -1, sizeof(seen_a));
    memset(seen_b, -1, sizeof(seen_b));
    long rows = 0, cols = 0;
    for (int x = 0, first = 0; x < 8; x++) {
      const int count = grid / 8 + (x < grid % 8);
      for (int k = 0; k < count; k++) {
        const int w = runs ? first + k : x + 8 * k;
        if (seen_a[a[w]] != x) { seen_a[a[w]] = (signed char)x; rows++; }
        if (seen_b[b[w]] != x) { seen_b[b[w]] = (signed char)x; cols++; }
      }
      first += count;
    }
    fetched[runs] = rows * bm + cols * bn;
  }
  kept = {grid, g.tiles_m, g.tiles_n, g.nchunks, g.splits, bm, bn, by_chunk, (double)fetched[1] < RUNS_MIN_GAIN * (double)fetched[0]};
  return kept.runs;
}
constexpr double PARTIAL_ROUND_LOSS = 0.6;

// Two workgroups of the 128x128 kernel fit one compute unit (64 KB of LDS and at most 220 registers per lane each) and
// hide each other's barriers and load latencies: 4096^3 on 1024 such tiles 0.165 -> 0.129 ms, 1536 x 4096 x 2048 0.044 ->
// 0.029 ms.  Every other kernel takes the unit's registers or LDS for itself.  With units reserved the 128x128 kernel
// goes back to one workgroup per unit: the dispatcher would spread a larger grid over the reserved units as well.
int workgroups_per_unit(int variant) { return variant == 3 && g_reserved_cus == 0 ? 2 : 1; }

extern const char *const SPLIT_REFUSALS[];
int split_refused(const Problem &p, const DevFacts &dev, int variant, int splits);

// Whether the 32-bit offsets of a K step of `step` elements reach: they are counted for all of its rows, also for those that a short slice does not have.
// Beyond 4 GiB they would wrap around to rows that it has.
bool reaches(const Problem &p, int step) {
  const long long es = p.in_dtype == MS_DTYPE_BF16 ? 2 : 4;
  const long long a_blk = p.flow == RS ? 8LL * p.lda * es : 0, b_blk = p.flow == LS ? 0 : p.b_blk ? (long long)p.b_blk : 8LL * p.ldb * es;
  return step / 8 * (a_blk > b_blk ? a_blk : b_blk) <= 0x100000000LL;
}

// tile BM x BN, WGM x WGN waves, NS ring stages of BK_ k-elements; contraction split `splits` ways; FAR: for operands that the tile does not reach
template <int BM, int BN, int WGM, int WGN, int BK_, int NS, int KIND = 0, bool FAR = false>
int launch_bf16_tile(const Problem &p, const DevFacts &dev, hipStream_t stream, int variant, int splits) {
  msk::GemmArgs g;
  memset(&g, 0, sizeof(g));
  for (int i = 0; i < p.na; i++) g.a[i] = p.a[i];
  for (int i = 0; i < p.nb; i++) g.b[i] = p.b[i];
  for (int i = 0; i < p.nc; i++) g.c[i] = p.c[i];
  const bool one_output = p.flow == OS || p.sum;
  g.nchunks = one_output ? 1 : p.S;
  g.nkslices = one_output ? p.S : 1;
  g.a_by_chunk = !one_output && (p.flow == RS || p.na > 1);      // (several devices' products: a pointer for every chunk)
  g.b_by_chunk = !one_output && (p.flow == LS || p.nb > 1);
  g.M = p.M; g.N = p.N; g.K = p.K;
  g.lda = p.lda; g.ldb = p.ldb; g.ldc = p.ldc; g.b_blk = p.b_blk ? p.b_blk : (int)((long long)p.ldb * 8 * (p.in_dtype == MS_DTYPE_BF16 ? 2 : 4));
  g.tiles_m = (p.M + BM - 1) / BM;
  g.tiles_n = (p.N + BN - 1) / BN;
  const long total = (long)g.tiles_m * g.tiles_n * g.nchunks;
  if (total > 0x7FFFFFFF) return fail(MS_ERR_ARG, "problem has too many tiles");
  g.total_tiles = (int)total;
  g.splits = 1;
  g.chunk_done = p.chunk_done;
  g.slice_ready = p.slice_ready; g.gate_ticks = p.gate_ticks;
  g_last_tiles_per_chunk = g.tiles_m * g.tiles_n;
  if (splits > 1) {
    const int why = split_refused(p, dev, variant, splits);
    if (why) return fail(MS_ERR_ARG, "contraction cannot be split %d ways here: %s", splits, SPLIT_REFUSALS[why]);
    g.splits = splits;
    g.ws_count = static_cast<int *>(p.ws);
    g.ws_tiles = static_cast<char *>(p.ws) + WS_HEADER_BYTES;
  }
  const long items = total * g.splits;
  const int grid = balanced_grid(items, workgroups_per_unit(variant) * dev.cus);
  g.group_m = ROWS_WALKED;
  g.xcd_runs = xcds_take_runs(g, grid, BM, BN, g.a_by_chunk, g.b_by_chunk);
  msk::set_walk(g, grid);
  dim3 gd(grid), bd(WGM * WGN * 64);
  const bool obf = p.out_dtype == MS_DTYPE_BF16;
  g.act = p.act; g.res = p.res; g.ldr = p.ldr; g.row_sum = p.row_sum; g.row_sumsq = p.row_sumsq;
  const bool epi = p.act != 0 || p.res || p.row_sum || p.row_sumsq;
  if constexpr (FAR) {
    if (p.sum) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, false, false, true, false, true, false, true><<<gd, bd, 0, stream>>>(g);
    else if (p.flow == OS && epi && obf) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, false, true, true, false, false, true><<<gd, bd, 0, stream>>>(g);
    else if (p.flow == OS && epi) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, false, false, true, false, false, true><<<gd, bd, 0, stream>>>(g);
    else if (p.flow == OS && obf) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, false, true, false, false, false, true><<<gd, bd, 0, stream>>>(g);
    else if (p.flow == OS) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, false, false, false, false, false, true><<<gd, bd, 0, stream>>>(g);
    else if (obf) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, false, false, true, false, false, false, true><<<gd, bd, 0, stream>>>(g);
    else msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, false, false, false, false, false, false, true><<<gd, bd, 0, stream>>>(g);
  } else if (p.sum) {
    if constexpr (KIND == 0 && NS == 3 && BM > 64) {
      if (g.splits > 1) {
        if (p.flow == LS) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, true, true, false, true, true><<<gd, bd, 0, stream>>>(g);
        else msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, false, false, true, false, true, true><<<gd, bd, 0, stream>>>(g);
      } else if (p.flow == LS) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, true, true, false, true><<<gd, bd, 0, stream>>>(g);
      else msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, false, false, true, false, true><<<gd, bd, 0, stream>>>(g);
    } else {
      return fail(MS_ERR_UNSUPPORTED, "tile variant %d does not add up several devices' partial sums", variant);
    }
  } else if (p.flow == OS && g.splits > 1 && epi) {      // (split_refused lets the small tiles do that)
    if constexpr (KIND == 0 && NS == 3 && BM == BN && BN <= 128) {
      if (obf) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, false, true, true, false, true><<<gd, bd, 0, stream>>>(g);
      else msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, false, false, true, false, true><<<gd, bd, 0, stream>>>(g);
    } else {
      return fail(MS_ERR_UNSUPPORTED, "tile variant %d does not split products with a fused epilogue", variant);
    }
  } else if (p.flow == OS && g.splits > 1) {      // (split_refused has seen to it that this tile has the exchange)
    if constexpr (KIND == 0 && !(BM == 256 && BN == 256 && WGN == 2)) {
      if (obf) msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, false, true, false, false, true><<<gd, bd, 0, stream>>>(g);
      else msk::gemm_bf16_ring_kernel<BM, BN, BK_, NS, WGM, WGN, true, false, false, false, false, true><<<gd, bd, 0, stream>>>(g);
    } else if constexpr (KIND == 1) {
      if (obf) launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, true, false, true, false>(gd, bd, stream, g);
      else launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, true, false, false, false>(gd, bd, stream, g);
    } else {
      return fail(MS_ERR_UNSUPPORTED, "tile variant %d has no split path", variant);
    }
  } else if (p.flow == OS) {
    if (epi) {
      if (obf) launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, true, false, true, true>(gd, bd, stream, g);
      else launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, true, false, false, true>(gd, bd, stream, g);
    } else {
      if (obf) launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, true, false, true, false>(gd, bd, stream, g);
      else launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, true, false, false, false>(gd, bd, stream, g);
    }
  } else if (p.flow == LS) {
    if (obf) launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, true, true, true, false>(gd, bd, stream, g);
    else launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, true, true, false, false>(gd, bd, stream, g);
  } else {
    if (obf) launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, false, false, true, false>(gd, bd, stream, g);
    else launch_one<KIND, BM, BN, BK_, NS, WGM, WGN, false, false, false, false>(gd, bd, stream, g);
  }
  if (g_launches == 0) g_last_grid = grid;
  g_launches++;
  MS_HIP(hipGetLastError());
  return MS_OK;
}

// Kernel variants (tile, waves, ring stages x k-elements per stage):
//   1: 256x256, 4 waves, 2 x 64     2: 192x192, 4 waves, 3 x 64     3: 128x128, 4 waves, 2 x 64
//   4: 128x192, 4 waves, 3 x 64     5: 256x192, 4 waves, 4 x 32     6: 192x256, 4 waves, 4 x 32
//   7: 256x256, 8 waves, 2 x 64     8: 256x192, 4 waves, 2 x 64     9: 192x256, 4 waves, 2 x 64
//  10: 256x384, 4 waves, 2 x 64 (gemm_bf16_big_kernel<4, 6>)     11: 384x192, 4 waves, 2 x 64 (gemm_bf16_big_kernel<6, 3>)
//  12: 256x384, 4 waves, 2 x 64 on the 16x16x32 MFMA (gemm_bf16_x16_kernel)     13: 256x256, the same kernel
//  14: 128x128, 4 waves, 3 x 64 (one workgroup per unit: for products of at most one round of such tiles, where a third
//      stage covers the load latency that two 64-deep stages do not: 2048^3 in 20.7 us against 26.3 us, 1536^3 14.7 against 18.8)
//      (1 is never picked, 13 and 7 are faster: an id that can be forced, as before)
//      2 and 4 are for outputs of one or two hundred such tiles, where 128x128 pays for more operand bytes per FLOP and
//      256-wide tiles leave units idle: 2048 x 3072 x 4096 on 128x192 43 us, 128x128 50, 256x192 61; 3072^3 on 192x192 48 us, 256x192
//      52; 1499 x 4104 x 3096 on 192x192 46 us, 128x128 57.  (128x256, 256x128 and 192x128 as well would give another 0.3 % over drawn products.)
//  18: 64x64, 4 waves, 3 x 128: outputs of a few dozen 128x128 tiles.  A unit's K step is its operand stream (the loads alone take as long:
//      32 KB per 64 elements of the contraction on 128x128 in 0.31 us, 16 KB on 64x64 in 0.13), so four units with a quarter of the tile
//      each take half the time or less, and the 128-deep step reads three lines where two 64-deep ones read four of rows that start inside a line (64-deep: 0.16).
//      RS 296 x 456 x 11997 in two chunks 73.7 -> 51.0 us, LS 151 x 800 x 8328 in four 69.9 -> 29.7, OS 80 x 512 x 10336 in eight parts 20.6 -> 12.1,
//      200 drawn products of up to 1e11 operations 0.83; the bits of an unsplit product are the other tiles'
//  19: 64x128, 4 waves, 3 x 64: between 18 and 14, where 14 leaves units idle and 18 makes two rounds: LS 1339 x 72 x 1760 in
//      eight chunks 15.5 -> 12.2 us, OS 1261 x 1272 x 2304 22.2 -> 17.7, 220 drawn products 0.975.  (Two to a unit, which their
//      LDS would allow, are no faster than 128x128: 510 of them 39 us, 31.7 on 128x192.)
// The default picks the tile shape that wastes the least of the machine: a launch runs in ceil(work items / CUs) rounds of
// one item per CU (a partly filled last round is charged in part, see balanced_grid), so the estimate is rounds x tile area x
// (contraction + a tile's overhead) / the tile's rate (TILE_RATES).  With two m/n-contiguous operands (RS) the 192-wide ring tiles
// do best on four 32-deep stages, else on two 64-deep ones: whole 128-byte lines per request, half as many barriers.
//
// An output-stationary product with fewer tiles than compute units may split its contraction (work items = tiles x
// splits, see split_k_exchange): a split item costs 1 / splits of the tile, and the whole launch pays for the exchange
// of partial tiles, which is bound by memory bandwidth (splits x m x n fp32 values written through to memory and read
// back: about 2.8 TB/s) plus a fixed few microseconds.  In the estimate's units (tile area x share of the contraction,
// one compute unit doing about 5.7 TFLOP/s) that is (SPLIT_FIX + splits x (SPLIT_PER_PART + m x n x SPLIT_PER_ELEMENT)) / K.
// Measured on 2048 x 1536 x 12288: 80 us unsplit on 192 tiles of 128x128, 68 on 128 of 128x192 in two parts.
struct Pick { int v, splits; double cost; };

constexpr int VARIANTS = 14;
constexpr int SMALL = 18, FLAT = 19;              // the 64x64 and 64x128 tiles (15 to 17: the sums over devices on 14, 4, 2)
constexpr int F32_FIRST = 21, F32_LAST = 25;      // ids of the fp32 kernel's tiles (ms_set_variant, MS_QUERY_LAST_VARIANT)
constexpr int F32_WAVES = 28;                     // gemm_f32_waves_kernel
constexpr int F32_STEP = 32, F32_FAR = 24;        // its K step, and the tile of operands that this does not reach
constexpr int F32_NARROW = 26;                    // and of the two that only the chooser takes (64 x 192, 64 x 128; not ms_set_variant)
struct TileShape { int bm, bn; };
constexpr TileShape TILE_OF[FLAT + 1] = {{0, 0},     {256, 256}, {192, 192}, {128, 128}, {128, 192}, {256, 192},
                                             {192, 256}, {256, 256}, {256, 192}, {192, 256}, {256, 384}, {384, 192},
                                             {256, 384}, {256, 256}, {128, 128}, {0, 0},     {0, 0},     {0, 0},
                                             {64, 64},   {64, 128}};
// a bf16 tile that ms_set_variant names
bool is_bf16_tile(int v) { return (v >= 1 && v <= VARIANTS) || v == SMALL || v == FLAT; }
// contraction elements per step of a tile's K loop, where the split parts are whole steps
int k_step(int v) { return v == SMALL ? 128 : 64; }
// unsplit 256x256 is the 16x16x32 kernel (variant 13), split the eight-wave ring kernel (variant 7); with two m/n-contiguous operands (RS)
// the former loses beyond some 6000 contraction elements per chunk (10240 x 2560 x 12288 in two chunks: 0.622 against 0.555 ms),
// so there the ring kernel stays
constexpr int X16_RS_MAX_K = 6144;
constexpr int SPLIT_CHOICES[] = {1, 2, 3, 4, 6, 8};
constexpr int SPLIT_MAX = 8;
constexpr long SPLIT_MIN_K = 256;            // contraction elements per split item, at least
constexpr double SPLIT_FIX = 4e6;            // fixed cost of an exchange (about 1.4 us),
// a sum over devices has more to gain from staying whole: its parts are the devices, however short each one's share is.  On 300 drawn sums of 2 to 8 devices
// (m and n 64 to 12288) the choice takes 1.0047 of the best tile's and way's time with this, 1.0075 with SPLIT_FIX, 1.0049 with 1.0e7, 1.0069 with 1.7e7: RS 384 x 3712
// x 736 of four devices 23.0 us whole, 29.5 in four parts, LS 411 x 1280 x 280 of four 16.6 and 20.2
constexpr double SUM_SPLIT_FIX = 1.3e7;
constexpr double SPLIT_PER_PART = 1.3e6;     // per part (half a microsecond: a block's last arriver reads the parts one after the other),
constexpr double SPLIT_PER_ELEMENT = 7.9;    // per part and output element (8 bytes through memory)

const char *const SPLIT_REFUSALS[] = {"", "only output-stationary products split their contraction", "no workspace was given",
                                      "more work items than compute units", "too many output tiles for the workspace's counters",
                                      "the partial tiles do not fit the workspace", "too few contraction steps per split",
                                      "split count outside [2, 8]", "this tile variant has no split path",
                                      "of the products with a fused epilogue only those on tiles 14 and 18 are split"};

// 0 if problem p can run on tile variant v with its contraction split `splits` ways, else an index into SPLIT_REFUSALS
int split_refused(const Problem &p, const DevFacts &dev, int v, int splits) {
  const int bm = TILE_OF[v].bm, bn = TILE_OF[v].bn;
  if (splits < 2 || splits > SPLIT_MAX) return 7;
  if (v == 1 || v == 12 || v == 13) return 8;     // 256x256 on four waves: see gemm_bf16_ring_kernel; the 16x16x32 kernels have none
  if (v != SMALL && v != 14 && (p.act || p.res || p.row_sum || p.row_sumsq)) return 9;   // see gemm_bf16_ring_kernel, big_can_split
  if (p.sum ? splits != p.S : p.flow != OS) return 1;      // (the parts of a sum over devices are the devices)
  if (!p.ws) return 2;
  const long tiles = (long)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
  if (tiles * splits > dev.cus) return 3;
  if (tiles > WS_MAX_TILES) return 4;
  if ((size_t)(tiles * splits) * bm * bn * sizeof(float) + WS_HEADER_BYTES > p.ws_bytes) return 5;
  if (((long)(p.K + k_step(v) - 1) / k_step(v)) * p.S < splits) return 6;     // every part needs at least one K step
  return 0;
}

// Relative rates of the tiles as the chooser prices them, by dataflow (256x256 on the eight-wave ring kernel of an OS product = 1): `os`,
// `ls`, `rs` for an unsplit product (128x128 in two stages: a unit that holds one workgroup, PAIRED_* per workgroup where two
// share it; 7 and 10 stand for 13 and 12), `split` for a split one; 0: not for that dataflow.  Fitted, with the constants above and
// below, to every tile and split count forced on 580 drawn products (m 64 to 8192, n and k 256 to 12288, one to sixteen slices, half of
// them at pitches that are no whole lines): the choice takes 1.024 (OS), 1.008 (LS), 1.007 (RS) of the best pair's time in the geometric
// mean and 1.13, 1.04, 1.03 at the 95th percentile; before this fit, and without tiles 2 and 4, 1.046, 1.026, 1.031 and 1.21, 1.14, 1.18.
// The 64x64 tile's were fitted beside them to 400 drawn products of up to 4e10 operations: 1.017, 1.005, 1.004 of the best pair's time; 1.17, 1.32, 1.14 without it.
// The 64x128 tile's to 400 others: 1.016, 1.009, 1.006; 1.044, 1.032, 1.026 without it.
struct TileRate { int v; double os, ls, rs, split; };
constexpr TileRate TILE_RATES[] = {{7, 1.11, 1.065, 0.945, 1.0}, {10, 1.2, 1.146, 1.076, 1.14}, {11, 0.98, 0.939, 0.986, 0.98}, {8, 0.93, 0.972, 0.0, 0.93},
                                   {9, 0.95, 0.972, 0.0, 0.95}, {5, 0.0, 0.0, 0.994, 0.0}, {6, 0.0, 0.0, 0.959, 0.0}, {3, 0.486, 0.458, 0.5, 0.486},
                                   {14, 0.66, 0.706, 0.69, 0.66}, {4, 0.795, 0.814, 0.86, 0.795}, {2, 0.93, 0.938, 0.96, 0.93},
                                   {SMALL, 0.31, 0.38, 0.33, 0.4}, {FLAT, 0.4, 0.43, 0.43, 0.48}};
constexpr double PAIRED_OS = 0.38, PAIRED_LS = 0.424, PAIRED_RS = 0.424;
// prologue and write-out of a tile, as contraction elements
constexpr double TILE_OVERHEAD_K = 80.0;
// what a tile loses of a last round that is partly filled: units idle then let the others clock higher, but only on the tiles that
// reach the power limit
double partial_round_loss(int v) { return v == 3 || v == 14 || v == SMALL || v == FLAT ? 1.0 : v == 2 || v == 4 ? 0.87 : PARTIAL_ROUND_LOSS; }

// tiles that carry the sum over devices, and what the end of a device's share costs them (its accumulators join the totals,
// 0.7 to 1 us of vector work), as contraction elements
bool carries_sum(int v) { return v == 2 || v == 4 || v == 14; }
constexpr double FOLD_K = 90.0;

// Unsplit output-stationary products of more than half a round of 64x64 tiles take them below this many contraction elements: from there on 128x128
// in three or four parts is ahead on ten of twelve drawn products (483 x 1944 x 9472: 30.1 against 44.2 us, 1406 x 472 x 4488 20.4 against
// 22.1; 1024 x 768 x 4096 is one that loses, 17.6 against 15.0).
constexpr double SMALL_OS_MAX_K = 4096.0;
// what each further round of them costs besides its share (about 0.9 us: 480 x 296 x 696 in eight chunks, 320 such tiles in two rounds,
// 10.0 us against 8.9 on 96 of 128x128), and their rate where the whole device runs them for more than one (LS 1871 x 24 x 10016 in sixteen chunks, 480
// tiles, 85 us against 71 on 240 of 128x128)
constexpr double SMALL_ROUND = 2.5e6, SMALL_CROWDED = 1.1;
constexpr double L2S_BYTES = 28e6;      // what of an operand the eight XCDs' L2s (32 MB) hold beside the rest

// the tile shape and split count with the lowest estimated cost for the whole problem (`small`: the 64-row tiles among them)
Pick pick_variant(const Problem &p, const DevFacts &dev, bool small = true) {
  const bool rs = p.flow == RS, ls = p.flow == LS;
  const long chunks = p.flow == OS || p.sum ? 1 : p.S;
  const double total_k = p.flow == OS || p.sum ? (double)p.K * p.S : (double)p.K;
  const double whole_k = (double)((p.K + 63) / 64 * 64) * (p.flow == OS || p.sum ? p.S : 1);      // (the 64x64 tile feels the tails of short slices: 500 drawn OS products take 1.016 of the best tile's time with tails rounded up to 64, 1.018 to its step of 128, or not at all)
  const long small_tiles = (long)((p.M + 63) / 64) * ((p.N + 63) / 64) * chunks;
  const int forced_splits = p.sum ? 0 : g_splits;      // (a split count is forced on output-stationary products)
  Pick best = {0, 1, 0};
  for (const TileRate &c : TILE_RATES) {
    if (p.sum && !carries_sum(c.v)) continue;
    if ((c.v == SMALL && (!small || !reaches(p, k_step(SMALL)))) || (c.v == FLAT && !small)) continue;
    const int bm = TILE_OF[c.v].bm, bn = TILE_OF[c.v].bn;
    const bool pairs = workgroups_per_unit(c.v) == 2;
    const double rate = rs ? c.rs : ls ? c.ls : c.os;
    const long tiles = (long)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn) * chunks;
    for (int splits : SPLIT_CHOICES) {
      if (forced_splits != 0 && splits != forced_splits) continue;
      if (splits == 1 ? rate == 0.0 : c.split == 0.0) continue;
      // (64x128 is for where 64x64 makes more than half a round: below, the smaller tile is ahead, 365 x 368 x 432 in six slices 6.8 against 8.2 us)
      if (c.v == FLAT && splits == 1 && 2 * small_tiles <= dev.cus) continue;
      // (chunks of one 64-row tile leave it no more tiles than 128x128 and half the bytes in flight: RS 48 x 5432 x 4393 in four chunks 39 us against 32; up to
      // 2048 contraction elements its shorter steps win, RS 40 x 1496 x 1361 in sixteen 10.7 against 12.2, but less of it where 128x128 makes one round of two
      // workgroups a unit and it makes two: RS 256 x 4048 x 642 in sixteen, 512 tiles, 15.4 against 17.5, 512 x 3904 x 889 15.3 against 20.0; 384 x 3520 x 292, 448 tiles, 8.6 against 8.3)
      if (c.v == FLAT && splits == 1 && p.M <= 64 && (total_k >= 2048.0 || (tiles > dev.cus && tiles <= 2L * dev.cus && tiles * total_k >= 1200.0 * dev.cus))) continue;
      // (RS chunks of one 64-row tile do nothing but stream W, and of a W whose rows are no whole lines 64 columns fetch two lines for one.  With most of the units at that,
      // and W beyond what the L2s hold, the fabric is what they wait for: RS 72 x 5256 x 9701 in three chunks 82.8 us, 64.4 on 126 tiles of 128x128, 112 x 7024 x 7648 in two
      // 54.4 and 45.9, 48 x 2632 x 6867 in six 43.1 and 40.3; of ten such products in 1200 drawn ones two lose, 0.92 and 0.94)
      if (c.v == SMALL && splits == 1 && rs && p.M <= 64 && p.N % 64 != 0 && tiles <= dev.cus && 4 * tiles > 3L * dev.cus && 2.0 * p.N * total_k > L2S_BYTES) continue;
      if (c.v == SMALL && splits == 1 && forced_splits == 0 && 2 * tiles > dev.cus && total_k >= SMALL_OS_MAX_K && !split_refused(p, dev, 14, 3)) continue;
      if (splits > 1 && (split_refused(p, dev, c.v, splits) || (forced_splits == 0 && total_k / splits < SPLIT_MIN_K))) continue;
      // rounds the launch is charged: whole ones, or with the last round partly filled (see balanced_grid) its filled
      // share plus a part of the rest; a launch of less than one round is charged the same way, down to 0.7 of a round (the
      // idle units' power lets the busy ones clock up to 1.4 times higher)
      const long slots = (long)dev.cus * (splits == 1 && pairs ? 2 : 1);     // (a split launch is one item per unit)
      const double exact = (double)(tiles * splits) / slots;
      const double whole = (double)((tiles * splits + slots - 1) / slots);
      const double loss = partial_round_loss(c.v);
      const double part = exact + loss * (1.0 - exact);
      const double rounds = exact <= 1.0 ? (part > 0.7 ? part : 0.7) : exact + loss * (whole - exact);
      const double exchange = splits == 1 ? 0.0 : (p.sum ? SUM_SPLIT_FIX : SPLIT_FIX) + splits * (SPLIT_PER_PART + (double)p.M * p.N * SPLIT_PER_ELEMENT);
      // (two 128x128 workgroups share a unit only where there are more tiles than units)
      const double shared = !pairs || tiles * splits <= dev.cus ? 0.0 : tiles * splits >= 2L * dev.cus ? 1.0 : (double)(tiles * splits - dev.cus) / dev.cus;
      const double eff = splits > 1 ? c.split : rate - (pairs ? (rate - (rs ? PAIRED_RS : ls ? PAIRED_LS : PAIRED_OS)) * shared : 0.0);
      const double crowded = c.v == SMALL && whole > 1.0 ? SMALL_CROWDED : 1.0;
      const double cost = (rounds * crowded * bm * bn / eff * ((c.v == SMALL ? whole_k : total_k) / splits + TILE_OVERHEAD_K + (p.sum && splits == 1 ? FOLD_K * p.S : 0.0)) + exchange + (c.v == SMALL ? SMALL_ROUND * (whole - 1.0) : 0.0)) / total_k;
      if (best.v == 0 || cost < best.cost) best = {c.v, splits, cost};
    }
  }
  if (p.sum) return best;
  // An unsplit 256x384 product runs on the 16x16x32 kernel: 4-8 % faster than the 32x32x16 one, which stays selectable
  // as variant 10 and carries the split contraction.
  if (best.splits == 1 && best.v == 10) best.v = 12;
  // Likewise an unsplit 256x256 product (4096^3 in 0.093-0.095 ms against 0.106 ms on the ring kernel, 4096 x 4096 x 14336 in
  // 0.302-0.309 against 0.344 ms); the eight-wave ring kernel stays selectable as variant 7 and carries the split contraction.
  // (not where an LS chunk is a single tile column: every XCD then streams all of A, the product is bound by the fabric, and
  // two waves per SIMD ride that out better: 8192 x 256 x 8192 in eight chunks 0.217 against 0.262 ms)
  const bool one_column_chunks = ls && p.N <= 256;
  if (best.splits == 1 && best.v == 7 && !(rs && p.K > X16_RS_MAX_K) && !one_column_chunks) best.v = 13;
  return best;
}

int launch_variant(int v, int splits, const Problem &p, const DevFacts &dev, hipStream_t stream) {
  if (p.slice_ready && v == 1) return fail(MS_ERR_UNSUPPORTED, "tile variant %d has no input gate (256x256 on four waves of the ring kernel)", v);
  if (!reaches(p, k_step(v))) return fail(MS_ERR_UNSUPPORTED, "tile variant %d does not reach rows of more than %d MB", v, 4096 / k_step(v));
  // (the kernels that add up devices' sums go by ids of their own: 15 to 17 for the tiles 14, 4 and 2)
  if (g_launches == 0) { g_last_variant = !p.sum ? v : v == 14 ? 15 : v == 4 ? 16 : 17; g_last_splits = splits; }
  switch (v) {
    case 1: return launch_bf16_tile<256, 256, 2, 2, 64, 2>(p, dev, stream, 1, splits);
    case 2: return launch_bf16_tile<192, 192, 2, 2, 64, 3>(p, dev, stream, 2, splits);
    case 3: return launch_bf16_tile<128, 128, 2, 2, 64, 2>(p, dev, stream, 3, splits);
    case 4: return launch_bf16_tile<128, 192, 2, 2, 64, 3>(p, dev, stream, 4, splits);
    case 5: return launch_bf16_tile<256, 192, 2, 2, 32, 4>(p, dev, stream, 5, splits);
    case 6: return launch_bf16_tile<192, 256, 2, 2, 32, 4>(p, dev, stream, 6, splits);
    case 7: return launch_bf16_tile<256, 256, 2, 4, 64, 2>(p, dev, stream, 7, splits);
    case 8: return launch_bf16_tile<256, 192, 2, 2, 64, 2>(p, dev, stream, 8, splits);
    case 9: return launch_bf16_tile<192, 256, 2, 2, 64, 2>(p, dev, stream, 9, splits);
    case 10: return launch_bf16_tile<256, 384, 2, 2, 64, 2, 1>(p, dev, stream, 10, splits);
    case 11: return launch_bf16_tile<384, 192, 2, 2, 64, 2, 1>(p, dev, stream, 11, splits);
    case 12: return launch_bf16_tile<256, 384, 2, 2, 64, 2, 2>(p, dev, stream, 12, splits);
    case 13: return launch_bf16_tile<256, 256, 2, 2, 64, 2, 2>(p, dev, stream, 13, splits);
    case 14: return launch_bf16_tile<128, 128, 2, 2, 64, 3>(p, dev, stream, 14, splits);
    case SMALL: return launch_bf16_tile<64, 64, 2, 2, 128, 3>(p, dev, stream, SMALL, splits);
    case FLAT: return launch_bf16_tile<64, 128, 2, 2, 64, 3>(p, dev, stream, FLAT, splits);
    default: return fail(MS_ERR_ARG, "unknown kernel variant %d", v);
  }
}

// An output-stationary product whose best single tile shape leaves much of its last round idle is done in two
// launches: the 256x384 tile on as many leading tile columns of C as fill whole rounds, the best shape for what
// is left on the remaining columns (4096x9216x12288: 256 tiles of 256x384 plus 256 tiles of 256x192, 0.67 ms,
// instead of 768 tiles of 256x192 in three rounds, 0.76 ms).  The second launch costs about a hundredth of a
// millisecond (launch gap, one more prologue), which the estimate charges as tile area.  LS / RS are not split:
// their chunks are promised in slice order.
int launch_bf16(const Problem &p, const DevFacts &dev, hipStream_t stream) {
  if (!dev.gfx950) return fail(MS_ERR_UNSUPPORTED, "the bf16 kernels need a gfx950 device");
  const bool forced = is_bf16_tile(g_variant) && (!p.sum || carries_sum(g_variant));
  if (!reaches(p, k_step(14))) {
    if ((forced && g_variant != 14) || (g_splits > 1 && !p.sum))
      return fail(MS_ERR_UNSUPPORTED, "tile variant %d in %d parts does not reach rows of more than %d MB", g_variant, g_splits > 1 ? g_splits : 1, 4096 / k_step(14));
    if (g_launches == 0) { g_last_variant = p.sum ? 15 : 14; g_last_splits = 1; }
    return launch_bf16_tile<128, 128, 2, 2, 64, 3, 0, true>(p, dev, stream, 14, 1);
  }
  if (forced) return launch_variant(g_variant, g_splits > 1 ? g_splits : 1, p, dev, stream);
  const Pick single = pick_variant(p, dev);
  // (a gated product stays one launch: a second one would stand in the stream behind the first while that waits for slices)
  if (p.flow == OS && single.splits == 1 && g_splits == 0 && !p.slice_ready) {
    constexpr int BM = 256, BN = 384;
    constexpr double EFF = 1.2;      // (TILE_RATES)
    const long tiles_m = (p.M + BM - 1) / BM;
    const long total_k = (long)p.K * p.S;
    // whole rounds of the big tile: the largest count of leading tile columns whose tiles are a multiple of the CUs
    long nb1 = p.N / BN;
    while (nb1 > 0 && (tiles_m * nb1) % dev.cus != 0) nb1--;
    const long n1 = nb1 * BN;
    if (nb1 > 0 && n1 < p.N) {
      Problem rest = p;
      rest.N = p.N - (int)n1;
      rest.ws = nullptr;   // the second launch is not split: the first may still be using the workspace's counters
      const Pick tail = pick_variant(rest, dev);
      const double second_launch = 3.4e7 / (double)total_k;      // ~12 us at the rate one CU computes tile area x K
      const double cost = (double)(tiles_m * nb1 / dev.cus) * BM * BN / EFF * (1.0 + TILE_OVERHEAD_K / (double)total_k) + tail.cost + second_launch;
      if (cost < 0.97 * single.cost) {
        const int es_in = 2, es_out = p.out_dtype == MS_DTYPE_BF16 ? 2 : 4;
        Problem head = p;
        head.N = (int)n1;
        int rc = launch_variant(12, 1, head, dev, stream);   // (see pick_variant)
        if (rc != MS_OK) return rc;
        const void *b2[MS_MAX_SLICES];
        void *c2[1] = {static_cast<char *>(p.c[0]) + n1 * es_out};
        for (int s = 0; s < p.nb; s++) b2[s] = static_cast<const char *>(p.b[s]) + n1 * es_in;
        rest.b = b2;
        rest.c = c2;
        if (p.res) rest.res = static_cast<const char *>(p.res) + n1 * es_out;
        return launch_variant(tail.v, 1, rest, dev, stream);
      }
    }
  }
  return launch_variant(single.v, single.splits, p, dev, stream);
}

// fp32 operands: gemm_f32_tile_kernel on one of its seven tiles (ids F32_FIRST ..: 256 x 128 and 128 x 192 on eight
// waves, 128 x 128, 64 x 64 and 192 x 192 on four; F32_NARROW ..: 64 x 192 and 64 x 128 on four); `share`: two workgroups
// of the 128 x 128 tile or of one of the 64-row tiles per compute unit
int f32_split_refused(const Problem &p, const DevFacts &dev, int bm, int bn, int splits);

int fill_f32_args(const Problem &p, int bm, int bn, msk::GemmArgs &g, long &total) {
  memset(&g, 0, sizeof(g));
  for (int i = 0; i < p.na; i++) g.a[i] = p.a[i];
  for (int i = 0; i < p.nb; i++) g.b[i] = p.b[i];
  for (int i = 0; i < p.nc; i++) g.c[i] = p.c[i];
  g.nchunks = p.flow == OS ? 1 : p.S;
  g.nkslices = p.flow == OS ? p.S : 1;
  g.a_by_chunk = p.flow == RS || (p.flow == LS && p.na > 1);      // (several devices' products: a pointer for every chunk)
  g.b_by_chunk = p.flow == LS || (p.flow == RS && p.nb > 1);
  g.M = p.M; g.N = p.N; g.K = p.K;
  g.lda = p.lda; g.ldb = p.ldb; g.ldc = p.ldc; g.b_blk = p.b_blk ? p.b_blk : (int)((long long)p.ldb * 8 * (p.in_dtype == MS_DTYPE_BF16 ? 2 : 4));
  g.tiles_m = (p.M + bm - 1) / bm;
  g.tiles_n = (p.N + bn - 1) / bn;
  total = (long)g.tiles_m * g.tiles_n * g.nchunks;
  if (total > 0x7FFFFFFF) return fail(MS_ERR_ARG, "problem has too many tiles");
  g.total_tiles = (int)total;
  g.splits = 1;
  g.chunk_done = p.chunk_done;
  g.slice_ready = p.slice_ready; g.gate_ticks = p.gate_ticks;
  g_last_tiles_per_chunk = g.tiles_m * g.tiles_n;
  return MS_OK;
}

template <int WGM, int WGN, int TM, int TN, bool FAR = false>
int launch_f32_tile(const Problem &p, const DevFacts &dev, hipStream_t stream, int id, bool share, int splits) {
  constexpr int BM = 32 * TM * WGM, BN = 32 * TN * WGN;
  msk::GemmArgs g;
  long total = 0;
  if (int rc = fill_f32_args(p, BM, BN, g, total)) return rc;
  if (splits > 1) {
    const int why = f32_split_refused(p, dev, BM, BN, splits);
    if (why) return fail(MS_ERR_ARG, "contraction cannot be split %d ways here: %s", splits, SPLIT_REFUSALS[why]);
    g.splits = splits;
    g.ws_count = static_cast<int *>(p.ws);
    g.ws_tiles = static_cast<char *>(p.ws) + WS_HEADER_BYTES;
  }
  const long items = total * g.splits;
  const int grid = !(share && WGM * WGN == 4) ? balanced_grid(items, dev.cus) : items <= 2L * dev.cus ? (int)items : balanced_grid(items, 2 * dev.cus);
  g.group_m = ROWS_WALKED;
  g.xcd_runs = xcds_take_runs(g, grid, BM, BN, g.a_by_chunk, g.b_by_chunk);
  msk::set_walk(g, grid);
  dim3 gd(grid), bd(WGM * WGN * 64);
  const bool obf = p.out_dtype == MS_DTYPE_BF16;
  if constexpr (FAR) {
    if (p.flow == OS && obf) msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, true, false, true><<<gd, bd, 0, stream>>>(g);
    else if (p.flow == OS) msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, false, false, true><<<gd, bd, 0, stream>>>(g);
    else if (obf) msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, false, false, true, false, true><<<gd, bd, 0, stream>>>(g);
    else msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, false, false, false, false, true><<<gd, bd, 0, stream>>>(g);
  } else if (p.flow == OS) {
    if (g.splits > 1) {
      if (obf) msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, true, true><<<gd, bd, 0, stream>>>(g);
      else msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, false, true><<<gd, bd, 0, stream>>>(g);
    } else if (obf) msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, true><<<gd, bd, 0, stream>>>(g);
    else msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, false, false><<<gd, bd, 0, stream>>>(g);
  } else if (p.flow == LS) {
    if (obf) msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, true, true><<<gd, bd, 0, stream>>>(g);
    else msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, true, true, false><<<gd, bd, 0, stream>>>(g);
  } else {
    if (obf) msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, false, false, true><<<gd, bd, 0, stream>>>(g);
    else msk::gemm_f32_tile_kernel<WGM, WGN, TM, TN, false, false, false><<<gd, bd, 0, stream>>>(g);
  }
  if (g_launches == 0) { g_last_grid = (int)gd.x; g_last_variant = id; g_last_splits = g.splits; }
  g_launches++;
  MS_HIP(hipGetLastError());
  return MS_OK;
}

// gemm_f32_waves_kernel: 32 x 32 tiles, the contraction shared out over a workgroup's waves
int launch_f32_waves(const Problem &p, const DevFacts &dev, hipStream_t stream) {
  msk::GemmArgs g;
  long total = 0;
  if (int rc = fill_f32_args(p, 32, 32, g, total)) return rc;
  const dim3 gd(balanced_grid(total, dev.cus)), bd(256);
  g.group_m = ROWS_WALKED;
  g.xcd_runs = xcds_take_runs(g, (int)gd.x, 32, 32, g.a_by_chunk, g.b_by_chunk);
  msk::set_walk(g, (int)gd.x);
  const bool obf = p.out_dtype == MS_DTYPE_BF16;
  if (p.flow == OS) {
    if (obf) msk::gemm_f32_waves_kernel<true, false, true><<<gd, bd, 0, stream>>>(g);
    else msk::gemm_f32_waves_kernel<true, false, false><<<gd, bd, 0, stream>>>(g);
  } else if (p.flow == LS) {
    if (obf) msk::gemm_f32_waves_kernel<true, true, true><<<gd, bd, 0, stream>>>(g);
    else msk::gemm_f32_waves_kernel<true, true, false><<<gd, bd, 0, stream>>>(g);
  } else {
    if (obf) msk::gemm_f32_waves_kernel<false, false, true><<<gd, bd, 0, stream>>>(g);
    else msk::gemm_f32_waves_kernel<false, false, false><<<gd, bd, 0, stream>>>(g);
  }
  if (g_launches == 0) { g_last_grid = (int)gd.x; g_last_variant = F32_WAVES; g_last_splits = 1; }
  g_launches++;
  MS_HIP(hipGetLastError());
  return MS_OK;
}

// 0 if the fp32 product p can run on a bm x bn tile with its contraction split `splits` ways, else an index into SPLIT_REFUSALS
int f32_split_refused(const Problem &p, const DevFacts &dev, int bm, int bn, int splits) {
  if (splits < 2 || splits > SPLIT_MAX) return 7;
  if (p.flow != OS) return 1;
  if (!p.ws) return 2;
  const long tiles = (long)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
  if (tiles * splits > dev.cus) return 3;
  if (tiles > WS_MAX_TILES) return 4;
  if ((size_t)(tiles * splits) * bm * bn * sizeof(float) + WS_HEADER_BYTES > p.ws_bytes) return 5;
  if (((long)(p.K + 31) / 32) * p.S < splits) return 6;     // every part needs at least one K step
  return 0;
}

// The fp32 tiles as the chooser prices them: time per output element and contraction step relative to the 256 x 128
// tile's, for a unit that holds one workgroup, and the factor by which a unit that holds two four-wave workgroups takes
// longer over the pair.  Fitted to ten products from 512^2 x 1024 to 4096^3 (one round of 256 tiles of 128 x 192 on
// 4096 contraction elements 363 us, of 256 x 128 468 us, of 128 x 128 on 8192 elements 510 us; 512 tiles of 64 x 64
// shared 133 us, alone in two rounds 150 us; 1024 tiles of 128 x 128 shared 957 us; one round of 256 tiles of 192 x 192,
// four waves of 3 x 3 tiles each, 567 us).  Unlike the bf16 kernels this one
// does not sit on the power limit: a partly filled round costs a whole one.
// The two 64-row tiles with more columns than rows are for outputs whose rows fill a 128-row tile badly, and for the step
// from one round to two between 64 x 64 and 128 x 128 (256 tiles on 2048 contraction elements: 64 x 192 105 us, two per unit
// 192 us a pair; 64 x 128 73 and 129 us).  Four chunks of 260 x 2056 on 1023 elements: 220 tiles of 64 x 192 in 55 us, 204 of
// 128 x 128 or 660 of 64 x 64 in 63; three of 500 x 1500 on 1500: 80 against 92 us; 700 x 900 x 4000 in four parts: 61
// against 71 us; 2048^3 on 512 tiles of 64 x 128: 129 against 134 us.
struct F32Tile { int id, bm, bn; bool pairs; double cost, shared; };      // pairs: two such workgroups fit a compute unit
constexpr F32Tile F32_TILES[] = {{F32_FIRST, 256, 128, false, 1.0, 0.0}, {F32_FIRST + 1, 128, 192, false, 1.0 / 0.967, 0.0},
                                 {F32_FIRST + 2, 128, 128, true, 1.0 / 0.918, 1.88}, {F32_FIRST + 3, 64, 64, true, 1.0 / 0.78, 1.78},
                                 {F32_FIRST + 4, 192, 192, false, 1.0 / 0.93, 0.0},
                                 {F32_NARROW, 64, 192, true, 1.0 / 0.87, 1.85}, {F32_NARROW + 1, 64, 128, true, 1.0 / 0.85, 1.82}};

int launch_f32_id(int id, bool share, int splits, const Problem &p, const DevFacts &dev, hipStream_t stream) {
  switch (id) {
    case F32_FIRST: return launch_f32_tile<4, 2, 2, 2>(p, dev, stream, id, false, splits);
    case F32_FIRST + 1: return launch_f32_tile<4, 2, 1, 3>(p, dev, stream, id, false, splits);
    case F32_FIRST + 2: return launch_f32_tile<2, 2, 2, 2>(p, dev, stream, id, share, splits);
    case F32_FIRST + 3: return launch_f32_tile<2, 2, 1, 1>(p, dev, stream, id, share, splits);
    case F32_NARROW: return launch_f32_tile<2, 2, 1, 3>(p, dev, stream, id, share, splits);
    case F32_NARROW + 1: return launch_f32_tile<2, 2, 1, 2>(p, dev, stream, id, share, splits);
    case F32_WAVES: return launch_f32_waves(p, dev, stream);
    default: return launch_f32_tile<2, 2, 3, 3>(p, dev, stream, id, false, splits);
  }
}

// An output-stationary fp32 product whose tiles leave compute units idle may split its contraction like the bf16 ones
// (work items = tiles x splits, see split_k_exchange).  The exchange of the partial tiles is priced, in the chooser's
// unit (the 256 x 128 tile's time per output element and contraction step, 3.5e-6 us), at
// (F32_SPLIT_FIX + splits x (F32_SPLIT_PART + m x n x F32_SPLIT_PER_ELEMENT)) / K: about 4 us, 0.35 us a part and 2 us per
// million partial elements.  A part's K loop runs whole summation blocks (four steps of 32): 60 steps in seven parts are
// twelve steps each, not nine.  Priced as shares of the contraction, 140 x 1360 x 1888 took 64 x 128 in seven parts (23 us)
// for 64 x 64 in three (five blocks, 19 us), and one product in thirty was more than 2 % slower than on the tiles with ids up
// to 25 alone.  Fitted to every tile and split count on 400 products from 64 x 256 x 256 to 8192 x 12288 x 12288 (2e10 operations at
// most): the choice takes 1.006 of the best pair's time in the geometric mean, 1.03 at the 95th percentile (shares: 1.015, 1.09).
constexpr double F32_SPLIT_FIX = 1.2e6, F32_SPLIT_PART = 1e5, F32_SPLIT_PER_ELEMENT = 0.6;
constexpr long F32_SPLIT_MIN_K = 256;      // contraction elements per split item, at least

// gemm_f32_waves_kernel: a round of 32 x 32 tiles takes 0.605 us for every four steps of the contraction, and another round 2.5 us of its own
// (fitted to 200 drawn products; 8 % off at the 95th percentile).  Chunk products take it wherever it is priced lower, output-stationary
// ones up to 1536 contraction elements: beyond, the tiles above with their contraction split are level or ahead on nine in ten (256 x 256 x
// 4096: 64 x 64 in eight parts 19.9 us, this 24.9).  The choice takes 1.007 of the better one's time in the geometric mean, 1.05 at the
// 95th percentile.
constexpr double F32_WAVES_STEPS4_US = 0.605, F32_WAVES_ROUND_US = 2.5, F32_UNIT_US = 3.5e-6;
constexpr long F32_WAVES_OS_MAX_K = 1536;

// the fp32 tile, whether its workgroups pair up on the units, and the split count with the lowest estimated cost (id 0: a
// forced tile and split count that cannot be)
struct F32Pick { int id, splits; bool share; };
F32Pick pick_f32(const Problem &p, const DevFacts &dev) {
  const long chunks = p.flow == OS ? 1 : p.S;
  const long total_k = (long)p.K * (p.flow == OS ? p.S : 1);
  const long ksteps = (long)((p.K + 31) / 32) * (p.flow == OS ? p.S : 1);
  const bool forced_tile = g_variant >= F32_FIRST && g_variant != F32_WAVES;
  F32Pick best = {0, 1, false};
  double best_cost = 0.0;
  for (const F32Tile &t : F32_TILES) {
    if (forced_tile && g_variant != t.id) continue;
    const long tiles = (long)((p.M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn) * chunks;
    const double area = (double)t.bm * t.bn * t.cost;
    for (int splits = 1; splits <= SPLIT_MAX; splits++) {
      if (forced_tile && g_splits != 0 && splits != g_splits) continue;
      if (!forced_tile && g_splits != 0) { if (splits > 1) break; }      // (a split forced for the bf16 tiles says nothing here)
      if (splits > 1 && (f32_split_refused(p, dev, t.bm, t.bn, splits) || (!(forced_tile && g_splits != 0) && total_k / splits < F32_SPLIT_MIN_K))) continue;
      const long items = tiles * splits;
      const double item = area * 128.0 * (double)(((ksteps + splits - 1) / splits + 3) / 4) / total_k;      // whole summation blocks
      double cost = (double)((items + dev.cus - 1) / dev.cus) * item;
      bool share = false;
      if (t.pairs && g_reserved_cus == 0 && items > dev.cus) {
        const double both = (double)((items + 2L * dev.cus - 1) / (2L * dev.cus)) * item * t.shared;
        if (both < cost) { cost = both; share = true; }
      }
      if (splits > 1) cost += (F32_SPLIT_FIX + splits * (F32_SPLIT_PART + (double)p.M * p.N * F32_SPLIT_PER_ELEMENT)) / total_k;
      if (best.id == 0 || cost < best_cost) { best = {t.id, splits, share}; best_cost = cost; }
    }
  }
  if (!forced_tile && (p.flow != OS || total_k <= F32_WAVES_OS_MAX_K)) {
    const long rounds = ((long)((p.M + 31) / 32) * ((p.N + 31) / 32) * chunks + dev.cus - 1) / dev.cus;
    const double us = (double)(rounds * ((ksteps + 3) / 4)) * F32_WAVES_STEPS4_US + (double)(rounds - 1) * F32_WAVES_ROUND_US;
    if (us / F32_UNIT_US / (double)total_k < best_cost) best = {F32_WAVES, 1, false};
  }
  return best;
}

int launch_f32(const Problem &p, const DevFacts &dev, hipStream_t stream) {
  if (!reaches(p, F32_STEP)) {
    if (g_splits > 1 || (g_variant >= F32_FIRST && g_variant != F32_FAR)) return fail(MS_ERR_UNSUPPORTED, "fp32 tile variant %d does not reach rows of more than %d MB", g_variant, 4096 / F32_STEP);
    return launch_f32_tile<2, 2, 1, 1, true>(p, dev, stream, F32_FAR, false, 1);
  }
  if (g_variant == F32_WAVES) return launch_f32_waves(p, dev, stream);
  const F32Pick best = pick_f32(p, dev);
  if (best.id == 0) return fail(MS_ERR_ARG, "contraction cannot be split %d ways on fp32 tile %d here", g_splits, g_variant);
  return launch_f32_id(best.id, best.share, best.splits, p, dev, stream);
}

// the device as this thread's launches may use it: without the compute units it has been told to leave free
DevFacts usable(const DevInfo &dev) {
  DevFacts f = dev;
  f.cus = f.cus - g_reserved_cus > 0 ? f.cus - g_reserved_cus : 1;
  return f;
}

int run(const Problem &p, void *stream) {
  int rc = validate(p);
  if (rc) return rc;
  DevInfo *dev = nullptr;
  rc = dev_info(&dev);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  g_launches = 0;
  g_last_variant = 0;
  g_last_splits = 1;
  // the kernels are persistent, one workgroup per compute unit: with units reserved they run on the rest, and the
  // tile choice plans for that many
  const DevFacts facts = usable(*dev);
  return p.in_dtype == MS_DTYPE_BF16 ? launch_bf16(p, facts, st) : launch_f32(p, facts, st);
}

int timed(const Problem &p, void *stream, int warmup, int reps, float *ms_out) {
  if (warmup < 0 || reps < 1 || !ms_out) return fail(MS_ERR_ARG, "timing: need warmup >= 0, reps >= 1 and an output array");
  hipStream_t st = (hipStream_t)stream;
  for (int i = 0; i < warmup; i++) {
    int rc = run(p, stream);
    if (rc) return rc;
  }
  hipEvent_t e0, e1;
  MS_HIP(hipEventCreate(&e0));
  MS_HIP(hipEventCreate(&e1));
  int rc = MS_OK;
  for (int r = 0; r < reps && rc == MS_OK; r++) {
    (void)hipEventRecord(e0, st);
    rc = run(p, stream);
    (void)hipEventRecord(e1, st);
    if (hipEventSynchronize(e1) != hipSuccess) rc = fail(MS_ERR_HIP, "hipEventSynchronize failed");
    float ms = 0.f;
    if (rc == MS_OK && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = fail(MS_ERR_HIP, "hipEventElapsedTime failed");
    ms_out[r] = ms;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc == MS_OK) MS_HIP(hipStreamSynchronize(st));
  return rc;
}

Problem make_problem(Flow flow, const void *const *a, const void *const *b, void *const *c, int na, int nb, int nc, int S,
                     int m, int n, int k, int lda, int ldb, int ldc, int in_dtype, int out_dtype) {
  Problem p;
  p.flow = flow; p.a = a; p.b = b; p.c = c; p.na = na; p.nb = nb; p.nc = nc; p.S = S;
  p.M = m; p.N = n; p.K = k; p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.in_dtype = in_dtype; p.out_dtype = out_dtype;
  if (S < 1 || S > MS_MAX_SLICES) p.na = p.nb = p.nc = 0;   // the pointer tables are not read for a bad S
  return p;
}
Problem make_os(const void *const *A, const void *const *B, int S, int m, int n, int k, int lda, int ldb,
                void *const *C, int ldc, int in_dtype, int out_dtype) {
  return make_problem(OS, A, B, C, S, S, 1, S, m, n, k, lda, ldb, ldc, in_dtype, out_dtype);
}
Problem make_ls(const void *const *A, int lda, const void *const *W, int ldw, int S, int m, int n, int k,
                void *const *Y, int ldy, int in_dtype, int out_dtype = MS_DTYPE_F32) {
  return make_problem(LS, A, W, Y, 1, S, S, S, m, n, k, lda, ldw, ldy, in_dtype, out_dtype);
}
Problem make_rs(const void *const *X, int ldx, const void *const *W, int ldw, int S, int m, int n, int k,
                void *const *Y, int ldy, int in_dtype, int out_dtype = MS_DTYPE_F32) {
  return make_problem(RS, X, W, Y, S, 1, S, S, m, n, k, ldx, ldw, ldy, in_dtype, out_dtype);
}

}  // namespace

MS_API int ms_version(void) { return 100; }

MS_API const char *ms_last_error(void) { return g_err; }

MS_API long ms_query(int what) {
  if (what == MS_QUERY_MAX_SLICES) return MS_MAX_SLICES;
  if (what == MS_QUERY_LAST_LAUNCHES) return g_launches;
  if (what == MS_QUERY_LAST_VARIANT) return g_last_variant;
  if (what == MS_QUERY_LAST_SPLITS) return g_last_splits;
  if (what == MS_QUERY_LAST_GRID) return g_last_grid;
  DevInfo *d = nullptr;
  if (dev_info(&d) != MS_OK) return -1;
  switch (what) {
    case MS_QUERY_CU_COUNT: return d->cus;
    case MS_QUERY_CLOCK_KHZ: return d->clock_khz;
    case MS_QUERY_IS_GFX950: return d->gfx950;
    case MS_QUERY_LDS_BYTES: return d->lds;
    default: fail(MS_ERR_ARG, "ms_query: unknown selector %d", what); return -1;
  }
}

MS_API int ms_set_variant(int variant) {
  const int v = variant % 100, splits = variant / 100;
  const bool known = v == 0 || is_bf16_tile(v) || (v >= F32_FIRST && v <= F32_LAST) || (v == F32_WAVES && splits == 0);
  if (variant < 0 || !known || splits == 1 || splits > SPLIT_MAX) return fail(MS_ERR_ARG, "ms_set_variant: unknown variant %d", variant);
  g_variant = v;
  g_splits = splits;
  return MS_OK;
}

MS_API int ms_set_reserved_cus(int n) {
  if (n < 0 || n > 1024) return fail(MS_ERR_ARG, "ms_set_reserved_cus: %d out of range", n);
  g_reserved_cus = n;
  return MS_OK;
}

// Scratch of the entry point that allocates nothing (ms_gemm_os_noalloc): a split-contraction workspace that lives in
// the code object.  Every device the library runs on holds its own copy, at its own address, until the process ends; the
// name below is only a handle for hipGetSymbolAddress, host code never passes it to a kernel.
constexpr size_t NOALLOC_SCRATCH_BYTES = WS_HEADER_BYTES + (size_t)256 * 256 * 192 * sizeof(float);   // 256 partial tiles of 256 x 192
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

namespace {
struct ScratchAddr {
  std::mutex lock;
  void *ptr = nullptr;             // device address of `scratch` on this device, once looked up
  hipStream_t last_stream = nullptr;
  bool used = false;               // a call has used the scratch on last_stream
};
ScratchAddr g_scratch[64];

// The scratch entry of the calling thread's current device; its address is looked up with that device current on the
// first call that gets an answer (a failed look-up is reported and tried again by the next call).
int scratch_address(ScratchAddr **entry) {
  int d = 0;
  MS_HIP(hipGetDevice(&d));
  if (d < 0 || d >= 64) return fail(MS_ERR_HIP, "device ordinal %d out of range", d);
  ScratchAddr &sa = g_scratch[d];
  std::lock_guard<std::mutex> hold(sa.lock);
  if (!sa.ptr) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return fail(MS_ERR_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    sa.ptr = p;
  }
  *entry = &sa;
  return MS_OK;
}

__global__ void ws_clear_kernel(int *counters, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) counters[i] = 0;
}
}  // namespace

MS_API size_t ms_workspace_bytes(void) {
  DevInfo *d = nullptr;
  if (dev_info(&d) != MS_OK) return 0;
  // one partial tile of the largest shape (256 x 384 fp32) per compute unit
  return WS_HEADER_BYTES + (size_t)d->cus * 256 * 384 * sizeof(float);
}

MS_API int ms_workspace_init(void *workspace, size_t bytes, void *stream) {
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255) || bytes < WS_HEADER_BYTES)
    return fail(MS_ERR_ARG, "ms_workspace_init: a workspace must be 256-byte aligned and hold at least %zu bytes", WS_HEADER_BYTES);
  // a fill kernel, not hipMemsetAsync, so that the call may be captured into a HIP graph
  hipLaunchKernelGGL(ws_clear_kernel, dim3(WS_COUNTERS / 256), dim3(256), 0, (hipStream_t)stream, static_cast<int *>(workspace), WS_COUNTERS);
  MS_HIP(hipGetLastError());
  return MS_OK;
}

MS_API int ms_gemm_os(const void *const *A_slices, const void *const *B_slices, int S, int m, int n, int k_slice,
                      int lda, int ldb, void *C, int ldc, int in_dtype, int out_dtype, void *stream) {
  void *c1[1] = {C};
  return run(make_os(A_slices, B_slices, S, m, n, k_slice, lda, ldb, c1, ldc, in_dtype, out_dtype), stream);
}

MS_API int ms_gemm_os_fused(const void *const *A_slices, const void *const *B_slices, int S, int m, int n, int k_slice,
                            int lda, int ldb, void *C, int ldc, int in_dtype, int out_dtype, int activation,
                            const void *residual, int ldr, float *row_sum, float *row_sumsq, void *stream) {
  void *c1[1] = {C};
  Problem p = make_os(A_slices, B_slices, S, m, n, k_slice, lda, ldb, c1, ldc, in_dtype, out_dtype);
  p.act = activation; p.res = residual; p.ldr = ldr; p.row_sum = row_sum; p.row_sumsq = row_sumsq;
  return run(p, stream);
}

MS_API int ms_gemm_os_ws(const void *const *A_slices, const void *const *B_slices, int S, int m, int n, int k_slice,
                         int lda, int ldb, void *C, int ldc, int in_dtype, int out_dtype, int activation,
                         const void *residual, int ldr, float *row_sum, float *row_sumsq,
                         void *workspace, size_t workspace_bytes, void *stream) {
  void *c1[1] = {C};
  Problem p = make_os(A_slices, B_slices, S, m, n, k_slice, lda, ldb, c1, ldc, in_dtype, out_dtype);
  p.act = activation; p.res = residual; p.ldr = ldr; p.row_sum = row_sum; p.row_sumsq = row_sumsq;
  p.ws = workspace; p.ws_bytes = workspace ? workspace_bytes : 0;
  return run(p, stream);
}

// The slices of W in place: slice s begins at row 8 s and its blocks of eight rows lie S blocks apart, which for a kernel that loads
// whole rows is another step between blocks of rows, not another access pattern.
MS_API int ms_gemm_os_cyclic(const void *const *A_slices, const void *W, int S, int m, int n, int k_slice, int lda, int ldw, void *C, int ldc,
                             int in_dtype, int out_dtype, void *workspace, size_t workspace_bytes, void *stream) {
  const char *fn = "ms_gemm_os_cyclic";
  if (S < 1 || S > MS_MAX_SLICES) return fail(MS_ERR_ARG, "%s: S = %d outside [1, %d]", fn, S, MS_MAX_SLICES);
  const long long es = in_dtype == MS_DTYPE_BF16 ? 2 : 4;
  if (k_slice <= 0 || k_slice % 8) return fail(MS_ERR_ARG, "%s: k_slice = %d is not a number of blocks of eight rows", fn, k_slice);
  if (ldw < 0 || (long long)k_slice * S * ldw * es > 0x7FFFFFFFLL) return fail(MS_ERR_UNSUPPORTED, "%s: W spans 2 GiB or more", fn);
  // (a K step's loads reach up to eight blocks of rows on, with 32-bit offsets also where the slice has fewer: wrapped around they would
  // fetch some of its rows a second time, against zeros, which infinities turn into NaN)
  if ((long long)S * 8 * ldw * es * 8 > 0x100000000LL) return fail(MS_ERR_UNSUPPORTED, "%s: eight blocks of a slice's rows span more than 4 GiB of W", fn);
  const void *b[MS_MAX_SLICES];
  for (int s = 0; s < S; s++) b[s] = W ? static_cast<const char *>(W) + (long long)s * 8 * ldw * es : nullptr;
  void *c1[1] = {C};
  Problem p = make_os(A_slices, b, S, m, n, k_slice, lda, ldw, c1, ldc, in_dtype, out_dtype);
  p.b_blk = (int)((long long)S * 8 * ldw * es);
  p.ws = workspace; p.ws_bytes = workspace ? workspace_bytes : 0;
  return run(p, stream);
}

__global__ void signal_set_kernel(unsigned *flag, unsigned value) {
  // everything enqueued on the stream before this kernel has ended; the release makes it visible to whoever then reads the flag
  __hip_atomic_store(flag, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// the gate's half of a Problem: the flags, and the longest wait for one of them in ticks of wall_clock64()
namespace {
int set_gate(Problem &p, unsigned *slice_ready, unsigned timeout_ms, const char *fn) {
  if (!slice_ready || (reinterpret_cast<uintptr_t>(slice_ready) & 3))
    return fail(MS_ERR_ARG, "%s: slice_ready must be a 4-byte aligned device pointer to S + 1 words", fn);
  if (timeout_ms == 0 || timeout_ms > 60000) return fail(MS_ERR_ARG, "%s: timeout_ms %u outside [1, 60000]", fn, timeout_ms);
  p.slice_ready = slice_ready;
  int device = 0, wall_khz = 0;
  MS_HIP(hipGetDevice(&device));
  MS_HIP(hipDeviceGetAttribute(&wall_khz, hipDeviceAttributeWallClockRate, device));
  p.gate_ticks = (unsigned long long)timeout_ms * (unsigned long long)(wall_khz > 0 ? wall_khz : 100000);
  return MS_OK;
}
}  // namespace

MS_API int ms_gemm_os_gated(const void *const *A_slices, const void *const *B_slices, int S, int m, int n, int k_slice,
                            int lda, int ldb, void *C, int ldc, int in_dtype, int out_dtype,
                            void *workspace, size_t workspace_bytes, unsigned *slice_ready, unsigned timeout_ms, void *stream) {
  void *c1[1] = {C};
  Problem p = make_os(A_slices, B_slices, S, m, n, k_slice, lda, ldb, c1, ldc, in_dtype, out_dtype);
  p.ws = workspace; p.ws_bytes = workspace ? workspace_bytes : 0;
  const int rc = set_gate(p, slice_ready, timeout_ms, "ms_gemm_os_gated");
  return rc ? rc : run(p, stream);
}

MS_API int ms_signal_set(unsigned *flag, unsigned value, void *stream) {
  if (!flag || (reinterpret_cast<uintptr_t>(flag) & 3)) return fail(MS_ERR_ARG, "ms_signal_set: flag must be a 4-byte aligned device pointer");
  hipLaunchKernelGGL(signal_set_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, flag, value);
  MS_HIP(hipGetLastError());
  return MS_OK;
}

MS_API int ms_gemm_os_noalloc(const void *const *A_slices, const void *const *B_slices, int S, int m, int n, int k_slice,
                              int lda, int ldb, void *C, int ldc, int in_dtype, int out_dtype, void *stream) {
  void *c1[1] = {C};
  Problem p = make_os(A_slices, B_slices, S, m, n, k_slice, lda, ldb, c1, ldc, in_dtype, out_dtype);
  int rc = validate(p);
  if (rc) return rc;
  DevInfo *dev = nullptr;
  rc = dev_info(&dev);
  if (rc) return rc;
  // what the library would do with room to spare decides whether the built-in scratch is needed, and whether it is enough
  p.ws = reinterpret_cast<void *>(uintptr_t(256));    // stands for "a workspace": only its size is looked at here
  p.ws_bytes = g_variant ? ~size_t(0) : NOALLOC_SCRATCH_BYTES;      // (the library's own choice is one that fits)
  int splits = 1, bm = 0, bn = 0;
  if (in_dtype == MS_DTYPE_BF16) {
    const Pick want = is_bf16_tile(g_variant) ? Pick{g_variant, g_splits > 1 ? g_splits : 1, 0.0} : pick_variant(p, usable(*dev));
    splits = want.splits; bm = TILE_OF[want.v].bm; bn = TILE_OF[want.v].bn;
  } else {
    const F32Pick want = pick_f32(p, usable(*dev));
    splits = want.id ? want.splits : 1;
    for (const F32Tile &t : F32_TILES) if (t.id == want.id) { bm = t.bm; bn = t.bn; }
  }
  if (splits <= 1) {
    // an unsplit product exchanges nothing (without a workspace the library makes the same choice: splits are only ever added,
    // and products that SMALL_OS_MAX_K keeps off the 64x64 tile split, all of 200000 drawn ones)
    p.ws = nullptr;
    p.ws_bytes = 0;
    return run(p, stream);
  }
  const size_t tiles = (size_t)((m + bm - 1) / bm) * ((n + bn - 1) / bn);
  const size_t need = WS_HEADER_BYTES + tiles * splits * bm * bn * sizeof(float);
  if (need > NOALLOC_SCRATCH_BYTES)
    return fail(MS_ERR_UNSUPPORTED, "ms_gemm_os_noalloc: this product (m=%d n=%d k=%d x %d slices) would exchange %zu bytes of partial "
                "tiles, the built-in scratch holds %zu; use ms_gemm_os_ws with a workspace of ms_workspace_bytes()",
                m, n, k_slice, S, need, NOALLOC_SCRATCH_BYTES);
  ScratchAddr *sa = nullptr;
  rc = scratch_address(&sa);
  if (rc) return rc;
  // A product that splits leaves counters and partial tiles in the one array of its device, so two such calls must not
  // overlap.  Calls on one stream never do.  A call that comes on ANOTHER stream than the array's previous user first
  // waits for the device to go idle (hipDeviceSynchronize: allocates nothing), and the entry stays locked until this
  // call's kernels are queued, so eager calls from several streams or host threads cannot meet in the array.  A stream
  // under capture launches nothing now and cannot be waited for: how replays of such a graph are ordered against the
  // array's other users is the caller's business.
  std::lock_guard<std::mutex> hold(sa->lock);
  hipStream_t st = (hipStream_t)stream;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  MS_HIP(hipStreamIsCapturing(st, &capturing));
  if (capturing == hipStreamCaptureStatusNone) {
    if (sa->used && sa->last_stream != st) MS_HIP(hipDeviceSynchronize());
    sa->last_stream = st;
    sa->used = true;
  }
  p.ws = sa->ptr;
  p.ws_bytes = NOALLOC_SCRATCH_BYTES;
  // the array keeps what the last call left: the counters must start at zero (a fill kernel, so that the call can be captured)
  hipLaunchKernelGGL(ws_clear_kernel, dim3(WS_COUNTERS / 256), dim3(256), 0, st, static_cast<int *>(sa->ptr), WS_COUNTERS);
  MS_HIP(hipGetLastError());
  return run(p, stream);
}

MS_API int ms_gemm_ls(const void *A, int lda, const void *const *W_slices, int ldw, int S, int m, int n_slice, int k,
                      float *const *Y_chunks, int ldy, int in_dtype, void *stream) {
  const void *a1[1] = {A};
  return run(make_ls(a1, lda, W_slices, ldw, S, m, n_slice, k, (void *const *)Y_chunks, ldy, in_dtype), stream);
}

MS_API int ms_gemm_rs(const void *const *X_slices, int ldx, const void *W, int ldw, int S, int m_slice, int n, int k,
                      float *const *Y_chunks, int ldy, int in_dtype, void *stream) {
  const void *w1[1] = {W};
  return run(make_rs(X_slices, ldx, w1, ldw, S, m_slice, n, k, (void *const *)Y_chunks, ldy, in_dtype), stream);
}

MS_API int ms_gemm_ls_ex(const void *A, int lda, const void *const *W_slices, int ldw, int S, int m, int n_slice, int k,
                         void *const *Y_chunks, int ldy, int in_dtype, int out_dtype, void *stream) {
  const void *a1[1] = {A};
  return run(make_ls(a1, lda, W_slices, ldw, S, m, n_slice, k, Y_chunks, ldy, in_dtype, out_dtype), stream);
}

// W's slices in place, as ms_gemm_os_cyclic has B's: for a kernel that loads rows of the contraction, too, another step between blocks of
// rows (one device of a 2x4 mesh, 4096 x 4096 x 8192 in eight slices: 44 us with the slices cut out first, 35 without)
MS_API int ms_gemm_ls_cyclic(const void *A, int lda, const void *W, int ldw, int S, int m, int n_slice, int k,
                             void *const *Y_chunks, int ldy, int in_dtype, int out_dtype, void *stream) {
  const char *fn = "ms_gemm_ls_cyclic";
  if (S < 1 || S > MS_MAX_SLICES) return fail(MS_ERR_ARG, "%s: S = %d outside [1, %d]", fn, S, MS_MAX_SLICES);
  const long long es = in_dtype == MS_DTYPE_BF16 ? 2 : 4;
  if (n_slice <= 0 || n_slice % 8) return fail(MS_ERR_ARG, "%s: n_slice = %d is not a number of blocks of eight rows", fn, n_slice);
  if (ldw < 0 || (long long)n_slice * S * ldw * es > 0x7FFFFFFFLL) return fail(MS_ERR_UNSUPPORTED, "%s: W spans 2 GiB or more", fn);
  const void *a1[1] = {A}, *w[MS_MAX_SLICES];
  for (int s = 0; s < S; s++) w[s] = W ? static_cast<const char *>(W) + (long long)s * 8 * ldw * es : nullptr;
  Problem p = make_ls(a1, lda, w, ldw, S, m, n_slice, k, Y_chunks, ldy, in_dtype, out_dtype);
  p.b_blk = (int)((long long)S * 8 * ldw * es);
  return run(p, stream);
}

MS_API int ms_gemm_rs_ex(const void *const *X_slices, int ldx, const void *W, int ldw, int S, int m_slice, int n, int k,
                         void *const *Y_chunks, int ldy, int in_dtype, int out_dtype, void *stream) {
  const void *w1[1] = {W};
  return run(make_rs(X_slices, ldx, w1, ldw, S, m_slice, n, k, Y_chunks, ldy, in_dtype, out_dtype), stream);
}

// The chunk-producing products of several mesh devices in one launch: device p's S chunks are chunks p * S .. of one call
// whose stationary operand has an entry for every chunk.  The devices of a mesh line have equal shapes, and one of them alone
// often leaves compute units idle (see the header).
namespace {
int spread_over_chunks(const void *const *per_device, int P, int S, const void **per_chunk, const char *fn) {
  if (P < 1 || S < 1 || (long)P * S > MS_MAX_SLICES) return fail(MS_ERR_ARG, "%s: P * S = %d * %d outside [1, %d]", fn, P, S, MS_MAX_SLICES);
  if (!per_device) return fail(MS_ERR_ARG, "%s: null pointer table", fn);
  for (int c = 0; c < P * S; c++) per_chunk[c] = per_device[c / S];
  return MS_OK;
}
}  // namespace

MS_API int ms_gemm_ls_peers(const void *const *A, int lda, const void *const *W_slices, int ldw, int P, int S, int m, int n_slice, int k,
                            void *const *Y_chunks, int ldy, int in_dtype, int out_dtype, void *stream) {
  const void *a[MS_MAX_SLICES];
  if (int rc = spread_over_chunks(A, P, S, a, "ms_gemm_ls_peers")) return rc;
  return run(make_problem(LS, a, W_slices, Y_chunks, P * S, P * S, P * S, P * S, m, n_slice, k, lda, ldw, ldy, in_dtype, out_dtype), stream);
}

MS_API int ms_gemm_rs_peers(const void *const *X_slices, int ldx, const void *const *W, int ldw, int P, int S, int m_slice, int n, int k,
                            void *const *Y_chunks, int ldy, int in_dtype, int out_dtype, void *stream) {
  const void *w[MS_MAX_SLICES];
  if (int rc = spread_over_chunks(W, P, S, w, "ms_gemm_rs_peers")) return rc;
  return run(make_problem(RS, X_slices, w, Y_chunks, P * S, P * S, P * S, P * S, m_slice, n, k, ldx, ldw, ldy, in_dtype, out_dtype), stream);
}

// The same products with the devices' partial sums added up on the way out instead of in chunks through memory (see the header).
namespace {
int run_sum(Problem p, void *workspace, size_t workspace_bytes, void *stream, const char *fn) {
  if (p.S < 1 || p.S > MS_MAX_SLICES) return fail(MS_ERR_ARG, "%s: P = %d outside [1, %d]", fn, p.S, MS_MAX_SLICES);
  if (p.in_dtype != MS_DTYPE_BF16 || p.out_dtype != MS_DTYPE_BF16) return fail(MS_ERR_UNSUPPORTED, "%s: bf16 operands and results only", fn);
  p.sum = p.S > 1;      // (one device's partial sum is its product)
  if (p.sum) { p.ws = workspace; p.ws_bytes = workspace ? workspace_bytes : 0; }
  return run(p, stream);
}
}  // namespace

// Whether the sum over a mesh line of P devices is priced lower in registers (one launch on the tiles that carry it) than in fp32 chunks that a
// layout kernel adds up (the chunk product on any tile, its chunks out and in again, the copy of the operand that is sliced or gathered for
// it, two more launches).  The first is one workgroup a tile for the whole contraction (or one a device, for a few line lengths): few output
// tiles under a long contraction leave the device idle, which P times as many chunk tiles do not; and its tiles are slower per FLOP than
// the 256x384 one, which counts where the contraction makes up for the chunks' bytes.  Measured on 1404 products drawn and listed (m and n
// 64 to 16384, 64 to 24576 contraction elements a device, 2 to 16 devices, one to eight slices), registers -> chunks: RS 256 x 640 of sixteen
// devices of 12864 elements 1699 -> 180 us, 1024 x 4096 of four of 16384 589 -> 454, 8192 x 12288 of two of 8192 2645 -> 2409; RS 3072 x 12288
// x 1024 of two 76 <- 149, LS 8192 x 8192 of two of 8192 1696 <- 1713.  The choice takes 1.003 of the better one's time in the geometric mean
// and 1.14 at the 99th percentile (1.001 and at most 1.17 on 600 products that it was not fitted to); registers always would take 1.048 and 3.5,
// chunks always 1.86.  Up to SUM_ALWAYS_K contraction elements of the whole line registers were never behind.
namespace {
constexpr long SUM_ALWAYS_K = 10240;
constexpr double SUM_UNIT_US = 3.5e-7;                                       // pick_variant's unit
constexpr double SUM_SCALE = 0.93, SUM_LAUNCH_US = 3.0;
constexpr double SUM_RS_PART_LINES = 0.08;                                   // RS rows that are no whole 128-byte lines: half of it for each operand
constexpr double SUM_COLD_US_PER_MB = 0.05;                                  // operands beyond the 256 MB of the last-level cache
constexpr double CHUNK_SCALE = 0.95, CHUNK_LAUNCHES_US = 30.0;
constexpr double CHUNK_US_PER_MB = 0.33, CHUNK_COPY_US_PER_MB = 0.3;         // chunk bytes out and in; the operand that is copied
// the host's part of the chunk path, which a stream of such calls cannot go below
constexpr double CHUNK_HOST_US = 35.0, CHUNK_HOST_PEER_US = 5.0, CHUNK_HOST_SLICE_US = 2.6;
constexpr double CHUNK_MARGIN = 0.93;                                        // chunks are taken where they are this much cheaper
}  // namespace

MS_API int ms_prefers_sum(int rs, int P, int S, int m, int n, int k) {
  if (P < 2 || P > MS_MAX_SLICES || S < 1 || (long)P * S > MS_MAX_SLICES || m < 1 || n < 1 || k < 1 || (rs ? m : n) % S) return 1;
  if (is_bf16_tile(g_variant)) return carries_sum(g_variant);      // (a forced tile is the one that runs)
  if ((long)P * k <= SUM_ALWAYS_K) return 1;
  DevInfo *dev = nullptr;
  if (dev_info(&dev) != MS_OK) return 1;
  const DevFacts facts = usable(*dev);
  Problem p;
  p.flow = rs ? RS : LS;
  p.in_dtype = MS_DTYPE_BF16; p.K = k;
  Problem chunks = p;
  p.sum = true; p.S = P; p.M = m; p.N = n; p.out_dtype = MS_DTYPE_BF16;
  p.ws = reinterpret_cast<void *>(uintptr_t(256));      // stands for "a workspace", as in ms_gemm_os_noalloc
  p.ws_bytes = WS_HEADER_BYTES + (size_t)dev->cus * 256 * 384 * sizeof(float);
  chunks.S = P * S; chunks.M = rs ? m / S : m; chunks.N = rs ? n : n / S; chunks.out_dtype = MS_DTYPE_F32;
  const double mb = 1e-6, part_lines = rs ? 0.5 * ((m % 64 != 0) + (n % 64 != 0)) : 0.0;
  const double operands = 2.0 * ((double)m + n) * P * k, copied = 2.0 * (rs ? m : n) * (double)P * k, chunk_bytes = 4.0 * P * (double)m * n;
  const double cold = operands > 256e6 ? operands - 256e6 : 0.0;
  // (chunks run on the 64-row tiles as well where those are faster, but the constants were fitted to their price without: the choice errs to the side of registers)
  const double sum_us = pick_variant(p, facts).cost * P * k * SUM_UNIT_US * SUM_SCALE * (1.0 + SUM_RS_PART_LINES * part_lines) + SUM_LAUNCH_US + cold * mb * SUM_COLD_US_PER_MB;
  double chunks_us = pick_variant(chunks, facts, false).cost * k * SUM_UNIT_US * CHUNK_SCALE + chunk_bytes * mb * CHUNK_US_PER_MB + copied * mb * CHUNK_COPY_US_PER_MB + CHUNK_LAUNCHES_US;
  const double host_us = CHUNK_HOST_US + P * (CHUNK_HOST_PEER_US + CHUNK_HOST_SLICE_US * (S - 1));
  if (host_us > chunks_us) chunks_us = host_us;
  return chunks_us < CHUNK_MARGIN * sum_us ? 0 : 1;
}

MS_API int ms_gemm_ls_sum(const void *const *A, int lda, const void *const *W, int ldw, int P, int m, int n, int k, void *C, int ldc,
                          int in_dtype, int out_dtype, void *workspace, size_t workspace_bytes, void *stream) {
  void *c1[1] = {C};
  return run_sum(make_problem(LS, A, W, c1, P, P, 1, P, m, n, k, lda, ldw, ldc, in_dtype, out_dtype), workspace, workspace_bytes, stream, "ms_gemm_ls_sum");
}

MS_API int ms_gemm_rs_sum(const void *const *X, int ldx, const void *const *W, int ldw, int P, int m, int n, int k, void *C, int ldc,
                          int in_dtype, int out_dtype, void *workspace, size_t workspace_bytes, void *stream) {
  void *c1[1] = {C};
  return run_sum(make_problem(RS, X, W, c1, P, P, 1, P, m, n, k, ldx, ldw, ldc, in_dtype, out_dtype), workspace, workspace_bytes, stream, "ms_gemm_rs_sum");
}

// the chunk-producing calls with completion counters
namespace {
int run_signal(Problem p, unsigned *chunk_done, int *tiles_per_chunk, void *stream, const char *fn) {
  if (!chunk_done || !tiles_per_chunk) return fail(MS_ERR_ARG, "%s: null chunk_done / tiles_per_chunk", fn);
  if (reinterpret_cast<uintptr_t>(chunk_done) & 3) return fail(MS_ERR_ARG, "%s: chunk_done must be 4-byte aligned", fn);
  p.chunk_done = chunk_done;
  const int rc = run(p, stream);
  if (rc == MS_OK) *tiles_per_chunk = g_last_tiles_per_chunk;
  return rc;
}
}  // namespace

MS_API int ms_gemm_ls_signal(const void *A, int lda, const void *const *W_slices, int ldw, int S, int m, int n_slice, int k,
                             void *const *Y_chunks, int ldy, int in_dtype, int out_dtype,
                             unsigned *chunk_done, int *tiles_per_chunk, void *stream) {
  const void *a1[1] = {A};
  return run_signal(make_ls(a1, lda, W_slices, ldw, S, m, n_slice, k, Y_chunks, ldy, in_dtype, out_dtype), chunk_done, tiles_per_chunk, stream, "ms_gemm_ls_signal");
}

MS_API int ms_gemm_rs_signal(const void *const *X_slices, int ldx, const void *W, int ldw, int S, int m_slice, int n, int k,
                             void *const *Y_chunks, int ldy, int in_dtype, int out_dtype,
                             unsigned *chunk_done, int *tiles_per_chunk, void *stream) {
  const void *w1[1] = {W};
  return run_signal(make_rs(X_slices, ldx, w1, ldw, S, m_slice, n, k, Y_chunks, ldy, in_dtype, out_dtype), chunk_done, tiles_per_chunk, stream, "ms_gemm_rs_signal");
}

// the chunk-producing calls behind the input gate; the completion counters are optional here
namespace {
int run_chunks_gated(Problem p, unsigned *chunk_done, int *tiles_per_chunk, unsigned *slice_ready, unsigned timeout_ms, void *stream, const char *fn) {
  if ((chunk_done == nullptr) != (tiles_per_chunk == nullptr)) return fail(MS_ERR_ARG, "%s: chunk_done and tiles_per_chunk come together or not at all", fn);
  const int rc = set_gate(p, slice_ready, timeout_ms, fn);
  if (rc) return rc;
  return chunk_done ? run_signal(p, chunk_done, tiles_per_chunk, stream, fn) : run(p, stream);
}
}  // namespace

MS_API int ms_gemm_ls_gated(const void *A, int lda, const void *const *W_slices, int ldw, int S, int m, int n_slice, int k,
                            void *const *Y_chunks, int ldy, int in_dtype, int out_dtype,
                            unsigned *chunk_done, int *tiles_per_chunk, unsigned *slice_ready, unsigned timeout_ms, void *stream) {
  const void *a1[1] = {A};
  return run_chunks_gated(make_ls(a1, lda, W_slices, ldw, S, m, n_slice, k, Y_chunks, ldy, in_dtype, out_dtype), chunk_done, tiles_per_chunk,
                          slice_ready, timeout_ms, stream, "ms_gemm_ls_gated");
}

MS_API int ms_gemm_rs_gated(const void *const *X_slices, int ldx, const void *W, int ldw, int S, int m_slice, int n, int k,
                            void *const *Y_chunks, int ldy, int in_dtype, int out_dtype,
                            unsigned *chunk_done, int *tiles_per_chunk, unsigned *slice_ready, unsigned timeout_ms, void *stream) {
  const void *w1[1] = {W};
  return run_chunks_gated(make_rs(X_slices, ldx, w1, ldw, S, m_slice, n, k, Y_chunks, ldy, in_dtype, out_dtype), chunk_done, tiles_per_chunk,
                          slice_ready, timeout_ms, stream, "ms_gemm_rs_gated");
}

MS_API int ms_time_os(const void *const *A_slices, const void *const *B_slices, int S, int m, int n, int k_slice,
                      int lda, int ldb, void *C, int ldc, int in_dtype, int out_dtype, void *stream,
                      int warmup, int reps, float *ms_out) {
  void *c1[1] = {C};
  return timed(make_os(A_slices, B_slices, S, m, n, k_slice, lda, ldb, c1, ldc, in_dtype, out_dtype), stream, warmup, reps, ms_out);
}

MS_API int ms_time_os_ws(const void *const *A_slices, const void *const *B_slices, int S, int m, int n, int k_slice,
                         int lda, int ldb, void *C, int ldc, int in_dtype, int out_dtype,
                         void *workspace, size_t workspace_bytes, void *stream, int warmup, int reps, float *ms_out) {
  void *c1[1] = {C};
  Problem p = make_os(A_slices, B_slices, S, m, n, k_slice, lda, ldb, c1, ldc, in_dtype, out_dtype);
  p.ws = workspace; p.ws_bytes = workspace ? workspace_bytes : 0;
  return timed(p, stream, warmup, reps, ms_out);
}

MS_API int ms_time_ls_ex(const void *A, int lda, const void *const *W_slices, int ldw, int S, int m, int n_slice, int k,
                         void *const *Y_chunks, int ldy, int in_dtype, int out_dtype, void *stream,
                         int warmup, int reps, float *ms_out) {
  const void *a1[1] = {A};
  return timed(make_ls(a1, lda, W_slices, ldw, S, m, n_slice, k, Y_chunks, ldy, in_dtype, out_dtype), stream, warmup, reps, ms_out);
}

MS_API int ms_time_rs_ex(const void *const *X_slices, int ldx, const void *W, int ldw, int S, int m_slice, int n, int k,
                         void *const *Y_chunks, int ldy, int in_dtype, int out_dtype, void *stream,
                         int warmup, int reps, float *ms_out) {
  const void *w1[1] = {W};
  return timed(make_rs(X_slices, ldx, w1, ldw, S, m_slice, n, k, Y_chunks, ldy, in_dtype, out_dtype), stream, warmup, reps, ms_out);
}

MS_API int ms_time_ls(const void *A, int lda, const void *const *W_slices, int ldw, int S, int m, int n_slice, int k,
                      float *const *Y_chunks, int ldy, int in_dtype, void *stream, int warmup, int reps, float *ms_out) {
  return ms_time_ls_ex(A, lda, W_slices, ldw, S, m, n_slice, k, (void *const *)Y_chunks, ldy, in_dtype, MS_DTYPE_F32, stream, warmup, reps, ms_out);
}

MS_API int ms_time_rs(const void *const *X_slices, int ldx, const void *W, int ldw, int S, int m_slice, int n, int k,
                      float *const *Y_chunks, int ldy, int in_dtype, void *stream, int warmup, int reps, float *ms_out) {
  return ms_time_rs_ex(X_slices, ldx, W, ldw, S, m_slice, n, k, (void *const *)Y_chunks, ldy, in_dtype, MS_DTYPE_F32, stream, warmup, reps, ms_out);
}
