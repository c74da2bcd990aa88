// libmeshslice_hip.so — C ABI over the block-cyclic layout kernels (declarations: include/meshslice_hip.h).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ms_common.hip.inc"

#include "ms_layout.hip.inc"

namespace {

using msi::fail;

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int elem_bytes(int dtype) { return dtype == MS_DTYPE_BF16 ? 2 : dtype == MS_DTYPE_F32 ? 4 : 0; }

// Threads along the row: the smallest of 64 / 128 / 256 that covers it.
int pick_tx(int ucols) { return ucols <= 64 ? 64 : ucols <= 128 ? 128 : 256; }

// Distance between consecutive table entries if it is the same (and not zero) for all of them, else 0.
long long table_stride(const void *const *tab, int n) {
  if (n < 2) return 0;
  const long long d = (long long)(reinterpret_cast<intptr_t>(tab[1]) - reinterpret_cast<intptr_t>(tab[0]));
  for (int i = 2; i < n; i++)
    if ((long long)(reinterpret_cast<intptr_t>(tab[i]) - reinterpret_cast<intptr_t>(tab[i - 1])) != d) return 0;
  return d;
}

// Rows per thread, 16-byte units: one.  A thread then has little in flight by itself, but the launch has eight times the
// blocks of eight rows, and these kernels live on loads in flight over the whole device.  S = 4 or 8 slices, eight rows per
// thread -> one: reducing four peers' fp32 chunks to a bf16 shard of 512 x 256 15.3 -> 3.9 us, 1024 x 768 18.4 -> 5.7,
// 2048 x 3072 30.2 -> 24.5, 4096 x 12288 171 -> 159; cutting 1024 x 768 bf16 3.3 -> 2.8, 4096 x 12288 35.3 -> 34.2 us.
// Two for what only moves (a cut, or one peer's chunks) in rows that leave a fifth of their waves' lanes idle, as long as
// that fills the device (512 blocks, two per compute unit): there the waves to start are what costs (one row, two, eight:
// 14427 x 72 fp32 cut in three 5.0, 4.3, 4.2 us; 12992 x 232 bf16 cut by rows 5.0, 4.4, 4.4; one peer's 15874 x 352 fp32 9.4,
// 8.6, 8.4).  Of 409 cuts from 16 x 64 to 16384 x 16384 one in forty is more than 3 % slower than with eight rows; with one row
// for all it was one in thirteen.
// Shards that move element by element take the largest count that fills the device: the two divisions per thread weigh most
// there (254 x 3536 bf16: one row 4.5, four 3.5, eight 3.7 us; 6984 x 7244 fp32 of four peers 304, 190, 190 us).
// More rows than the grid's second extent covers double the count.
constexpr int GRID_Y_MAX = 65535, FULL_BLOCKS = 512;
int rows_per_thread(int rows, int ucols, int tx, bool wide, bool moves) {
  const int rows_per_block = 256 / tx;
  const auto blocks_y = [&](int rt) { return ((long long)rows + rows_per_block * rt - 1) / (rows_per_block * rt); };
  const auto full = [&](int rt) { return blocks_y(rt) * ((ucols + tx - 1) / tx) >= FULL_BLOCKS; };
  int rt = 1;
  if (!wide) {
    for (rt = msk::LAYOUT_RT; rt > 1 && !full(rt);) rt /= 2;
  } else if (moves && 5LL * ucols < 4LL * ((ucols + 63) / 64 * 64) && full(2)) {
    rt = 2;
  }
  while (rt < msk::LAYOUT_RT && blocks_y(rt) > GRID_Y_MAX) rt *= 2;
  return rt;
}

int grid_for(int rows, int ucols, int tx, int rt, dim3 *g, const char *fn) {
  const int rows_per_block = (256 / tx) * rt;
  const long long gy = ((long long)rows + rows_per_block - 1) / rows_per_block;
  if (gy > GRID_Y_MAX) return fail(MS_ERR_UNSUPPORTED, "%s: %d rows exceed one launch", fn, rows);
  *g = dim3((unsigned)((ucols + tx - 1) / tx), (unsigned)gy, 1);
  return MS_OK;
}

template <int UB>
int launch_pack(int axis, int tx, int rt, dim3 g, hipStream_t st, const msk::PackArgs &a) {
#define MS_PACK(TX, RT)                                                                                  \
  if (tx == TX && rt == RT) {                                                                            \
    if (axis == 1) hipLaunchKernelGGL((msk::pack_cols_kernel<UB, TX, RT>), g, dim3(256), 0, st, a);      \
    else hipLaunchKernelGGL((msk::pack_rows_kernel<UB, TX, RT>), g, dim3(256), 0, st, a);                \
  }
  MS_PACK(64, 1) MS_PACK(128, 1) MS_PACK(256, 1)
  MS_PACK(64, 2) MS_PACK(128, 2) MS_PACK(256, 2)
  MS_PACK(64, 4) MS_PACK(128, 4) MS_PACK(256, 4)
  MS_PACK(64, 8) MS_PACK(128, 8) MS_PACK(256, 8)
#undef MS_PACK
  MS_HIP(hipGetLastError());
  return MS_OK;
}

template <typename TIN, typename TOUT, int VEC>
int launch_unpack(int axis, int tx, int rt, dim3 g, hipStream_t st, const msk::UnpackArgs &a) {
#define MS_UNPACK(TX, RT)                                                                                          \
  if (tx == TX && rt == RT) {                                                                                      \
    if (axis == 1) hipLaunchKernelGGL((msk::unpack_cols_kernel<TIN, TOUT, VEC, TX, RT>), g, dim3(256), 0, st, a);  \
    else hipLaunchKernelGGL((msk::unpack_rows_kernel<TIN, TOUT, VEC, TX, RT>), g, dim3(256), 0, st, a);            \
  }
  MS_UNPACK(64, 1) MS_UNPACK(128, 1) MS_UNPACK(256, 1)
  MS_UNPACK(64, 2) MS_UNPACK(128, 2) MS_UNPACK(256, 2)
  MS_UNPACK(64, 4) MS_UNPACK(128, 4) MS_UNPACK(256, 4)
  MS_UNPACK(64, 8) MS_UNPACK(128, 8) MS_UNPACK(256, 8)
#undef MS_UNPACK
  MS_HIP(hipGetLastError());
  return MS_OK;
}

template <int VEC>
int launch_unpack_typed(int in_dtype, int out_dtype, int axis, int tx, int rt, dim3 g, hipStream_t st, const msk::UnpackArgs &a) {
  typedef unsigned short bf16_bits;
  if (in_dtype == MS_DTYPE_F32)
    return out_dtype == MS_DTYPE_F32 ? launch_unpack<float, float, VEC>(axis, tx, rt, g, st, a) : launch_unpack<float, bf16_bits, VEC>(axis, tx, rt, g, st, a);
  return out_dtype == MS_DTYPE_F32 ? launch_unpack<bf16_bits, float, VEC>(axis, tx, rt, g, st, a) : launch_unpack<bf16_bits, bf16_bits, VEC>(axis, tx, rt, g, st, a);
}

}  // namespace

MS_API int ms_pack_slices(const void *src, int ld_src, int rows, int cols, int axis, int S, int B,
                          void *const *dst_slices, int ld_dst, int dtype, void *stream) {
  const char *fn = "ms_pack_slices";
  const int es = elem_bytes(dtype);
  if (!es) return fail(MS_ERR_UNSUPPORTED, "%s: unknown dtype %d", fn, dtype);
  if (axis != 0 && axis != 1) return fail(MS_ERR_ARG, "%s: axis must be 0 (rows) or 1 (columns), got %d", fn, axis);
  if (S < 1 || S > MS_MAX_SLICES) return fail(MS_ERR_ARG, "%s: S = %d outside [1, %d]", fn, S, MS_MAX_SLICES);
  if (B < 1 || rows <= 0 || cols <= 0) return fail(MS_ERR_ARG, "%s: non-positive extent (rows=%d cols=%d B=%d)", fn, rows, cols, B);
  if (!src || !dst_slices) return fail(MS_ERR_ARG, "%s: null pointer", fn);
  const int sliced = axis == 1 ? cols : rows;
  if (sliced % ((long long)S * B)) return fail(MS_ERR_ARG, "%s: sliced extent %d is not a multiple of S*B = %d*%d", fn, sliced, S, B);
  const int dcols = axis == 1 ? cols / S : cols;
  if (ld_src < cols || ld_dst < dcols) return fail(MS_ERR_ARG, "%s: leading dimension smaller than the row length", fn);
  bool wide = aligned16(src) && ((long long)cols * es) % 16 == 0 && ((long long)ld_src * es) % 16 == 0 && ((long long)ld_dst * es) % 16 == 0 &&
              (axis == 0 || (B * es) % 16 == 0);
  for (int s = 0; s < S; s++) {
    if (!dst_slices[s]) return fail(MS_ERR_ARG, "%s: slice pointer %d is null", fn, s);
    if (reinterpret_cast<uintptr_t>(dst_slices[s]) % es) return fail(MS_ERR_ARG, "%s: slice pointer %d is not aligned to the element size", fn, s);
    wide = wide && aligned16(dst_slices[s]);
  }
  if (reinterpret_cast<uintptr_t>(src) % es) return fail(MS_ERR_ARG, "%s: source pointer is not aligned to the element size", fn);
  const int ub = wide ? 16 : es;
  msk::PackArgs a;
  a.src = src;
  for (int s = 0; s < S; s++) a.dst[s] = dst_slices[s];
  a.rows = rows;
  a.ucols = (int)((long long)cols * es / ub);
  a.ld_src = (int)((long long)ld_src * es / ub);
  a.ld_dst = (int)((long long)ld_dst * es / ub);
  a.S = S;
  a.G = axis == 1 ? B * es / ub : B;
  a.tab_stride = table_stride(dst_slices, S);
  const int tx = pick_tx(a.ucols), rt = rows_per_thread(rows, a.ucols, tx, wide, true);
  dim3 g;
  if (int rc = grid_for(rows, a.ucols, tx, rt, &g, fn)) return rc;
  hipStream_t st = (hipStream_t)stream;
  return ub == 16 ? launch_pack<16>(axis, tx, rt, g, st, a) : ub == 4 ? launch_pack<4>(axis, tx, rt, g, st, a) : launch_pack<2>(axis, tx, rt, g, st, a);
}

MS_API int ms_unpack_chunks(const void *const *chunks, int P, int S, int ld_chunk, int row_off, int col_off,
                            int rows, int cols, int axis, int B, void *out, int ld_out,
                            int in_dtype, int out_dtype, void *stream) {
  const char *fn = "ms_unpack_chunks";
  const int esi = elem_bytes(in_dtype), eso = elem_bytes(out_dtype);
  if (!esi || !eso) return fail(MS_ERR_UNSUPPORTED, "%s: unknown dtype (%d, %d)", fn, in_dtype, out_dtype);
  if (axis != 0 && axis != 1) return fail(MS_ERR_ARG, "%s: axis must be 0 (rows) or 1 (columns), got %d", fn, axis);
  if (S < 1 || P < 1 || (long long)P * S > msk::LAYOUT_MAX_PTRS) return fail(MS_ERR_ARG, "%s: P*S = %d*%d outside [1, %d]", fn, P, S, msk::LAYOUT_MAX_PTRS);
  if (B < 1 || rows <= 0 || cols <= 0) return fail(MS_ERR_ARG, "%s: non-positive extent (rows=%d cols=%d B=%d)", fn, rows, cols, B);
  if (row_off < 0 || col_off < 0) return fail(MS_ERR_ARG, "%s: negative window offset", fn);
  if (!chunks || !out) return fail(MS_ERR_ARG, "%s: null pointer", fn);
  const int sliced = axis == 1 ? cols : rows;
  if (sliced % ((long long)S * B)) return fail(MS_ERR_ARG, "%s: interleaved extent %d is not a multiple of S*B = %d*%d", fn, sliced, S, B);
  const int wcols = axis == 1 ? cols / S : cols;  // columns of the window kept from each chunk
  if ((long long)col_off + wcols > ld_chunk || ld_out < cols) return fail(MS_ERR_ARG, "%s: leading dimension smaller than the row length", fn);
  bool wide = aligned16(out) && cols % 8 == 0 && col_off % 8 == 0 && ld_chunk % 8 == 0 && ld_out % 8 == 0 && (axis == 0 || B % 8 == 0);
  if (reinterpret_cast<uintptr_t>(out) % eso) return fail(MS_ERR_ARG, "%s: output pointer is not aligned to the element size", fn);
  msk::UnpackArgs a;
  for (int i = 0; i < P * S; i++) {
    if (!chunks[i]) return fail(MS_ERR_ARG, "%s: chunk pointer %d is null", fn, i);
    if (reinterpret_cast<uintptr_t>(chunks[i]) % esi) return fail(MS_ERR_ARG, "%s: chunk pointer %d is not aligned to the element size", fn, i);
    wide = wide && aligned16(chunks[i]);
    a.src[i] = chunks[i];
  }
  a.dst = out;
  a.rows = rows;
  // eight elements per thread, or the four of one 16-byte unit when fp32 chunks of one peer are only moved
  const bool move_f32 = wide && P == 1 && in_dtype == MS_DTYPE_F32 && out_dtype == MS_DTYPE_F32;
  const int vec = !wide ? 1 : move_f32 ? 4 : 8;
  a.ucols = cols / vec;
  a.ld_src = ld_chunk;
  a.ld_dst = ld_out;
  a.row_off = row_off;
  a.col_off = col_off;
  a.P = P;
  a.S = S;
  a.B = B;
  a.tab_stride = table_stride(chunks, P * S);
  const int tx = pick_tx(a.ucols), rt = rows_per_thread(rows, a.ucols, tx, wide, P == 1);
  dim3 g;
  if (int rc = grid_for(rows, a.ucols, tx, rt, &g, fn)) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (move_f32) return launch_unpack<float, float, 4>(axis, tx, rt, g, st, a);
  return wide ? launch_unpack_typed<8>(in_dtype, out_dtype, axis, tx, rt, g, st, a) : launch_unpack_typed<1>(in_dtype, out_dtype, axis, tx, rt, g, st, a);
}
