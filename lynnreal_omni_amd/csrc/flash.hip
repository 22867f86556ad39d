// flash.hip - Flash token selection: row gather, residual restore and the
// nearest-anchor search of the selection layout.
//
// Restates model/flash.py:6-33 (spatial_layout: each dropped video row maps to
// its nearest retained row of the same time step) and :71-85 (compress: the
// hidden rows, adaLN indices and rotary rows of the kept tokens are selected
// before the compressed blocks; restore: full + gain * (current - input),
// gathered back through the inverse map, before the first full block).
//
// All three are HBM-bound (the search is a small O(dropped x anchors) pass
// over positions that sit in LDS). Rows are moved as 16-byte chunks by one
// 256-thread block per output row.
#include "lr_device.h"
#include "lr_runtime.h"

namespace lr {
namespace {

constexpr int kThreads = 256;

// -------------------------------------------------------------- gather ----
// dst[o, i, :] = src[o, index[i], :] for rows of `units` 16-byte chunks.
// Indices past the source are clamped (the callers' maps are in range by
// construction; the clamp keeps a bad map inside the buffer).
// One block per output row; all of a thread's chunks are loaded before the first
// is stored (rows of up to CPT * 256 chunks). A row's bytes are the bound: 3683 of
// 12605 rows of 10240 bytes 15.4 -> 15.1 us, of 16384 bytes 23.4 -> 22.6 us,
// against one chunk at a time. One source needs no division.
template <int CPT>
__global__ __launch_bounds__(kThreads) void gather_rows16(const uint4* __restrict__ src,
                                                          const int64_t* __restrict__ index,
                                                          uint4* __restrict__ dst, int64_t src_rows,
                                                          int64_t dst_rows, int64_t units) {
  const int64_t r = blockIdx.x;  // output row over [outer, dst_rows]
  const int64_t o = r < dst_rows ? 0 : r / dst_rows, i = r - o * dst_rows;
  const int64_t s = clamp_index(index[i], src_rows);
  const auto from = row_rsrc(src + (o * src_rows + s) * units, 16 * units);
  const auto to = row_rsrc(dst + r * units, 16 * units);
  uint4 v[CPT];
#pragma unroll
  for (int c = 0; c < CPT; ++c) v[c] = buf_load16(from, 16u * threadIdx.x, 4096u * c);
#pragma unroll
  for (int c = 0; c < CPT; ++c) buf_store16_nt(to, 16u * threadIdx.x + 4096u * c, v[c]);
}

// One chunk at a time: rows wider than that, and rows of at most one chunk per
// thread, where there is nothing to overlap (2048 bytes: 5.1 us, 5.4 with CPT 1).
__global__ __launch_bounds__(kThreads) void gather_rows16_loop(const uint4* __restrict__ src,
                                                               const int64_t* __restrict__ index,
                                                               uint4* __restrict__ dst, int64_t src_rows,
                                                               int64_t dst_rows, int64_t units) {
  const int64_t r = blockIdx.x;
  const int64_t o = r / dst_rows, i = r - o * dst_rows;
  const int64_t s = clamp_index(index[i], src_rows);
  const uint4* from = src + (o * src_rows + s) * units;
  uint4* to = dst + r * units;
  for (int64_t u = threadIdx.x; u < units; u += kThreads) store_nt(to + u, load_nt(from + u));
}

// Narrow rows (rotary rows): one thread per 16 bytes, several rows per block, and
// 32-bit index arithmetic (total < 2^31). 3683 of 12605 rows of 256 bytes: 3.4 us,
// 3.8 with a block per row; the launch itself is about 3.
__global__ __launch_bounds__(kThreads) void gather_rows16_narrow(const uint4* __restrict__ src,
                                                                 const int64_t* __restrict__ index,
                                                                 uint4* __restrict__ dst,
                                                                 int64_t src_rows, uint32_t dst_rows,
                                                                 uint32_t units, uint32_t total) {
  const uint32_t e = blockIdx.x * (uint32_t)kThreads + threadIdx.x;
  if (e >= total) return;
  const uint32_t r = e / units, c = e - r * units;
  const uint32_t o = r / dst_rows, i = r - o * dst_rows;
  const int64_t s = clamp_index(index[i], src_rows);
  dst[e] = src[((int64_t)o * src_rows + s) * units + c];
}

// Any row width: one thread per byte, rows of `width` bytes.
__global__ __launch_bounds__(kThreads) void gather_rows_bytes(const uint8_t* __restrict__ src,
                                                              const int64_t* __restrict__ index,
                                                              uint8_t* __restrict__ dst,
                                                              int64_t src_rows, int64_t dst_rows,
                                                              int64_t width, int64_t total) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= total) return;
  const int64_t r = e / width, c = e - r * width;
  const int64_t o = r / dst_rows, i = r - o * dst_rows;
  const int64_t s = clamp_index(index[i], src_rows);
  dst[e] = src[(o * src_rows + s) * width + c];
}

// ------------------------------------------------------------- restore ----
// out[o, t, c] = bf16(full[o, t, c] + bf16(bf16(cur - inp)[o, inv[t], c] * gain))
// (bf16 tensor ops: each op computes in fp32 and rounds once).
__device__ __forceinline__ float restore1(float full, float cur, float inp, float gain) {
  return full + round_bf(round_bf(cur - inp) * gain);
}

// One output row per block; all of a thread's chunks of the three rows are loaded
// before the first is used (rows of up to CPT * 256 chunks; CPT 0: any width, one
// chunk at a time). Memory is the bound: 12605 rows restored from 3683, of width
// 5120 55.2 -> 52.0 us, of 8192 92 -> 82 us, against one chunk at a time.
template <int CPT>
__global__ __launch_bounds__(kThreads) void restore_rows8(const uint4* __restrict__ full,
                                                          const uint4* __restrict__ cur,
                                                          const uint4* __restrict__ inp,
                                                          const int64_t* __restrict__ inverse,
                                                          uint4* __restrict__ out, int64_t out_rows,
                                                          int64_t rows, int64_t compressed,
                                                          int64_t units, float gain) {
  // Consecutive blocks go to different XCDs (round robin over 8). Give each
  // XCD a contiguous range of output rows instead, so that the neighbouring
  // rows that restore from one compressed row share that XCD's L2.
  const int64_t per_xcd = (int64_t)gridDim.x / 8;
  const int64_t r = (int64_t)(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (r >= out_rows) return;
  const int64_t o = r < rows ? 0 : r / rows, t = r - o * rows;
  const int64_t s = o * compressed + clamp_index(inverse[t], compressed);
  auto one = [&](const uint4& fv, const uint4& cv, const uint4& xv) {
    float f[8], c[8], x[8];
    unpack8(fv, f);
    unpack8(cv, c);
    unpack8(xv, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = restore1(f[e], c[e], x[e], gain);
    return pack8(f);
  };
  if constexpr (CPT > 0) {
    const auto rf = row_rsrc(full + r * units, 16 * units);
    const auto rc = row_rsrc(cur + s * units, 16 * units), rx = row_rsrc(inp + s * units, 16 * units);
    const auto ro = row_rsrc(out + r * units, 16 * units);
    const uint32_t off = 16u * threadIdx.x;
    uint4 f[CPT], c[CPT], x[CPT];
#pragma unroll
    for (int i = 0; i < CPT; ++i) f[i] = buf_load16(rf, off, 4096u * i);
#pragma unroll
    for (int i = 0; i < CPT; ++i) c[i] = buf_load16_reused(rc, off, 4096u * i);
#pragma unroll
    for (int i = 0; i < CPT; ++i) x[i] = buf_load16_reused(rx, off, 4096u * i);
#pragma unroll
    for (int i = 0; i < CPT; ++i) buf_store16_nt(ro, off + 4096u * i, one(f[i], c[i], x[i]));
  } else {
    for (int64_t u = threadIdx.x; u < units; u += kThreads)
      store_nt(out + r * units + u, one(load_nt(full + r * units + u), cur[s * units + u], inp[s * units + u]));
  }
}

__global__ __launch_bounds__(kThreads) void restore_rows_any(const uint16_t* __restrict__ full,
                                                             const uint16_t* __restrict__ cur,
                                                             const uint16_t* __restrict__ inp,
                                                             const int64_t* __restrict__ inverse,
                                                             uint16_t* __restrict__ out,
                                                             int64_t rows, int64_t compressed,
                                                             int64_t width, int64_t total,
                                                             float gain) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= total) return;
  const int64_t r = e / width, c = e - r * width;
  const int64_t o = r / rows, t = r - o * rows;
  const int64_t s = (o * compressed + clamp_index(inverse[t], compressed)) * width + c;
  const float v = restore1(bf_to_f(full[e]), bf_to_f(cur[s]), bf_to_f(inp[s]), gain);
  out[e] = (uint16_t)(pack_bf2(v, 0.0f) & 0xffffu);
}

// ------------------------------------------------------ nearest anchor ----
// For dropped row d, over anchors a in increasing order: skip those whose
// time pos[a, 0] differs from pos[d, 0]; keep the first a with the smallest
// (h_d - h_a)^2 + (w_d - w_a)^2. Coordinates are fp32 (the reference casts
// positions with .float()); the distance is formed in fp64, whose rounding
// lies far below the fp32 spacing of the coordinates, and exact ties (integer
// or dyadic grids) resolve to the first anchor, as torch's argmin does. No
// anchor of the same time leaves a = 0, as argmin over a row of +inf does.
// Then inverse[dropped[d]] = inverse[anchors[a]]. Row numbers past `tokens`
// are clamped, like the gather's indices.
//
// One wave per dropped row: lane l scans anchors l, l + 64, ... of each tile
// of anchor positions staged in LDS for the block's rows, keeping its first
// nearest one, and a wave minimum over (distance, anchor index) then gives
// the first nearest anchor of all.
constexpr int kAnchorTile = 1024;
constexpr int kAnchorRows = kThreads / 64;  // dropped rows per block

__global__ __launch_bounds__(kThreads) void nearest_anchor(const float* __restrict__ pos,
                                                           const int64_t* __restrict__ dropped,
                                                           const int64_t* __restrict__ anchors,
                                                           int64_t* __restrict__ inverse,
                                                           int64_t tokens, int64_t n_dropped,
                                                           int64_t n_anchors) {
  __shared__ float tt[kAnchorTile], th[kAnchorTile], tw[kAnchorTile];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t d = (int64_t)blockIdx.x * kAnchorRows + wave;
  const bool live = d < n_dropped;
  const int64_t row = live ? clamp_index(dropped[d], tokens) : 0;
  const float t0 = live ? pos[3 * row] : 0.0f;
  const double h0 = live ? (double)pos[3 * row + 1] : 0.0;
  const double w0 = live ? (double)pos[3 * row + 2] : 0.0;
  double best = __builtin_inf();
  int64_t best_a = 0;
  for (int64_t base = 0; base < n_anchors; base += kAnchorTile) {
    const int n = (int)min((int64_t)kAnchorTile, n_anchors - base);
    __syncthreads();
    for (int j = threadIdx.x; j < n; j += kThreads) {
      const int64_t a = clamp_index(anchors[base + j], tokens);
      tt[j] = pos[3 * a];
      th[j] = pos[3 * a + 1];
      tw[j] = pos[3 * a + 2];
    }
    __syncthreads();
    for (int j = lane; j < n; j += 64) {
      if (tt[j] != t0) continue;
      const double dh = h0 - (double)th[j], dw = w0 - (double)tw[j];
      const double dist = dh * dh + dw * dw;
      if (dist < best) {
        best = dist;
        best_a = base + j;
      }
    }
  }
  // The first anchor of the smallest distance over the wave; lanes that found
  // none hold (+inf, 0), so a row with no anchor of its time keeps a = 0.
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double od = __shfl_xor(best, off);
    const int64_t oa = __shfl_xor(best_a, off);
    if (od < best || (od == best && oa < best_a)) {
      best = od;
      best_a = oa;
    }
  }
  if (live && lane == 0) inverse[row] = inverse[clamp_index(anchors[best_a], tokens)];
}

}  // namespace
}  // namespace lr

using namespace lr;

extern "C" int lr_gather_rows(const void* src, const int64_t* index, void* dst, int64_t outer,
                              int64_t src_rows, int64_t dst_rows, int64_t row_bytes,
                              void* stream) {
  LR_REQUIRE(outer >= 0 && src_rows >= 0 && dst_rows >= 0 && row_bytes >= 0,
             "gather_rows: negative shape");
  const int64_t rows = outer * dst_rows;
  if (rows == 0 || row_bytes == 0) return LR_OK;
  LR_REQUIRE(src_rows > 0, "gather_rows: index into an empty source");
  LR_REQUIRE(src && index && dst, "gather_rows: null pointer");
  hipStream_t st = as_stream(stream);
  if (row_bytes % 16 == 0 && aligned(src, 16) && aligned(dst, 16)) {
    const int64_t units = row_bytes / 16;
    LR_REQUIRE(rows <= kMaxBlocks || (units < 64 && rows * units < 0x7fffff00LL), "gather_rows: too many rows");
    const uint4* from = static_cast<const uint4*>(src);
    uint4* to = static_cast<uint4*>(dst);
    const dim3 grid((unsigned)rows), block(kThreads);
    // Below 1 KB a block per row would leave three of its four waves idle; from
    // there on a block per row is as good (1024 bytes: 4.2 us, 4.5 shared).
    if (units < 64 && rows * units < 0x7fffff00LL) {
      const uint32_t total = (uint32_t)(rows * units);
      hipLaunchKernelGGL(gather_rows16_narrow, dim3((total + kThreads - 1) / kThreads), block, 0, st, from,
                         index, to, src_rows, (uint32_t)dst_rows, (uint32_t)units, total);
    } else if (units <= kThreads || units > 4 * kThreads) {
      hipLaunchKernelGGL(gather_rows16_loop, grid, block, 0, st, from, index, to, src_rows, dst_rows, units);
    } else if (units <= 2 * kThreads) {
      hipLaunchKernelGGL(gather_rows16<2>, grid, block, 0, st, from, index, to, src_rows, dst_rows, units);
    } else if (units <= 3 * kThreads) {
      hipLaunchKernelGGL(gather_rows16<3>, grid, block, 0, st, from, index, to, src_rows, dst_rows, units);
    } else {
      hipLaunchKernelGGL(gather_rows16<4>, grid, block, 0, st, from, index, to, src_rows, dst_rows, units);
    }
  } else {
    const int64_t total = rows * row_bytes;
    const int64_t blocks = (total + kThreads - 1) / kThreads;
    LR_REQUIRE(blocks <= kMaxBlocks, "gather_rows: too many bytes");
    hipLaunchKernelGGL(gather_rows_bytes, dim3((unsigned)blocks), dim3(kThreads), 0, st,
                       (const uint8_t*)src, index, (uint8_t*)dst, src_rows, dst_rows, row_bytes,
                       total);
  }
  return check_launch("gather_rows");
}

extern "C" int lr_flash_restore(const void* full, const void* current, const void* input,
                                const int64_t* inverse, void* out, int64_t outer, int64_t rows,
                                int64_t compressed_rows, int64_t width, float gain, void* stream) {
  LR_REQUIRE(outer >= 0 && rows >= 0 && compressed_rows >= 0 && width >= 0,
             "flash_restore: negative shape");
  const int64_t out_rows = outer * rows;
  if (out_rows == 0 || width == 0) return LR_OK;
  LR_REQUIRE(compressed_rows > 0, "flash_restore: no compressed rows to restore from");
  LR_REQUIRE(full && current && input && inverse && out, "flash_restore: null pointer");
  hipStream_t st = as_stream(stream);
  if (width % 8 == 0 && aligned(full, 16) && aligned(current, 16) && aligned(input, 16) &&
      aligned(out, 16)) {
    const int64_t blocks = 8 * ((out_rows + 7) / 8);  // a whole number of rows per XCD
    LR_REQUIRE(blocks <= kMaxBlocks, "flash_restore: too many rows");
    const int64_t units = width / 8;
#define LR_RESTORE(C)                                                                              \
  hipLaunchKernelGGL(restore_rows8<C>, dim3((unsigned)blocks), dim3(kThreads), 0, st,               \
                     (const uint4*)full, (const uint4*)current, (const uint4*)input, inverse,       \
                     (uint4*)out, out_rows, rows, compressed_rows, units, gain)
    // At most one chunk per thread leaves nothing to overlap, and the loop is the
    // lighter kernel (12605 rows of 1024: 12.9 us, 15.1 up front).
    if (units <= kThreads || units > 4 * kThreads) LR_RESTORE(0);
    else if (units <= 2 * kThreads) LR_RESTORE(2);
    else if (units <= 3 * kThreads) LR_RESTORE(3);
    else LR_RESTORE(4);
#undef LR_RESTORE
  } else {
    const int64_t total = out_rows * width;
    const int64_t blocks = (total + kThreads - 1) / kThreads;
    LR_REQUIRE(blocks <= kMaxBlocks, "flash_restore: too many elements");
    hipLaunchKernelGGL(restore_rows_any, dim3((unsigned)blocks), dim3(kThreads), 0, st,
                       (const uint16_t*)full, (const uint16_t*)current, (const uint16_t*)input,
                       inverse, (uint16_t*)out, rows, compressed_rows, width, total, gain);
  }
  return check_launch("flash_restore");
}

extern "C" int lr_flash_nearest_anchor(const float* positions, int64_t tokens,
                                       const int64_t* dropped, int64_t n_dropped,
                                       const int64_t* anchors, int64_t n_anchors,
                                       int64_t* inverse, void* stream) {
  LR_REQUIRE(tokens >= 0 && n_dropped >= 0 && n_anchors >= 0, "nearest_anchor: negative shape");
  if (n_dropped == 0) return LR_OK;
  LR_REQUIRE(n_anchors > 0 && tokens > 0, "nearest_anchor: dropped rows but no anchors");
  LR_REQUIRE(positions && dropped && anchors && inverse, "nearest_anchor: null pointer");
  const int64_t blocks = (n_dropped + kAnchorRows - 1) / kAnchorRows;
  LR_REQUIRE(blocks <= kMaxBlocks, "nearest_anchor: too many rows");
  hipLaunchKernelGGL(nearest_anchor, dim3((unsigned)blocks), dim3(kThreads), 0, as_stream(stream),
                     positions, dropped, anchors, inverse, tokens, n_dropped, n_anchors);
  return check_launch("nearest_anchor");
}
