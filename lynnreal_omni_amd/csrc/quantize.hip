// quantize.hip - per-row INT8 activation quantizer and the stand-alone
// INT32 -> bf16 dequant epilogue.
//
// quantize_rows restates model/int8.py:66-67 (the torch path; the Triton
// kernel model/kernels.py:8-16 computes the same values). Narrow rows (under
// 4096): one wave per row, four rows per 256-thread block; lane l holds 16-byte
// chunks l, l+64, ... in registers, the absmax is a wave butterfly, and the
// row is quantized from registers and written with 8-byte stores. Rows of 4096 and
// more, and at most 512 rows wider than 2048: one 256-thread block per row, same
// scheme with a block reduction. HBM
// traffic is the algorithmic 3 bytes/element plus 4 bytes/row.
#include "lr_device.h"
#include "lr_runtime.h"

namespace lr {
namespace {

constexpr int kThreads = 256;

template <int CPL>
__global__ __launch_bounds__(kThreads) void quantize_rows_wave(const uint4* __restrict__ x,
                                                               uint2* __restrict__ q,
                                                               float* __restrict__ scales,
                                                               int64_t rows, int chunks) {
  const int lane = threadIdx.x & 63;
  const int64_t row = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  if (row >= rows) return;  // whole wave
  // Buffer accesses: past the row end loads give zero and stores are dropped.
  const auto src = row_rsrc(x + row * chunks, 16 * (int64_t)chunks);
  const auto dst = row_rsrc(q + row * chunks, 8 * (int64_t)chunks);
  uint4 v[CPL];
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < CPL; ++i) v[i] = buf_load16(src, 16u * lane, 1024u * i);
#pragma unroll
  for (int i = 0; i < CPL; ++i) m = absmax8(v[i], m);
  const float s = quant_scale(wave_max(m));
  const float inv = 1.0f / s;
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    buf_store8(dst, 8u * lane, 512u * i, quant8_bf(v[i], s, inv));
    __builtin_amdgcn_sched_barrier(0);
  }
  if (lane == 0) scales[row] = s;
}

// One block per row, for rows of 4096 and more and for few rows wider than 2048,
// where a wave per row has more serial work than it hides. Loads and stores go
// through descriptors that end with the row. NT: non-temporal loads, for inputs
// past 32 MB; smaller ones are read through the caches, for layers that are called
// on the same rows again (layer calls of 2048 x 5120 rows 51.6 us, 52.8
// non-temporal); rows read once are faster non-temporally (2048 x 5120 from memory
// 7.4 us, 8.1 through the caches; just written 5.5 and 6.1). Rows past 8192 always
// load non-temporally (the other form is not built for them) and are stored
// write-back (20480 wide, 12605 rows 116.7 against 123.9 us non-temporal), narrower
// ones non-temporally.
template <int CPT, bool NT>
__global__ __launch_bounds__(kThreads) void quantize_rows_block(const uint4* __restrict__ x,
                                                                uint2* __restrict__ q,
                                                                float* __restrict__ scales,
                                                                int64_t chunks) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  const auto src = row_rsrc(x + row * chunks, 16 * chunks);
  const auto dst = row_rsrc(q + row * chunks, 8 * chunks);
  uint4 v[CPT];
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < CPT; ++i)
    v[i] = NT ? buf_load16(src, 16u * threadIdx.x, 4096u * i) : buf_load16_reused(src, 16u * threadIdx.x, 4096u * i);
#pragma unroll
  for (int i = 0; i < CPT; ++i) m = absmax8(v[i], m);
  m = block256_max(m, red);
  const float s = quant_scale(m);
  const float inv = 1.0f / s;
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const uint2 b = quant8_bf(v[i], s, inv);
    if (CPT > 4) buf_store8_cached(dst, 8u * threadIdx.x, 2048u * i, b);
    else buf_store8(dst, 8u * threadIdx.x, 2048u * i, b);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (threadIdx.x == 0) scales[row] = s;
}

// Any width / alignment: two passes over global memory, element-wise.
__global__ __launch_bounds__(kThreads) void quantize_rows_any(const uint16_t* __restrict__ x,
                                                              int8_t* __restrict__ q,
                                                              float* __restrict__ scales,
                                                              int64_t width) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  const uint16_t* src = x + row * width;
  float m = 0.0f;
  for (int64_t c = threadIdx.x; c < width; c += kThreads) m = fmaxf(m, __builtin_fabsf(bf_to_f(src[c])));
  m = block256_max(m, red);
  const float s = quant_scale(m);
  const float inv = 1.0f / s;
  for (int64_t c = threadIdx.x; c < width; c += kThreads)
    q[row * width + c] = (int8_t)quant_one(bf_to_f(src[c]), s, inv);
  if (threadIdx.x == 0) scales[row] = s;
}

// fp16 and fp32 rows (the reference's Triton quantizer loads any float type
// as fp32, model/kernels.py:12): the same scale, and the IEEE quotient x / s
// itself (the corrected-reciprocal form above is proven for bf16 values
// only). One block per row, two passes over the row (the second from L2).
template <typename T>
__device__ __forceinline__ float as_float(T v) { return (float)v; }

template <typename T>
__global__ __launch_bounds__(kThreads) void quantize_rows_typed(const T* __restrict__ x,
                                                                int8_t* __restrict__ q,
                                                                float* __restrict__ scales,
                                                                int64_t width) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  const T* src = x + row * width;
  float m = 0.0f;
  for (int64_t c = threadIdx.x; c < width; c += kThreads) m = fmaxf(m, __builtin_fabsf(as_float(src[c])));
  m = block256_max(m, red);
  const float s = quant_scale(m);
  for (int64_t c = threadIdx.x; c < width; c += kThreads) {
    const float v = __builtin_rintf(as_float(src[c]) / s);
    q[row * width + c] = (int8_t)fminf(fmaxf(v, -127.0f), 127.0f);
  }
  if (threadIdx.x == 0) scales[row] = s;
}

template <int CPT, bool NT>
void launch_quant_block(const void* x, int8_t* q, float* s, int64_t rows, int64_t chunks,
                        hipStream_t st) {
  hipLaunchKernelGGL((quantize_rows_block<CPT, NT>), dim3((unsigned)rows), dim3(kThreads), 0, st,
                     (const uint4*)x, (uint2*)q, s, chunks);
}

// us, wave per row / block per row (graph-replayed, rotating inputs): 7168 wide,
// 16 rows 4.1 / 2.5, 512 rows 4.8 / 3.8, 3683 rows 16.5 / 14.7, 12605 rows 45.5 /
// 43.3; 5120 wide 256 rows 3.8 / 2.7, 12605 rows 32.5 / 31.6; 3072 wide 512 rows
// 3.3 / 2.9, 12605 rows 20.1 / 21.8; 1024 wide slower at every count.
void launch_quant_rows(const void* x, int8_t* q, float* s, int64_t rows, int64_t chunks,
                       hipStream_t st) {
  const int need = (int)((chunks + kThreads - 1) / kThreads);
  if (rows * chunks * 16 <= 32LL << 20 && need <= 4) {
    if (need <= 2) launch_quant_block<2, false>(x, q, s, rows, chunks, st);
    else if (need <= 3) launch_quant_block<3, false>(x, q, s, rows, chunks, st);
    else launch_quant_block<4, false>(x, q, s, rows, chunks, st);
  } else if (need <= 2) launch_quant_block<2, true>(x, q, s, rows, chunks, st);
  else if (need <= 3) launch_quant_block<3, true>(x, q, s, rows, chunks, st);
  else if (need <= 4) launch_quant_block<4, true>(x, q, s, rows, chunks, st);
  else if (need <= 6) launch_quant_block<6, true>(x, q, s, rows, chunks, st);
  else if (need <= 8) launch_quant_block<8, true>(x, q, s, rows, chunks, st);
  else if (need <= 10) launch_quant_block<10, true>(x, q, s, rows, chunks, st);
  else if (need <= 12) launch_quant_block<12, true>(x, q, s, rows, chunks, st);
  else launch_quant_block<16, true>(x, q, s, rows, chunks, st);
}

template <int CPL>
void launch_quant_wave(const void* x, int8_t* q, float* s, int64_t rows, int chunks,
                       hipStream_t st) {
  hipLaunchKernelGGL(quantize_rows_wave<CPL>, dim3((unsigned)((rows + 3) / 4)), dim3(kThreads), 0,
                     st, (const uint4*)x, (uint2*)q, s, rows, chunks);
}

// ------------------------------------------------------------ epilogue ----
// out = bf16(((float)acc * as[r]) * ws[c] + bias[c]); model/kernels.py:27-38.
template <bool HAS_BIAS>
__global__ __launch_bounds__(kThreads) void epilogue4(const int4* __restrict__ acc,
                                                      const float* __restrict__ as,
                                                      const float* __restrict__ ws,
                                                      const uint16_t* __restrict__ bias,
                                                      uint2* __restrict__ out, int64_t groups,
                                                      int64_t n4) {
  const int64_t g = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (g >= groups) return;
  const int64_t r = g / n4;
  const int64_t c = (g - r * n4) * 4;
  const int4 a = acc[g];
  const float rs = as[r];
  const float4 cs = *reinterpret_cast<const float4*>(ws + c);
  float v0 = ((float)a.x * rs) * cs.x, v1 = ((float)a.y * rs) * cs.y;
  float v2 = ((float)a.z * rs) * cs.z, v3 = ((float)a.w * rs) * cs.w;
  if (HAS_BIAS) {
    const uint2 b = *reinterpret_cast<const uint2*>(bias + c);
    v0 = v0 + bf_lo(b.x); v1 = v1 + bf_hi(b.x);
    v2 = v2 + bf_lo(b.y); v3 = v3 + bf_hi(b.y);
  }
  out[g] = make_uint2(pack_bf2(v0, v1), pack_bf2(v2, v3));
}

__global__ __launch_bounds__(kThreads) void epilogue1(const int32_t* __restrict__ acc,
                                                      const float* __restrict__ as,
                                                      const float* __restrict__ ws,
                                                      const uint16_t* __restrict__ bias,
                                                      uint16_t* __restrict__ out, int64_t total,
                                                      int64_t n) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= total) return;
  const int64_t r = e / n, c = e - r * n;
  float v = ((float)acc[e] * as[r]) * ws[c];
  if (bias) v = v + bf_to_f(bias[c]);
  out[e] = (uint16_t)(pack_bf2(v, 0.0f) & 0xffffu);
}

int launch_quant(const void* x, int8_t* q, float* scales, int64_t rows, int64_t width, hipStream_t st) {
  const int64_t chunks = width / 8;
  const bool vec = width % 8 == 0 && aligned(x, 16) && aligned(q, 8) && chunks <= 16 * kThreads &&
                   width > 0;
  if (vec && (chunks >= 512 || (chunks > 256 && rows <= 512))) {
    launch_quant_rows(x, q, scales, rows, chunks, st);
  } else if (vec) {
    const int need = (int)((chunks + 63) / 64);
    const int c = (int)chunks;
    if (need <= 1) launch_quant_wave<1>(x, q, scales, rows, c, st);
    else if (need <= 2) launch_quant_wave<2>(x, q, scales, rows, c, st);
    else if (need <= 3) launch_quant_wave<3>(x, q, scales, rows, c, st);
    else if (need <= 4) launch_quant_wave<4>(x, q, scales, rows, c, st);
    else if (need <= 6) launch_quant_wave<6>(x, q, scales, rows, c, st);
    else launch_quant_wave<8>(x, q, scales, rows, c, st);
  } else {
    hipLaunchKernelGGL(quantize_rows_any, dim3((unsigned)rows), dim3(kThreads), 0, st,
                       (const uint16_t*)x, q, scales, width);
  }
  return check_launch("quantize_rows");
}

template <typename T>
int launch_quant_typed(const T* x, int8_t* q, float* scales, int64_t rows, int64_t width, hipStream_t st) {
  hipLaunchKernelGGL(quantize_rows_typed<T>, dim3((unsigned)rows), dim3(kThreads), 0, st, x, q, scales, width);
  return check_launch("quantize_rows");
}

// launch(x, q, scales, rows) over at most kRowsPerLaunch rows at a time.
template <typename T, typename F>
int in_slices(const T* x, int8_t* q, float* scales, int64_t rows, int64_t width, F launch) {
  int rc = LR_OK;
  for (int64_t r = 0; r < rows && rc == LR_OK; r += kRowsPerLaunch)
    rc = launch(x + r * width, q + r * width, scales + r, rows - r < kRowsPerLaunch ? rows - r : kRowsPerLaunch);
  return rc;
}

}  // namespace
}  // namespace lr

using namespace lr;

extern "C" int lr_quantize_rows(const void* x, int64_t rows, int64_t width, int8_t* q,
                                float* scales, void* stream) {
  LR_REQUIRE(rows >= 0 && width >= 0, "quantize_rows: negative shape (%lld, %lld)",
             (long long)rows, (long long)width);
  if (rows == 0) return LR_OK;
  LR_REQUIRE(x && q && scales, "quantize_rows: null pointer");
  LR_REQUIRE(rows <= 0x7fffffffLL, "quantize_rows: too many rows (%lld)", (long long)rows);
  hipStream_t st = as_stream(stream);
  return in_slices(static_cast<const uint16_t*>(x), q, scales, rows, width,
                   [&](const uint16_t* from, int8_t* to, float* scale, int64_t count) {
                     return launch_quant(from, to, scale, count, width, st);
                   });
}

extern "C" int lr_quantize_rows_typed(const void* x, int dtype, int64_t rows, int64_t width,
                                      int8_t* q, float* scales, void* stream) {
  LR_REQUIRE(dtype == LR_DTYPE_BF16 || dtype == LR_DTYPE_F16 || dtype == LR_DTYPE_F32,
             "quantize_rows: unknown dtype %d", dtype);
  if (dtype == LR_DTYPE_BF16) return lr_quantize_rows(x, rows, width, q, scales, stream);
  LR_REQUIRE(rows >= 0 && width >= 0, "quantize_rows: negative shape (%lld, %lld)",
             (long long)rows, (long long)width);
  if (rows == 0) return LR_OK;
  LR_REQUIRE(x && q && scales, "quantize_rows: null pointer");
  LR_REQUIRE(rows <= 0x7fffffffLL, "quantize_rows: too many rows (%lld)", (long long)rows);
  hipStream_t st = as_stream(stream);
  auto launch = [&](auto* from, int8_t* to, float* scale, int64_t count) {
    return launch_quant_typed(from, to, scale, count, width, st);
  };
  if (dtype == LR_DTYPE_F16) return in_slices(static_cast<const _Float16*>(x), q, scales, rows, width, launch);
  return in_slices(static_cast<const float*>(x), q, scales, rows, width, launch);
}

extern "C" int lr_int8_epilogue(const int32_t* acc, const float* a_scale, const float* w_scale,
                                const void* bias, void* out, int64_t m, int64_t n,
                                void* stream) {
  LR_REQUIRE(m >= 0 && n >= 0, "int8_epilogue: negative shape");
  if (m == 0 || n == 0) return LR_OK;
  LR_REQUIRE(acc && a_scale && w_scale && out, "int8_epilogue: null pointer");
  hipStream_t st = as_stream(stream);
  const bool vec = n % 4 == 0 && aligned(acc, 16) && aligned(w_scale, 16) && aligned(out, 8) &&
                   (bias == nullptr || aligned(bias, 8));
  if (vec) {
    const int64_t groups = m * (n / 4);
    const int64_t blocks = (groups + kThreads - 1) / kThreads;
    LR_REQUIRE(blocks <= kMaxBlocks, "int8_epilogue: too large");
    if (bias)
      hipLaunchKernelGGL(epilogue4<true>, dim3((unsigned)blocks), dim3(kThreads), 0, st,
                         (const int4*)acc, a_scale, w_scale, (const uint16_t*)bias, (uint2*)out,
                         groups, n / 4);
    else
      hipLaunchKernelGGL(epilogue4<false>, dim3((unsigned)blocks), dim3(kThreads), 0, st,
                         (const int4*)acc, a_scale, w_scale, (const uint16_t*)bias, (uint2*)out,
                         groups, n / 4);
  } else {
    const int64_t total = m * n;
    const int64_t blocks = (total + kThreads - 1) / kThreads;
    LR_REQUIRE(blocks <= kMaxBlocks, "int8_epilogue: too large");
    hipLaunchKernelGGL(epilogue1, dim3((unsigned)blocks), dim3(kThreads), 0, st, acc, a_scale,
                       w_scale, (const uint16_t*)bias, (uint16_t*)out, total, n);
  }
  return check_launch("int8_epilogue");
}
