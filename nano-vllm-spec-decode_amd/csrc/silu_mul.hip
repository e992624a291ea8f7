// SiLU-and-multiply between the gate / up and the down projection (SiluAndMul.forward,
// nanovllm/layers/activation.py:8-11): out[m, i] = bf16(bf16(silu(gate[m, i])) * up[m, i]) with gate the first and
// up the second half of a row, silu(x) = x / (1 + e^-x) in fp32, rounded to bf16 before the product as the eager
// operations do. One thread per 8 columns; short calls are bound by their launch, long ones by HBM (6 bytes an
// element). As two library operations it took two launches, 5 us each at 80 rows x 12288, and 2 bytes an element
// written and read again.
#include "sd_common.h"
#include "../../include/sd_attn.h"

namespace sd {
namespace {

constexpr int kThreads = 256;

struct SiluArgs {
  const uint16_t* x;
  uint16_t* out;
  int64_t x_stride, out_stride;
  int32_t half;  // columns of gate, of up and of out
};

__device__ __forceinline__ float low(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float high(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
__device__ __forceinline__ float silu(float x) { return __fdiv_rn(x, 1.0f + expf(-x)); }

__global__ __launch_bounds__(kThreads) void silu_mul_rows(SiluArgs a) {
#pragma clang fp contract(off)
  const int c = 8 * (blockIdx.y * kThreads + threadIdx.x);
  if (c >= a.half) return;
  const uint16_t* x = a.x + (int64_t)blockIdx.x * a.x_stride + c;
  const u32x4 g = *(const u32x4*)x, u = *(const u32x4*)(x + a.half);
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t s = cvt_bf16x2(silu(low(g[i])), silu(high(g[i])));
    w[i] = cvt_bf16x2(low(s) * low(u[i]), high(s) * high(u[i]));
  }
  *(u32x4*)(a.out + (int64_t)blockIdx.x * a.out_stride + c) = w;
}

}  // namespace
}  // namespace sd

using namespace sd;

// x: bf16 rows [gate | up] of 2 * half columns, out: rows of half columns; rows 16-byte aligned, half a multiple of 8.
// For this package's layers (not declared in sd_attn.h).
extern "C" int sd_silu_mul(const void* x, int64_t x_row_stride, int32_t rows, int32_t half, void* out,
                           int64_t out_row_stride, void* stream) {
  const char* who = "sd_silu_mul";
  if (rows < 0 || half <= 0) return fail(kBadArgument, "%s: bad sizes (rows %d, columns %d)", who, rows, half);
  const int blocks = (half / 8 + kThreads - 1) / kThreads;
  if (half % 8 || blocks > 65535)
    return fail(kUnsupported, "%s: %d columns (a multiple of 8, at most 2^27)", who, half);
  if (rows == 0) return kOk;
  if (!x || !out) return fail(kBadArgument, "%s: null pointer", who);
  if (x_row_stride < 2 * (int64_t)half || out_row_stride < half)
    return fail(kBadArgument, "%s: a row stride is smaller than the row", who);
  if (((uintptr_t)x | (uintptr_t)out) % 16 || x_row_stride % 8 || out_row_stride % 8)
    return fail(kUnsupported, "%s: pointers must be 16-byte aligned and row strides multiples of 8", who);
  const SiluArgs a{(const uint16_t*)x, (uint16_t*)out, x_row_stride, out_row_stride, half};
  hipLaunchKernelGGL(silu_mul_rows, dim3((unsigned)rows, (unsigned)blocks), dim3(kThreads), 0, (hipStream_t)stream, a);
  return check_launch(who);
}
