// The 8-bit weight formats of the dequant GEMM (sqx_dqgemm.h): the prefill form of the int8 weight-only linear
// and of fp8_linear (fp8_weights.py:211-262, called by sqx_fp8.hip on the quantized rows).
#include "sqx_dqgemm.h"

namespace sqx {

int64_t fp8_gemm_workspace_bytes(int64_t m, int64_t rows, int64_t cols) {
  return dq_workspace_bytes(dq_plan(m, rows, ceil_div(cols, 64), kDqI8), m, rows);
}

bool gemm8_fits(int64_t m, int64_t rows, int64_t cols) {
  return m > 0 && rows > 0 && cols > 0 && cols % 8 == 0 && m * cols * 2 < ((int64_t)1 << 31) &&
         ceil_div(rows, 16) * ceil_div(cols, 64) * 1024 < ((int64_t)1 << 31) &&
         ceil_div(m, 128) * ceil_div(rows, 128) * 16 < ((int64_t)1 << 31);
}

hipError_t fp8_gemm(const uint8_t* wt, const float* w_scale, const float* x_scale, const uint16_t* vals, void* y,
                    bool yf32, const uint16_t* bias, int64_t m, int64_t rows, int64_t cols, float* ws, int64_t ws_bytes,
                    hipStream_t s) {
  const int KB = (int)ceil_div(cols, 64);
  if (yf32)
    return launch_dq<ActBF16, kDqF8, false, false, 64, 2>(vals, wt, nullptr, nullptr, w_scale, x_scale, y, nullptr, (int)m,
                                                          (int)rows, (int)cols, KB, ws, ws_bytes, s);
  return launch_dq<ActBF16, kDqF8, false, false, 64, 0>(vals, wt, nullptr, nullptr, w_scale, x_scale, y, bias, (int)m,
                                                        (int)rows, (int)cols, KB, ws, ws_bytes, s);
}

}  // namespace sqx

using namespace sqx;

// Where the GEMV's two passes over a small weight are faster than the GEMM's prologue and its few workgroups (us, GEMV
// and GEMM: 512 -> 512 at m = 65 / 96 / 128 7.9 / 9.2 / 10.9 and 10.6 / 10.8 / 11.0, 1024 -> 1024 at 65 / 100 9.0 / 11.5
// and 11.0 / 11.7, 1536 -> 3000 at 72 / 96 12.4 / 14.5 and 13.3 / 14.3, 2048 -> 2000 at 65 13.1 and 12.4).
static bool int8_gemv_ahead(int64_t m, int64_t rows, int64_t cols) {
  return (m <= 104 && rows <= 1024 && cols <= 1024) || (m <= 80 && rows <= 3072 && cols <= 1536);
}

extern "C" int64_t sqx_int8_gemm_workspace_bytes(int64_t m, int64_t rows, int64_t cols) {
  if (!gemm8_fits(m, rows, cols) || int8_gemv_ahead(m, rows, cols)) return -1;
  return dq_workspace_bytes(dq_plan(m, rows, ceil_div(cols, 64), kDqI8), m, rows);
}

extern "C" int sqx_int8_gemm(const uint8_t* wt, const float* scale, const void* x, int act_dtype, void* y,
                             const void* bias, int64_t m, int64_t rows, int64_t cols, void* ws, int64_t ws_bytes,
                             sqx_stream_t stream) {
  SQX_REQUIRE(act_dtype == SQX_DTYPE_BF16 || act_dtype == SQX_DTYPE_F16, SQX_E_ARG,
              "sqx_int8_gemm: activations must be BF16 or F16");
  if (m == 0) return SQX_OK;
  SQX_REQUIRE(gemm8_fits(m, rows, cols), SQX_E_ARG,
              "sqx_int8_gemm: bad shape m=%lld rows=%lld cols=%lld (cols %% 8 == 0, operands below 2 GiB)", (long long)m,
              (long long)rows, (long long)cols);
  SQX_REQUIRE(wt && scale && x && y, SQX_E_ARG, "sqx_int8_gemm: null pointer");
  SQX_REQUIRE(reinterpret_cast<uintptr_t>(wt) % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0, SQX_E_ARG,
              "sqx_int8_gemm: wt and x must be 16-byte aligned");
  const int KB = (int)ceil_div(cols, 64);
  const auto* xp = static_cast<const uint16_t*>(x);
  const auto* b16 = static_cast<const uint16_t*>(bias);
  auto* w32 = static_cast<float*>(ws);
  hipStream_t s = as_stream(stream);
  const hipError_t e =
      act_dtype == SQX_DTYPE_BF16
          ? launch_dq<ActBF16, kDqI8, false, false, 64, 0>(xp, wt, nullptr, nullptr, scale, nullptr, y, b16, (int)m, (int)rows,
                                                           (int)cols, KB, w32, ws_bytes, s)
          : launch_dq<ActF16, kDqI8, false, false, 64, 1>(xp, wt, nullptr, nullptr, scale, nullptr, y, b16, (int)m, (int)rows,
                                                          (int)cols, KB, w32, ws_bytes, s);
  SQX_REQUIRE(e == hipSuccess, SQX_E_HIP, "sqx_int8_gemm: launch failed: %s", hipGetErrorString(e));
  return SQX_OK;
}
