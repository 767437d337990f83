// General affine quantized matmul (4- or 8-bit, group 32/64/128) and the
// activation chunk-sum table of the cross-row lane.
//
//   y[m, n] = sum_k x[m, k] * (q[n, k] * s[n, k/gs] + b[n, k/gs])
//
// Weight format (MLX's affine quantization, as the reference's verify lanes
// read it: mtplx/verify_qmv.py:1256-1377 for 8-bit, mtplx/kernels/
// qmv4_matmul.py:158 / mtplx/verify_crossrow.py:57 for group 32): uint32
// [N, K*bits/32] with little-endian fields (value i of a word in bits
// bits*i .. bits*i + bits - 1), bf16 scales/biases [N, K/gs].
//
// This is the lane for the formats that have no tile-major pack (8-bit, group
// 32, K not a multiple of 256): the weights stream in place (qmv_inplace.hpp),
// the rows in tiles of 4 or 16.
#include "qmv_inplace.hpp"

namespace mtp {

namespace {

constexpr int kTableRows = 8;   // rows of the chunk-sum table

// out[(kb * 32 + lane) * 8 + m] = sum of x[m, kb*512 + lane*16 + i], i < 16,
// added in index order (fp32); rows m >= M are zero.
__global__ __launch_bounds__(256) void chunk_sums_kernel(const uint16_t* x, int M, int K, int ldx, float* out) {
  const int slot = blockIdx.x * 256 + threadIdx.x;
  const int lanes = (K / 512) * 32;
  if (slot >= lanes) return;
  const int base = (slot >> 5) * 512 + (slot & 31) * 16;
  for (int m = 0; m < 8; ++m) {
    float t = 0.f;
    if (m < M)
      for (int i = 0; i < 16; ++i) t += bf2f(x[(size_t)m * ldx + base + i]);
    out[(size_t)slot * 8 + m] = t;
  }
}

}  // namespace

}  // namespace mtp

using namespace mtp;

static int qmv_affine_run(const void* x, const float* xsums, const void* w, const void* scales, const void* biases,
                          void* y, void* yf, int M, int N, int K, int group_size, int bits, void* stream,
                          const char* who) {
  if (!x || !w || !scales || !biases || (!y && !yf) || M < 1 || N < 1 || K < 32 || K % 32) {
    set_error("%s: bad arguments (non-null x/w/scales/biases/output, M, N >= 1, K a positive multiple of 32)", who);
    return MTP_ERR_ARG;
  }
  if (bits != 4 && bits != 8) {
    set_error("%s: %d-bit weights unsupported (4 or 8)", who, bits);
    return MTP_ERR_UNSUPPORTED;
  }
  if ((group_size != 32 && group_size != 64 && group_size != 128) || K % group_size) {
    set_error("%s: group_size %d unsupported or does not divide K=%d (32, 64, 128)", who, group_size, K);
    return MTP_ERR_UNSUPPORTED;
  }
  if (((uintptr_t)w & 15)) {
    set_error("%s: weights must be 16-byte aligned", who);
    return MTP_ERR_ARG;
  }
  InplaceParams p = {};
  p.x = (const uint16_t*)x;
  p.w0 = (const uint8_t*)w;
  p.s0 = (const uint16_t*)scales;
  p.b0 = (const uint16_t*)biases;
  p.y = (uint16_t*)y;
  p.yf = (float*)yf;
  p.xsums = xsums;
  p.M = M;
  p.N = N;
  p.K = K;
  p.ldx = K;
  p.ldy = N;
  inplace_launch(p, bits, group_size, false, (hipStream_t)stream);
  return launch_check(who);
}

MTP_API int mtp_qmv_affine(const void* x, const void* w, const void* scales, const void* biases, void* y, void* yf,
                           int M, int N, int K, int group_size, int bits, void* stream) {
  return qmv_affine_run(x, nullptr, w, scales, biases, y, yf, M, N, K, group_size, bits, stream, "mtp_qmv_affine");
}

MTP_API int mtp_crossrow_qmm(const void* x, const float* xsums, const void* w, const void* scales,
                             const void* biases, void* y, int M, int N, int K, int group_size, void* stream) {
  const char* who = "mtp_crossrow_qmm";
  if (!xsums || M < 1 || M > kTableRows || K < 512 || K % 512) {
    set_error("%s: need the chunk-sum table (mtp_chunk_sums), 1 <= M <= %d and K a positive multiple of 512", who,
              kTableRows);
    return MTP_ERR_ARG;
  }
  if (group_size != 32 && group_size != 64) {
    set_error("%s: group_size %d unsupported (the cross-row lane takes 32 or 64)", who, group_size);
    return MTP_ERR_UNSUPPORTED;
  }
  return qmv_affine_run(x, xsums, w, scales, biases, y, nullptr, M, N, K, group_size, 4, stream, who);
}

MTP_API int mtp_chunk_sums(const void* x, int M, int K, float* out, void* stream) {
  if (!x || !out || M < 1 || M > 8 || K < 512 || K % 512) {
    set_error("mtp_chunk_sums: bad arguments (1 <= M <= 8, K a positive multiple of 512)");
    return MTP_ERR_ARG;
  }
  const int lanes = (K / 512) * 32;
  hipLaunchKernelGGL(chunk_sums_kernel, dim3((lanes + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)x, M, K, K, out);
  return launch_check("mtp_chunk_sums");
}
