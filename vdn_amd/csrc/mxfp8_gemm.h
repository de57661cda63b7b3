// Shared by the block-scaled GEMM kernels: the epilogue description and its helpers, the scale
// layout, and the launch interface of the stream kernel (mxfp8_gemm_stream.hip).
#pragma once

#include "mxfp8_common.h"

namespace vdn {

constexpr int kBK = 128;   // K per step: one scaled MFMA deep

// SWIZZLE_32_4_4 keeps the scale dwords (4 K-blocks of one 128-K step) of a 128-row block
// in one contiguous 512-byte run: row r's dword sits at 16 (r % 32) + 4 ((r % 128) / 32)
// of it. The run of block b for K step ks starts at (b * col_tiles + ks) * 512.
__device__ __forceinline__ int scale_in_block(int r) { return (r & 31) * 16 + ((r & 127) >> 5) * 4; }

// Epilogue of one output element y (the bf16-rounded accumulator), in this order:
//   y = bf16(y + bias[c])                    (bias: nullable, [n])
//   y = bf16(addend[r, c] + y)               (addend: nullable)
//   y = bf16(residual[r, c] + bf16(gate[c] * y))   (residual: nullable; gate nullable = 1)
// `out` may alias `addend` or `residual`: every element is read and written by one lane.
struct Epilogue {
  const uint16_t* bias;
  const uint16_t* addend;
  int64_t ld_add;
  const uint16_t* residual;
  int64_t ld_res;
  const uint16_t* gate;
  uint16_t* out;
  int64_t ldc;
  uint32_t* nonfinite;
  int vec;  // 16-byte accesses: n, every leading dimension and pointer 8-element aligned
  // Producer mode (q_out non-null): instead of bf16 `out`, y = bf16(bf16(acc) + bias) goes
  // through `act` (0 none, 1 GELU-tanh, rounded to bf16) and is stored as MXFP8 codes
  // q_out [mp, kp_out] + swizzled scales s_out, exactly what the producer kernels write
  // for that bf16 matrix. Rows >= out_rows and columns >= n are stored as zero.
  uint8_t* q_out;
  uint8_t* s_out;
  int64_t kp_out;
  int act;
};

// Epilogue arithmetic of one element (see Epilogue).
__device__ __forceinline__ float epilogue_value(float y, float b, float addend, float res, float gt,
                                                const Epilogue& ep) {
  if (ep.bias != nullptr) y = round_bf16(y + b);
  if (ep.addend != nullptr) y = round_bf16(addend + y);
  if (ep.residual != nullptr) {
    const float t = ep.gate != nullptr ? round_bf16(gt * y) : y;
    y = round_bf16(res + t);
  }
  return y;
}

__device__ __forceinline__ void unpack4(const u32x2 w, float* f) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    f[2 * i] = __uint_as_float(w[i] << 16);
    f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

__device__ __forceinline__ void unpack8(const u32x4 w, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = bf16_bits_to_f32(static_cast<uint16_t>(w[i] & 0xffff));
    f[2 * i + 1] = bf16_bits_to_f32(static_cast<uint16_t>(w[i] >> 16));
  }
}

// Operands of one GEMM launch (checked by the entry points).
struct GemmArgs {
  const uint8_t *a, *as, *w, *ws;
  int64_t mp, np, kp;
  Epilogue ep;
  int64_t out_rows, n;
};

// The epilogues: 0 bf16, 1 bf16 with a residual, 2 MXFP8 producer (no activation, GELU-tanh),
// 3 MXFP8 producer with SwiGLU.
inline int gemm_mode(const Epilogue& ep) {
  return ep.q_out != nullptr ? (ep.act == 2 ? 3 : 2) : ep.residual != nullptr ? 1 : 0;
}

// mxfp8_gemm.hip: the large-problem kernel (one workgroup per CU, 256 x 256 tiles).
int launch_persistent(const GemmArgs& g, hipStream_t stream);

// mxfp8_gemm_stream.hip: the large kernel, the stream kernel or both, by size.
int launch_gemm_planned(const GemmArgs& g, int mode, hipStream_t stream);
// Its choice: rows of the large kernel, and tile columns of the stream kernel below them (0: none).
void gemm_choice(int64_t mp, int64_t np, int64_t kp, int mode, int64_t* large_rows, int* tile_cols);

}  // namespace vdn
