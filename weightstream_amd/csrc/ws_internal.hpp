// Host-side helpers shared by the translation units of libweightstream_hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include "../../include/ws_hip.h"
#include "ws_device.hpp"

namespace ws {

// Status of the launch just issued: a configuration error is reported at
// launch, anything asynchronous surfaces on the caller's next sync.
inline int launch_status() {
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? WS_OK : (int)e;
}

// Math mode of this library build (math_mode.hip: WS_MATH_EXACT in
// libweightstream_hip.so, WS_MATH_NATIVE in libweightstream_hip_native.so).
int math_mode();

// Compute units of the current device (queried once per device).
int cu_count();

// Fused GEMVs (gemm.hip): f32 activations x [m <= 16][k] quantised per 1x32
// in the kernel, FP8 weights w [n or 2n][k] with 32 x 32 UE8M0 scales sw.
// kGemvAcc: out[m][n] += x.w^T; kGemvAcc2: out = out + (aux + x.w^T);
// kGemvSwiglu: out[m][n] = silu(min(g, L)) * clamp(u, -L, L) with g from
// weight rows [0, n) and u from rows [n, 2n). Bits equal to ws_emit8 then
// ws_fp8_gemm then the f32 adds / swiglu_emit8's h.
constexpr int kGemvAcc = 2, kGemvAcc2 = 3, kGemvSwiglu = 4;
int kp_gemv_fused(int omode, const float *x, const uint8_t *w, const uint8_t *sw, float *out,
                  const float *aux, float limit, int64_t m, int64_t n, int64_t k,
                  hipStream_t stream);

// gemm.hip: the f32 gate logits [m][E] of h (m <= 8, dim % 256 == 0) and
// hs = SwiGLU of the shared gate/up GEMV (kGemvSwiglu) in one launch.
int gate_w13_launch(const float *h, const float *gw, float *logits, const uint8_t *w13,
                    const uint8_t *s13, float *hs, int64_t m, int64_t dim, int64_t n_experts,
                    int64_t inter, float limit, hipStream_t stream);

// gemm_line.hip: the FP8 GEMM for row blocks of 33-128 rows with whole-K
// tiles (configuration cfg); -1 when the shape does not fit that tiling.
int line_gemm(int smode, int omode, const uint8_t *a, const void *sa, const uint8_t *b,
              const void *sb, void *out, int m, int n, int k, hipStream_t stream, int cfg,
              const float *aux = nullptr);
// gemm_tile.hip: the exact-math FP8 GEMM with bf16 results for many rows (whole-K
// tiles). -1 when the shape or alignment does not fit.
int tile_gemm_bf16(int smode, const uint8_t *a, const void *sa, const uint8_t *b, const void *sb,
                   void *out, int64_t m, int64_t n, int64_t k, hipStream_t stream);
// moe_tile.hip: the grouped gate/up (bf16 h out) and down steps over 96-slot
// groups, exact math; offsets and counts are the dispatch's. part: scratch of
// part_bytes for the gate/up sums of the first K part; moe_tile_parts says how
// it is used, -1 where it is too small for the shape.
int moe_tile_parts(size_t part_bytes, int slots, int dim, int inter);
int moe_tile_glu(const uint16_t *xbf, const int32_t *order, const float *layout_w,
                 const int32_t *exp_off, const int32_t *exp_cnt, const uint8_t *w1,
                 const uint8_t *s1, const uint8_t *w3, const uint8_t *s3, uint16_t *hbf,
                 uint8_t *part, size_t part_bytes, int slots, int dim, int inter, int n_experts,
                 int top_k, float limit, hipStream_t stream);
int moe_tile_down(const uint16_t *hbf, const int32_t *exp_off, const int32_t *exp_cnt,
                  const uint8_t *w2, const uint8_t *s2, float *out, int dim, int inter,
                  int n_experts, hipStream_t stream);
// C = C + (aux + A.B^T) with UE8M0 32 x 32 weight scales (gemm.hip)
int fp8_gemm_acc2(const uint8_t *a, const uint8_t *sa, const uint8_t *b, const uint8_t *sb,
                  float *c, const float *aux, int64_t m, int64_t n, int64_t k, hipStream_t stream);

}  // namespace ws
