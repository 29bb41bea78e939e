// Upload-time relayout of FP4 weight matrices into the fragment-major layout
// of ws_pack.hpp (the counterpart of weightstream-gpu engine.rs:842-884
// pack_expert_scales / tile_major_expert).
#include "ws_internal.hpp"
#include "ws_pack.hpp"

namespace ws {

// One wave per 16-row band and 8-step scale group: lane l (row l % 16, chunks
// 4 ks + l / 16) copies its eight 16-byte chunks, so the wave reads 64-byte
// row pieces and writes 8 KB in one run, and stores its eight scale bytes (127
// past the last step, so the packed buffer is deterministic) as one word
// pair. One 16-byte chunk per thread in row order scattered the stores:
// 188.7 M weights 77.6 -> 45 us.
__global__ __launch_bounds__(256) void prepack_fp4_kernel(const uint8_t *__restrict__ w,
                                                          const uint8_t *__restrict__ s,
                                                          uint8_t *__restrict__ pw,
                                                          uint8_t *__restrict__ ps, int64_t groups,
                                                          int cols) {
    const int64_t gi = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // band * ks8 + group
    if (gi >= groups) return;
    const int lane = threadIdx.x & 63;
    const int cpr = cols / 32, ksn = cols / 128, ks8 = (ksn + 7) / 8;
    const int64_t rt = gi / ks8;
    const int k0 = (int)(gi % ks8) * 8;
    const int64_t r = rt * 16 + (lane & 15);
    const uint8_t *src = w + r * (cols / 2), *sc = s + r * cpr;
    uint4 v[8];
    uint32_t b[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int c = 4 * min(k0 + u, ksn - 1) + (lane >> 4);
        v[u] = *(const uint4 *)(src + (int64_t)c * 16);
        b[u] = sc[c];
    }
    uint64_t sb = 0;
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const bool in = k0 + u < ksn;
        if (in) *(uint4 *)(pw + ((rt * ksn + k0 + u) * 64 + lane) * 16) = v[u];
        sb |= (uint64_t)(in ? b[u] : 127u) << (8 * u);
    }
    uint8_t *po = ps + (gi * 64 + lane) * 8;
    if (((uintptr_t)ps & 7) == 0) {
        *(uint64_t *)po = sb;
    } else {
#pragma unroll
        for (int u = 0; u < 8; u++) po[u] = (uint8_t)(sb >> (8 * u));
    }
}

}  // namespace ws

using namespace ws;

extern "C" {

size_t ws_packed_fp4_scale_bytes(int64_t rows, int64_t cols) {
    if (rows <= 0 || cols <= 0 || rows % 16 || cols % 128) return 0;
    return (size_t)packed_fp4_scale_bytes(rows, cols);
}

int ws_prepack_fp4(const uint8_t *w, const uint8_t *s, int64_t rows, int64_t cols, uint8_t *pw,
                   uint8_t *ps, ws_stream_t stream) {
    if (!w || !s || !pw || !ps || rows <= 0 || cols <= 0) return WS_ERR_INVALID_ARG;
    if (rows % 16 || cols % 128 || cols > (1 << 24)) return WS_ERR_SHAPE;
    if (((uintptr_t)w | (uintptr_t)pw) & 15) return WS_ERR_INVALID_ARG;
    const int64_t groups = (rows / 16) * ((cols / 128 + 7) / 8);
    hipLaunchKernelGGL(prepack_fp4_kernel, dim3((unsigned)((groups + 3) / 4)), dim3(256), 0, stream,
                       w, s, pw, ps, groups, (int)cols);
    return launch_status();
}

}  // extern "C"
