// Upload-time relayout of FP4 weight matrices into the fragment-major layout
// of ws_pack.hpp (the counterpart of weightstream-gpu engine.rs:842-884
// pack_expert_scales / tile_major_expert).
#include "ws_internal.hpp"
#include "ws_pack.hpp"

namespace ws {

// one thread per 16-byte chunk (row r, K [32c, 32c+32)) and its scale byte; cols
// in whole 8-step scale groups (cols % 1024 == 0), so that no byte is padding
__global__ __launch_bounds__(256) void prepack_fp4_chunk_kernel(const uint8_t *__restrict__ w,
                                                          const uint8_t *__restrict__ s,
                                                          uint8_t *__restrict__ pw,
                                                          uint8_t *__restrict__ ps, int64_t rows,
                                                          int cols) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int cpr = cols / 32;  // 32-value chunks per row
    if (i >= rows * cpr) return;
    const int64_t r = i / cpr;
    const int c = (int)(i % cpr);
    const int ks = c / 4, g = c % 4, ksn = cols / 128, ks8 = (ksn + 7) / 8;
    const int64_t rt = r / 16;
    const int lane = (int)(r % 16) + 16 * g;
    const uint4 v = *(const uint4 *)(w + r * (cols / 2) + (int64_t)c * 16);
    *(uint4 *)(pw + ((rt * ksn + ks) * 64 + lane) * 16) = v;
    ps[((rt * ks8 + ks / 8) * 64 + lane) * 8 + ks % 8] = s[r * cpr + c];
}

// One wave per two steps of a 16-row band: lane l (row l % 16, chunks 4 ks + l /
// 16) copies two 16-byte chunks, so the wave reads 64-byte row pieces and writes 2
// KB in one run, and stores its two scale bytes (127 past the last step, so the
// packed buffer is deterministic) at once. A workgroup is one 8-step scale group.
// A chunk per thread in row order scatters the stores: 245.8 M weights 84.3 -> 44.5
// us (eight steps per wave 51.4: fewer loads in flight on the chip).
__global__ __launch_bounds__(256) void prepack_fp4_kernel(const uint8_t *__restrict__ w,
                                                          const uint8_t *__restrict__ s,
                                                          uint8_t *__restrict__ pw,
                                                          uint8_t *__restrict__ ps, int cols) {
    constexpr int U = 2;
    const uint32_t gi = blockIdx.x, sub = threadIdx.x >> 6;  // gi: band * ks8 + group
    const int lane = threadIdx.x & 63;
    const int cpr = cols / 32, ksn = cols / 128;
    const uint32_t ks8 = (uint32_t)(ksn + 7) / 8, band = gi / ks8;
    const int k0 = (int)((gi - band * ks8) * 8 + sub * U);
    const int64_t rt = band, r = rt * 16 + (lane & 15);
    const uint8_t *src = w + r * (cols / 2), *sc = s + r * cpr;
    uint4 v[U];
    uint32_t b[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int c = 4 * min(k0 + u, ksn - 1) + (lane >> 4);
        v[u] = *(const uint4 *)(src + (int64_t)c * 16);
        b[u] = sc[c];
    }
    uint32_t sb = 0;
#pragma unroll
    for (int u = 0; u < U; u++) {
        const bool in = k0 + u < ksn;
        if (in) *(uint4 *)(pw + ((rt * ksn + k0 + u) * 64 + lane) * 16) = v[u];
        sb |= (in ? b[u] : 127u) << (8 * u);
    }
    uint8_t *po = ps + ((int64_t)gi * 64 + lane) * 8 + sub * U;
    if (((uintptr_t)ps & 1) == 0) {
        *(uint16_t *)po = (uint16_t)sb;
    } else {
#pragma unroll
        for (int u = 0; u < U; u++) po[u] = (uint8_t)(sb >> (8 * u));
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
    // a chunk per thread where its scattered stores cost least: rows of one scale
    // group at any size, longer ones when small. us, chunks / waves: 2304 x 1024
    // 2.18 / 2.33, 16384 x 1024 4.16 / 4.67; 2304 x 2048 2.85 / 2.92, 4608 x 2048
    // 3.85 / 3.70; 512 x 3072 2.31 / 2.29; 512 x 5120 2.96 / 2.33. (Below whole
    // groups it would need a launch for the padding bytes.)
    const int64_t ks8 = (cols / 128 + 7) / 8;
    if (cols % 1024 == 0 && rows * cols * (ks8 - 1) <= 4 * 1024 * 1024) {
        const int64_t n = rows * (cols / 32);
        hipLaunchKernelGGL(prepack_fp4_chunk_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                           stream, w, s, pw, ps, rows, (int)cols);
    } else {
        hipLaunchKernelGGL(prepack_fp4_kernel, dim3((unsigned)(rows / 16 * ks8)), dim3(256), 0, stream,
                           w, s, pw, ps, (int)cols);
    }
    return launch_status();
}

}  // extern "C"
