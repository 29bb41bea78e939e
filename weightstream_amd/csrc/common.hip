// Runtime entry points and activation quantisation kernels.
//
// Reference: weightstream-cuda/kernels/actquant.cu (act_quant_ue8m0_snap :9,
// act_quant_fp8_emit :47, pack_scale_words :87), launched by
// weightstream-gpu/src/launch.rs:296-326; CPU semantics weightstream-ref
// actquant.rs:21-57.
#include "ws_internal.hpp"

#include <atomic>

namespace ws {

// One thread per element; each 32-lane half of a wave is one 1x32 block.
template <int MODE>  // 0: emit bytes, 1: snap in place
__global__ __launch_bounds__(256) void act_quant_kernel(float *xio, const float *xin, uint8_t *q,
                                                        uint8_t *s, int64_t n,
                                                        int64_t packed_offset) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    bool live = i < n;  // n % 32 == 0, so a half-wave is all live or all dead
    float x = live ? (MODE == 1 ? xio[i] : xin[i]) : 0.0f;
    uint32_t sb;
    uint32_t qb = quant_fp8_block32(x, &sb);
    if (!live) return;
    if (MODE == 1) {
        float sc = __builtin_ldexpf(1.0f, (int)sb - 127);
        xio[i] = e4m3_to_f32(qb) * sc;
    } else {
        q[i] = (uint8_t)qb;
        if ((threadIdx.x & 31) == 0) {
            s[i / 32] = (uint8_t)sb;
            if (packed_offset > 0) s[packed_offset + i / 32] = (uint8_t)sb;
        }
    }
}

// Four values per lane and kAqPasses x 4 KB of f32 per workgroup (the loads of
// all passes are issued first), a block being 8 lanes: one float4 load and one
// 4-byte store per lane where the kernel above moves a float and a byte. What
// bounds it is the vector ALU (the bytes' rounding; 94% of its cycles), no longer the
// memory instructions. 33.5 M values (M = 4096, K = 8192): 105 -> 44 us (3.8
// TB/s). Same bytes; taken when the
// operands are aligned for it (x 16 bytes, q 4).
constexpr int kAqPasses = 2;
template <int MODE>  // 0: emit bytes, 1: snap in place
__global__ __launch_bounds__(256) void act_quant4_kernel(float *xio, const float *xin, uint8_t *q,
                                                         uint8_t *s, int64_t n,
                                                         int64_t packed_offset) {
    const int64_t i0 = ((int64_t)blockIdx.x * (256 * kAqPasses) + threadIdx.x) * 4;
    const float *x = MODE == 1 ? xio : xin;
    float4 v[kAqPasses];
#pragma unroll
    for (int p = 0; p < kAqPasses; p++) {
        const int64_t i = i0 + p * 1024;  // n % 32 == 0: a block is all live or all dead
        v[p] = i < n ? *(const float4 *)(x + i) : float4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int p = 0; p < kAqPasses; p++) {
        const int64_t i = i0 + p * 1024;
        uint32_t sb;
        const uint32_t qb = quant_fp8_block32_x4(v[p], &sb);
        if (i >= n) continue;
        if (MODE == 1) {
            const float sc = __builtin_ldexpf(1.0f, (int)sb - 127);
            *(float4 *)(xio + i) =
                float4{e4m3_to_f32(qb & 0xFF) * sc, e4m3_to_f32((qb >> 8) & 0xFF) * sc,
                       e4m3_to_f32((qb >> 16) & 0xFF) * sc, e4m3_to_f32(qb >> 24) * sc};
        } else {
            *(uint32_t *)(q + i) = qb;
            if ((threadIdx.x & 7) == 0) {
                s[i / 32] = (uint8_t)sb;
                if (packed_offset > 0) s[packed_offset + i / 32] = (uint8_t)sb;
            }
        }
    }
}

__global__ __launch_bounds__(256) void pack_scale_words_kernel(const uint8_t *src, uint32_t *dst,
                                                               int64_t words) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= words) return;
    const uint8_t *p = src + i * 4;
    dst[i] = (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) |
             ((uint32_t)p[3] << 24);
}

// f32-scale activation quant: one wave per 1x128 block, two values per lane.
__global__ __launch_bounds__(256) void act_quant_f32s_kernel(const float *x, uint8_t *q, float *s,
                                                             int64_t blocks) {
    int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (b >= blocks) return;  // whole wave exits together
    int l = threadIdx.x & 63;
    const float *v = x + b * 128;
    float x0 = v[l], x1 = v[l + 64];
    float amax = fmaxf(__builtin_fabsf(x0), __builtin_fabsf(x1));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    if (!(amax >= 1e-4f)) amax = 1e-4f;  // an all-NaN block too, as the reference's `a > amax` scan
    float sc = amax / 448.0f;
    // inf / inf (a block holding an infinity) is the host's invalid-operation
    // NaN, sign bit set on x86: byte 0xFF, as block_byte
    const bool inf_blk = sc == __builtin_inff();
    const uint32_t q0 = f32_to_e4m3(rclamp(x0 / sc, -448.0f, 448.0f));
    const uint32_t q1 = f32_to_e4m3(rclamp(x1 / sc, -448.0f, 448.0f));
    q[b * 128 + l] = (uint8_t)(inf_blk && __builtin_fabsf(x0) == sc ? 0xFFu : q0);
    q[b * 128 + l + 64] = (uint8_t)(inf_blk && __builtin_fabsf(x1) == sc ? 0xFFu : q1);
    if (l == 0) s[b] = sc;
}

// The same with half a wave per block and four consecutive values per lane (one
// float4 load and one 4-byte store): 21.0 M values 39.3 -> 30.9 us. Taken for
// many values (see the launch), x 16-byte and q 4-byte aligned.
__global__ __launch_bounds__(256) void act_quant_f32s4_kernel(const float *x, uint8_t *q, float *s,
                                                              int64_t blocks) {
    const int64_t b = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5);
    const bool live = b < blocks;
    const int l = threadIdx.x & 31;
    const float4 f = *(const float4 *)(x + (live ? b : 0) * 128 + 4 * l);
    float amax = half_wave_max(fmaxf(fmaxf(__builtin_fabsf(f.x), __builtin_fabsf(f.y)),
                                     fmaxf(__builtin_fabsf(f.z), __builtin_fabsf(f.w))));
    if (!(amax >= 1e-4f)) amax = 1e-4f;  // an all-NaN block too, as the reference's `a > amax` scan
    const float sc = amax / 448.0f;
    // inf / inf (a block holding an infinity) is the host's invalid-operation
    // NaN, sign bit set on x86: byte 0xFF, as block_byte
    const bool inf_blk = sc == __builtin_inff();
    auto byte = [&](float a) -> uint32_t {
        const uint32_t c = f32_to_e4m3(rclamp(a / sc, -448.0f, 448.0f));
        return inf_blk && __builtin_fabsf(a) == sc ? 0xFFu : c;
    };
    const uint32_t w = byte(f.x) | (byte(f.y) << 8) | (byte(f.z) << 16) | (byte(f.w) << 24);
    if (!live) return;
    *(uint32_t *)(q + b * 128 + 4 * l) = w;
    if (l == 0) s[b] = sc;
}

// ---- weight encoders (weightstream-ref store.rs:357-422) -------------------
// e2m1 code with the RNE thresholds of quant.rs:139-163.
__device__ __forceinline__ uint32_t f32_to_e2m1(float v) {
    uint32_t sign = (__float_as_uint(v) >> 31) ? 8u : 0u;
    float a = __builtin_fabsf(v);
    uint32_t c = a <= 0.25f ? 0 : a < 0.75f ? 1 : a <= 1.25f ? 2 : a < 1.75f ? 3
               : a <= 2.5f ? 4 : a < 3.5f ? 5 : a <= 5.0f ? 6 : 7;
    return sign | c;
}

// FP4: one scale per row per 32 columns; a half-wave owns one block, adjacent
// lanes pair into one byte (even column in the low nibble).
__global__ __launch_bounds__(256) void weight_quant_fp4_kernel(const float *w, uint8_t *q,
                                                               uint8_t *s, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    bool live = i < n;
    float v = live ? w[i] : 0.0f;
    float amax = half_wave_max(__builtin_fabsf(v));
    const float floor_ = 6.0f * __builtin_ldexpf(1.0f, -126);
    if (amax < floor_) amax = floor_;
    int e = log2_ceil(amax / 6.0f);
    float sc = __builtin_ldexpf(1.0f, e);
    uint32_t code = f32_to_e2m1(rclamp(v / sc, -6.0f, 6.0f));
    uint32_t hi = __shfl_xor(code, 1, 64);
    if (!live) return;
    if ((threadIdx.x & 1) == 0) q[i / 2] = (uint8_t)((code & 0xF) | (hi << 4));
    if ((threadIdx.x & 31) == 0) s[i / 32] = (uint8_t)(e + 127);
}

// f32_to_e2m1 for |v| <= 6 or NaN, by rounding: from 1 up the code is the
// exponent and one mantissa bit of v rounded to nearest even in its bits,
// below 1 it is v in halves rounded to nearest even. 7 instructions fewer
// than the threshold chain; equal to it on every such input
// (tests/test_gpu_kernels.py compares all thresholds and their neighbours).
__device__ __forceinline__ uint32_t f32_to_e2m1_sat(float v) {
    const uint32_t b = __float_as_uint(v), u = b & 0x7FFFFFFFu;
    const uint32_t big = ((u + 0x1FFFFFu + ((u >> 22) & 1)) >> 22) - (127u * 2 - 2);
    const uint32_t small = (uint32_t)__builtin_rintf(__uint_as_float(u) * 2.0f);
    const uint32_t c = u < 0x3F800000u ? small : (u > 0x7F800000u ? 7u : big);
    return ((b >> 28) & 8) | c;
}

// Eight consecutive values per lane, a block being 4 lanes: two float4 loads
// and one 4-byte store per lane, and the quotient by the power-of-two scale
// as a product (the same rounding of the same real value; a block holding an
// infinity, e = 128, or nothing but NaN, 129, keeps the division). 188.7 M values: 566 ->
// 150 us (5.7 TB/s). Taken when w is 16-byte and q 4-byte aligned.
__global__ __launch_bounds__(256) void weight_quant_fp4x8_kernel(const float *w, uint8_t *q,
                                                                 uint8_t *s, int64_t n) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    const bool live = i < n;  // n % 32 == 0: a block is all live or all dead
    float4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
    if (live) {
        a = *(const float4 *)(w + i);
        b = *(const float4 *)(w + i + 4);
    }
    float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    float amax = __builtin_fabsf(v[0]);
#pragma unroll
    for (int j = 1; j < 8; j++) amax = fmaxf(amax, __builtin_fabsf(v[j]));
    // the maximum over the quad: swap neighbours, then pairs
    amax = fmaxf(amax, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(amax), 0xB1, 0xF, 0xF, false)));
    amax = fmaxf(amax, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(amax), 0x4E, 0xF, 0xF, false)));
    const float floor_ = 6.0f * __builtin_ldexpf(1.0f, -126);
    if (amax < floor_) amax = floor_;
    const int e = log2_ceil(amax / 6.0f);  // [-126, 126], 128 or 129
    uint32_t out = 0;
    if (e <= 126) {
        const float inv = __builtin_ldexpf(1.0f, -e);
#pragma unroll
        for (int j = 0; j < 8; j++)
            out |= f32_to_e2m1_sat(rclamp(v[j] * inv, -6.0f, 6.0f)) << (4 * j);
    } else {
        const float sc = __builtin_ldexpf(1.0f, e);
#pragma unroll
        for (int j = 0; j < 8; j++) out |= f32_to_e2m1(rclamp(v[j] / sc, -6.0f, 6.0f)) << (4 * j);
    }
    if (!live) return;
    *(uint32_t *)(q + i / 2) = out;
    if ((threadIdx.x & 3) == 0) s[i / 32] = (uint8_t)(e + 127);
}

// FP8: one scale per 32x32 block; a workgroup of 256 threads owns one block
// (4 values per thread), amax over the whole block.
__global__ __launch_bounds__(256) void weight_quant_fp8_kernel(const float *w, uint8_t *q,
                                                               uint8_t *s, int rows, int cols) {
    __shared__ float wmax[4];
    const int rb = blockIdx.y, cb = blockIdx.x, t = threadIdx.x;
    const int c = cb * 32 + (t & 31);
    float v[4];
    float amax = 1e-4f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        int r = rb * 32 + (t >> 5) + 8 * j;
        v[j] = (r < rows) ? w[(size_t)r * cols + c] : 0.0f;
        amax = fmaxf(amax, __builtin_fabsf(v[j]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    if ((t & 63) == 0) wmax[t >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    int e = log2_ceil(amax / 448.0f);
    float sc = __builtin_ldexpf(1.0f, e);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        int r = rb * 32 + (t >> 5) + 8 * j;
        // an infinity over inf is the host's negative NaN (byte 0xFF), as block_byte
        const uint32_t b = f32_to_e4m3(rclamp(v[j] / sc, -448.0f, 448.0f));
        if (r < rows)
            q[(size_t)r * cols + c] =
                (uint8_t)(sc == __builtin_inff() && __builtin_fabsf(v[j]) == sc ? 0xFFu : b);
    }
    if (t == 0) s[(size_t)rb * (cols / 32) + cb] = (uint8_t)(e + 127);
}

// FP8, four 32x32 blocks side by side per workgroup (32 rows x 128 columns):
// whole 512-byte row pieces are read and 128-byte ones written, four values
// per lane; the block maxima meet in LDS. The quotient is a product with
// 2^-e (block_byte, the activations' rule: the same bytes). 217.6 M values: 369 ->
// 236 us. Taken when w is 16-byte and q 4-byte aligned.
__global__ __launch_bounds__(256) void weight_quant_fp8x4_kernel(const float *w, uint8_t *q,
                                                                 uint8_t *s, int rows, int cols) {
    __shared__ float bmax[8][4];
    const int t = threadIdx.x, rg = t >> 5;   // 8 row groups of 4 rows (rg + 8j)
    const int rb = blockIdx.y, c = blockIdx.x * 128 + 4 * (t & 31), blk = (t & 31) >> 3;
    const bool in = c < cols;                 // cols % 32 == 0: a block is all in or all out
    float4 v[4];
    float amax = 1e-4f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = rb * 32 + rg + 8 * j;
        v[j] = in && r < rows ? *(const float4 *)(w + (size_t)r * cols + c)
                              : float4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
        amax = fmaxf(amax, fmaxf(fmaxf(__builtin_fabsf(v[j].x), __builtin_fabsf(v[j].y)),
                                 fmaxf(__builtin_fabsf(v[j].z), __builtin_fabsf(v[j].w))));
    amax = max8_lanes(amax);
    if ((t & 7) == 0) bmax[rg][blk] = amax;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++) amax = fmaxf(amax, bmax[k][blk]);
    const int e = log2_ceil_div448(amax);
    const float inv = block_inv_scale(e);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = rb * 32 + rg + 8 * j;
        if (in && r < rows)
            *(uint32_t *)(q + (size_t)r * cols + c) =
                block_byte(v[j].x, inv) | (block_byte(v[j].y, inv) << 8) |
                (block_byte(v[j].z, inv) << 16) | (block_byte(v[j].w, inv) << 24);
    }
    if (in && (t & 7) == 0 && rg == 0) s[(size_t)rb * (cols / 32) + c / 32] = (uint8_t)(e + 127);
}

// ws_expf on inputs lo .. lo+n-1; the lane-table variant (ws_expf_lanes) is
// evaluated beside it and any difference is reported as 0x7fbadbad.
__global__ __launch_bounds__(256) void expf_probe_kernel(uint32_t lo, uint32_t n, uint32_t *out) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    const float x = __uint_as_float(lo + min(i, n - 1));
    const uint32_t a = __float_as_uint(ws_expf(x));
    const uint32_t b = __float_as_uint(ws_expf_lanes(x, ws_lane_exp2f_tab(threadIdx.x & 63)));
    if (i < n) out[i] = a == b ? a : 0x7fbadbadu;
}

// ---- swiglu_limit10 (moe.cu:143), elementwise in moe.rs:187-201 order ----
__global__ __launch_bounds__(256) void swiglu_kernel(const float *gate, const float *up, float *out,
                                                     int64_t n, float rw) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float u = rclamp(up[i], -10.0f, 10.0f);
    float g = fminf(gate[i], 10.0f);
    out[i] = ws_silu(g) * u * rw;
}

int cu_count() {
    static std::atomic<int> cache[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    int n = cache[dev].load(std::memory_order_relaxed);
    if (n > 0) return n;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
        n = 256;
    cache[dev].store(n, std::memory_order_relaxed);
    return n;
}

}  // namespace ws

using namespace ws;

extern "C" {

int ws_built_with_hip(void) { return 1; }

int ws_get_math_mode(void) { return math_mode(); }

const char *ws_error_string(int code) {
    switch (code) {
        case WS_OK: return "ok";
        case WS_ERR_INVALID_ARG: return "weightstream-hip: invalid argument";
        case WS_ERR_SHAPE: return "weightstream-hip: unsupported shape";
        case WS_ERR_NO_DEVICE: return "weightstream-hip: no gfx950 device";
        default: return hipGetErrorString((hipError_t)code);
    }
}

int ws_init(void) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) return (int)e;
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) return WS_ERR_NO_DEVICE;
    return WS_OK;
}

int ws_expf_probe(uint32_t lo, uint32_t n, uint32_t *out, ws_stream_t stream) {
    if (!out || n == 0) return WS_ERR_INVALID_ARG;
    hipLaunchKernelGGL(expf_probe_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, lo, n, out);
    return launch_status();
}

static int act_quant_launch(int mode, float *xio, const float *x, uint8_t *q, uint8_t *s,
                            int64_t n, int64_t packed, ws_stream_t stream) {
    if (n <= 0 || n % 32) return WS_ERR_SHAPE;
    // four values per lane and two passes when the loads and stores are aligned
    // for it and the workgroups fill the chip; below, a value per lane ends
    // sooner. us, one value / four: bytes 27 x 8192 values 2.48 / 2.74, 384 K
    // 2.90 / 2.84, 1 M 4.25 / 3.13; in place 27 x 8192 2.58 / 3.33, 640 K 3.66 /
    // 3.88, 768 K 3.88 / 3.85, 1 M 4.58 / 4.03.
    if (((uintptr_t)(mode == 1 ? xio : x) & 15) == 0 && ((uintptr_t)q & 3) == 0 &&
        n >= (mode == 1 ? 768 : 384) * 1024) {
        const dim3 grid((unsigned)((n + 1024 * kAqPasses - 1) / (1024 * kAqPasses)));
        if (mode == 1)
            hipLaunchKernelGGL(act_quant4_kernel<1>, grid, dim3(256), 0, stream, xio, x, q, s, n, packed);
        else
            hipLaunchKernelGGL(act_quant4_kernel<0>, grid, dim3(256), 0, stream, xio, x, q, s, n, packed);
        return launch_status();
    }
    dim3 grid((unsigned)((n + 255) / 256));
    if (mode == 1)
        hipLaunchKernelGGL(act_quant_kernel<1>, grid, dim3(256), 0, stream, xio, x, q, s, n, packed);
    else
        hipLaunchKernelGGL(act_quant_kernel<0>, grid, dim3(256), 0, stream, xio, x, q, s, n, packed);
    return launch_status();
}

int ws_snap8(float *x, int64_t n, ws_stream_t stream) {
    if (!x) return WS_ERR_INVALID_ARG;
    return act_quant_launch(1, x, nullptr, nullptr, nullptr, n, 0, stream);
}

int ws_emit8(const float *x, uint8_t *q, uint8_t *s, int64_t n, ws_stream_t stream) {
    if (!x || !q || !s) return WS_ERR_INVALID_ARG;
    return act_quant_launch(0, nullptr, x, q, s, n, 0, stream);
}

int ws_emit8_packed(const float *x, uint8_t *q, uint8_t *s, int64_t n, ws_stream_t stream) {
    if (!x || !q || !s) return WS_ERR_INVALID_ARG;
    int64_t raw = n / 32;
    int64_t packed = (raw + 15) / 16 * 16;
    return act_quant_launch(0, nullptr, x, q, s, n, packed, stream);
}

int ws_pack_scales(const uint8_t *src, uint32_t *dst, int64_t n, ws_stream_t stream) {
    if (!src || !dst) return WS_ERR_INVALID_ARG;
    if (n <= 0 || n % 128) return WS_ERR_SHAPE;
    int64_t words = n / 128;
    hipLaunchKernelGGL(pack_scale_words_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0,
                       stream, src, dst, words);
    return launch_status();
}

int ws_act_quant_f32s(const float *x, uint8_t *q, float *s, int64_t m, int64_t k,
                      ws_stream_t stream) {
    if (!x || !q || !s) return WS_ERR_INVALID_ARG;
    if (m <= 0 || k <= 0 || k % 128) return WS_ERR_SHAPE;
    int64_t blocks = m * (k / 128);
    // us, two values per lane / four: 27 x 4096 values 2.17 / 2.32, 384 K 2.49 /
    // 2.63, 448 K 2.80 / 2.75, 1 M 3.63 / 3.29
    if (((uintptr_t)x & 15) == 0 && ((uintptr_t)q & 3) == 0 && blocks >= 448 * 8)
        hipLaunchKernelGGL(act_quant_f32s4_kernel, dim3((unsigned)((blocks + 7) / 8)), dim3(256), 0,
                           stream, x, q, s, blocks);
    else
        hipLaunchKernelGGL(act_quant_f32s_kernel, dim3((unsigned)((blocks + 3) / 4)), dim3(256), 0,
                           stream, x, q, s, blocks);
    return launch_status();
}

int ws_weight_quant_fp4(const float *w, uint8_t *q, uint8_t *s, int64_t rows, int64_t cols,
                        ws_stream_t stream) {
    if (!w || !q || !s) return WS_ERR_INVALID_ARG;
    if (rows <= 0 || cols <= 0 || cols % 32) return WS_ERR_SHAPE;
    int64_t n = rows * cols;
    // us, one value per lane / eight: 128 x 512 2.29 / 2.41, 128 x 1024 2.39 /
    // 2.42, 256 x 1024 2.54 / 2.46, 512 x 1024 3.21 / 2.52
    if (((uintptr_t)w & 15) == 0 && ((uintptr_t)q & 3) == 0 && n >= 256 * 1024) {
        hipLaunchKernelGGL(weight_quant_fp4x8_kernel, dim3((unsigned)((n + 2047) / 2048)), dim3(256),
                           0, stream, w, q, s, n);
        return launch_status();
    }
    hipLaunchKernelGGL(weight_quant_fp4_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       stream, w, q, s, n);
    return launch_status();
}

int ws_weight_quant_fp8(const float *w, uint8_t *q, uint8_t *s, int64_t rows, int64_t cols,
                        ws_stream_t stream) {
    if (!w || !q || !s) return WS_ERR_INVALID_ARG;
    if (rows <= 0 || cols <= 0 || cols % 32 || rows > (1 << 24) || cols > (1 << 24))
        return WS_ERR_SHAPE;
    // us, one block per workgroup / four: 512 x 1024 3.29 / 3.75, 768 x 1024 3.61 /
    // 3.77, 1024 x 1024 4.06 / 3.79, 2048 x 1024 5.97 / 4.66; with one or two blocks
    // across half the workgroup idles: 32768 x 64 6.07 / 6.58, 16384 x 96 5.13 / 4.55
    if (((uintptr_t)w & 15) == 0 && ((uintptr_t)q & 3) == 0 && cols >= 96 &&
        rows * cols >= 1024 * 1024) {
        hipLaunchKernelGGL(weight_quant_fp8x4_kernel,
                           dim3((unsigned)((cols + 127) / 128), (unsigned)((rows + 31) / 32)),
                           dim3(256), 0, stream, w, q, s, (int)rows, (int)cols);
        return launch_status();
    }
    dim3 grid((unsigned)(cols / 32), (unsigned)((rows + 31) / 32));
    hipLaunchKernelGGL(weight_quant_fp8_kernel, grid, dim3(256), 0, stream, w, q, s, (int)rows,
                       (int)cols);
    return launch_status();
}

int ws_swiglu(const float *gate, const float *up, float *out, int64_t n, float rw,
              ws_stream_t stream) {
    if (!gate || !up || !out) return WS_ERR_INVALID_ARG;
    if (n <= 0) return WS_ERR_SHAPE;
    hipLaunchKernelGGL(swiglu_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, gate,
                       up, out, n, rw);
    return launch_status();
}

}  // extern "C"
