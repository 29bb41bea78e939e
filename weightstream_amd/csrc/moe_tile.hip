// Grouped routed-expert GEMMs for many tokens (exact math, ws_moe_prefill): the
// gate/up and down steps over groups of up to 96 of an expert's slots.
//
// CPU semantics: weightstream-ref moe.rs:162-208 per token; the reference's
// kernels are tilelang/moe_gate_up.cu and moe_down.cu. Layouts and the meaning
// of slots are moe_grouped.hip's; the A rows are the exact bf16 values of the
// quantised tokens (gate/up) or of the quantised hidden state (down).
//
// What bounds it: with 32 or more slots per expert the bf16 matrix cores, not
// the weight stream. A workgroup takes a unit (group, column block) and its
// eight waves (two per SIMD) split the block's columns, so
//  - every FP4 weight of the unit is read once, by the one wave that uses it,
//    and converted once for all the group's rows;
//  - the A rows of a 128-K step go to LDS once for all eight waves;
//  - both stream into LDS by direct copies in whole lines (weights: the packed
//    layout's 1 KB runs), A one 128-K step ahead and the weights, which come
//    from HBM, two: with one step ahead a step took its load latency, 3.3 us
//    where its MFMAs take 1.5. Three weight stages are why a group has 96 rows
//    and not 128;
//  - a wave's instruction stream alternates MFMAs with the conversions of the
//    next 32-K sub-step's weights, as in gemm_tile.hip;
//  - gate/up: a wave holds the w1 and the w3 rows of 32 intermediate columns,
//    one FP8 1x32 block per row, so SwiGLU and the re-quantisation need no
//    other wave;
//  - gate/up sums are p0 + p1 over the two K parts of moe_grouped.hip's
//    tile-streaming body, whose bits these are: with one chain more of the
//    re-quantised h moved by an e4m3 step (4096 tokens of 384 experts, dim 4096:
//    the outputs' 2-norm error against 64 bits 9.3e-5 and 8.0e-5 for two draws,
//    6.6e-5 and 4.7e-5 so). The registers hold one sum (192 of 256 would go to
//    two), so p0 waits in scratch memory, 192 KB per workgroup that its next unit
//    takes again (6 MB per XCD: they leave its L2, 0.54 GB written): 2099 -> 2159
//    us for that prefill.
// The strips (16 rows) multiplied are those that hold routes: six
// instantiations, 16 to 96 rows.
#include "ws_internal.hpp"
#include "ws_pack.hpp"
#include "ws_tile.hpp"

namespace ws {
namespace mt {

using namespace tile;

constexpr int kThreads = 512, kWaves = 8;
constexpr int kStrips = 6;               // 16-row strips per group
constexpr int kNB = 4;                   // 16-row weight bands per wave
constexpr int kNW = 3;                   // weight stages
constexpr int kW = kWaves * kNB * 1024;  // weight bytes of a stage
constexpr int kA = kStrips * 16 * 256;   // A bytes of a stage (bf16, 128 K)
constexpr int kScale = kWaves * kNB * 256;  // scale bytes of four steps
constexpr int kMaxE = 1024;
constexpr int kPartPiece = kNB * 1024;   // bytes of a wave's first sums of one strip
// LDS: weight stages, two A stages (whole multiples of 1 KB from LDS offset 0: the
// read addresses are formed by XOR), scale words, the table of groups before
// each expert
constexpr int kOffA = kNW * kW, kOffS = kOffA + 2 * kA, kOffT = kOffS + kScale;
constexpr int kLds = kOffT + (kMaxE + 1 + kWaves) * 4;
static_assert(kLds <= 160 * 1024, "LDS");

struct Args {
    const uint8_t *a;             // bf16 A rows: gate/up [tokens][K], down [slots][K]
    const int32_t *order;         // [slots] route or -1 (gate/up)
    const float *layout_w;        // [slots] routing weight (gate/up)
    const int32_t *exp_off, *exp_cnt;
    const uint8_t *wa, *sa, *wb, *sb;  // gate/up: w1, w3; down: w2
    uint16_t *hbf;                // gate/up out: bf16 h [slots][N]
    float *out;                   // down out: f32 [slots][N]
    uint8_t *part;                // gate/up: the first K part's sums,
    int part_by_slot;             // by strip and column, or by workgroup
    int K, N, n_experts, top_k;
    float limit;
};

// One unit of 16 * MF rows or fewer: slots [slot0, slot0 + rows) of expert e,
// column block cb.
template <int MODE, int MF>
__device__ __forceinline__ void unit(const Args &p, uint8_t *lds, int e, int slot0, int rows, int cb) {
    constexpr int AL = (MF + 1) / 2;       // A copies per wave and step (four rows each)
    constexpr int L = AL + kNB, T = 4 * MF;
    constexpr int kDPer = (L + T / 2 - 1) / (T / 2), kDStep = T / 2 * kDPer / L;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int K = p.K, N = p.N, n = K / 128, ks8 = (n + 7) / 8;

    // ---- direct copies: A rows (16-byte pieces permuted by the row)
    uint32_t ao[AL];
#pragma unroll
    for (int q = 0; q < AL; q++) {
        const int row = (w * AL + q) * 4 + (lane >> 4);
        const int slot = slot0 + (row < rows ? row : 0);
        uint32_t arow = (uint32_t)slot;
        if (MODE == 0) {
            const int route = p.order[slot];
            arow = route >= 0 ? (uint32_t)(route / p.top_k) : 0u;
        }
        ao[q] = arow * (uint32_t)(2 * K) + (uint32_t)(((lane & 15) ^ (row & 15)) * 16);
    }
    // this wave's bands: gate/up w1, w3 of columns 16h of its 32; down 64
    // columns. N is whole waves' columns, so a wave's are all in it or all past
    // it (the last ones repeated, unused). One address and the stride to the
    // next band: eight pointers were spilled to scratch
    const uint32_t l16 = lane * 16, l8 = lane * 8;
    const size_t wmat = (size_t)N * (K / 2), smat = (size_t)packed_fp4_scale_bytes(N, K);
    const int c0 = MODE == 0 ? cb * 256 + 32 * w : cb * 512 + 64 * w;  // first column
    const int rt = min(c0 / 16, N / 16 - (MODE == 0 ? 2 : 4));
    const size_t wat = e * wmat + (size_t)rt * n * 1024, sat = e * smat + (size_t)rt * ks8 * 512;
    const uint8_t *const wsrc[2] = {p.wa + wat, p.wb + wat}, *const ssrc[2] = {p.sa + sat, p.sb + sat};
    auto issue_a = [&](int q, int s, int buf) {
        dma16(p.a + (size_t)s * 256 + ao[q], lds + kOffA + buf * kA + (w * AL + q) * 1024);
    };
    auto issue_w = [&](int b, int s, int buf) {
        const int m = MODE == 0 ? b & 1 : 0, h = MODE == 0 ? b >> 1 : b;
        dma16(wsrc[m] + (uint32_t)(h * n + s) * 1024u + l16, lds + buf * kW + (w * kNB + b) * 1024);
    };
    auto issue_scales = [&](int grp) {  // steps 4 grp .. 4 grp + 3
#pragma unroll
        for (int b = 0; b < kNB; b++)
            dma4(ssrc[MODE == 0 ? b & 1 : 0] +
                     (uint32_t)((MODE == 0 ? b >> 1 : b) * ks8 + (grp >> 1)) * 512u + (grp & 1) * 4 + l8,
                 lds + kOffS + (w * kNB + b) * 256);
    };
    issue_scales(0);
#pragma unroll
    for (int q = 0; q < AL; q++) issue_a(q, 0, 0);
#pragma unroll
    for (int s = 0; s < kNW - 1; s++)
#pragma unroll
        for (int b = 0; b < kNB; b++) issue_w(b, min(s, n - 1), s);

    v4f acc[MF][kNB];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int b = 0; b < kNB; b++) acc[i][b] = v4f{0.f, 0.f, 0.f, 0.f};

    // ---- LDS reads: sub-step j of a row is 16-byte piece 4g + j
    const uint32_t ldsb = lds_addr(lds);
    const uint32_t ra = ldsb + kOffA + r * 256 + ((4 * g) ^ r) * 16;
    const uint32_t rw = ldsb + w * kNB * 1024 + lane * 16;
    const uint32_t rs = ldsb + kOffS + w * kNB * 256 + lane * 4;
    uint32_t sw[kNB];
    float fs[kNB];
    // a lane's scale bytes of four steps, one word per band: read before the first
    // of them, complete when this returns
    auto read_scales = [&]() {
        seq([&](auto bc) {
            constexpr int b = decltype(bc)::value;
            sw[b] = rd32<b * 256>(rs);
        }, WS_SEQ(kNB, b));
        lds_wait_all();
        seq([&](auto bc) { lds_ready(sw[decltype(bc)::value]); }, WS_SEQ(kNB, b));
    };
    // the weights and scales of a step are this wave's own copies: they are read
    // and the first sub-step's fragments converted before the step's barrier, so
    // that only A is waited for after it
    u32x4v xa[4], xw[kNB];
    uint32_t bq[2][kNB][4];
    auto read_w = [&](auto bc, uint32_t st) {
        constexpr int b = decltype(bc)::value;
        xw[b] = rd128<b * 1024>(rw + st);
    };
    auto conv_b = [&](auto jc, auto pc) {  // piece p: band p / 4
        constexpr int j = decltype(jc)::value, pp = decltype(pc)::value, b = pp / 4, q = pp % 4;
        bq[j & 1][b][q] = cvt4<q>(xw[b][j], fs[b]);
    };
    auto frag = [](const uint32_t (&x)[4]) {
        return __builtin_bit_cast(v8bf, u32x4v{x[0], x[1], x[2], x[3]});
    };
    using Z = std::integral_constant<int, 0>;
    auto settle_w = [&](int s) {  // after the wait for read_w
        seq([&](auto bc) {
            constexpr int b = decltype(bc)::value;
            lds_ready(xw[b]);
            fs[b] = e8m0_to_f32((sw[b] >> (8 * (s & 3))) & 0xFF);
        }, WS_SEQ(kNB, b));
    };
    mem_order();
    wait_vm<(kNW - 2) * kNB>();
    read_scales();
    seq([&](auto bc) { read_w(bc, 0); }, WS_SEQ(kNB, b));
    lds_wait_all();
    settle_w(0);
    seq([&](auto pc) { conv_b(Z{}, pc); }, WS_SEQ(16, p));

    // gate/up: the step at which the second K part begins (0: it is the whole),
    // and where the first one's sums of strip i wait, 16 bytes per lane and band
    int kh = 0, kend;
    if (MODE == 0) k_part8(n, 1, 2, kh, kend);
    if (c0 >= N) kh = 0;  // uniform: a wave past the last column keeps nothing
    const uint32_t pstride = (uint32_t)(MODE == 0 && p.part_by_slot ? N / 32 : kWaves) * kPartPiece;
    auto part_at = [&]() {  // strip 0's; formed at each use: nothing is held over the loop
        int sl = slot0;
        __asm__ volatile("" : "+s"(sl));
        const size_t at = p.part_by_slot ? (size_t)(sl / 16) * (N / 32) + c0 / 32
                                         : (size_t)(blockIdx.x * kStrips) * kWaves + w;
        return p.part + at * kPartPiece + l16;
    };

    int w1 = 1;  // (s + 1) % kNW
    for (int s = 0; s < n; s++) {
        if (MODE == 0 && s == kh && kh > 0) {  // uniform
            uint8_t *const pt = part_at();
#pragma unroll
            for (int i = 0; i < MF; i++)
#pragma unroll
                for (int b = 0; b < kNB; b++) {
                    *(v4f *)(pt + i * (size_t)pstride + b * 1024) = acc[i][b];
                    acc[i][b] = v4f{0.f, 0.f, 0.f, 0.f};
                }
        }
        raw_barrier();  // step s is in LDS; the other stage has been read by every wave
        const uint32_t a0 = ra + (s & 1) * kA;
        const uint32_t stn = w1 * kW;
        const int w2 = w1 == kNW - 1 ? 0 : w1 + 1;  // (s + kNW - 1) % kNW
        auto read_a = [&](auto tc) {
            constexpr int tt = decltype(tc)::value, i = tt % MF, j = tt / MF;
            xa[tt % 4] = rd128<i * 4096>(a0 ^ (j << 4));
        };
        seq([&](auto tc) { read_a(tc); }, WS_SEQ(3, t));
        if ((s & 3) == 0 && s + 4 < n) issue_scales((s >> 2) + 1);
        // past the last step: repeated, not read
        const int sla = min(s + 1, n - 1), slw = min(s + kNW - 1, n - 1);
        pin();
        seq([&](auto tc) {
            constexpr int tt = decltype(tc)::value, i = tt % MF, j = tt / MF;
            constexpr auto wr = [](int x) constexpr { return x == 3 * MF ? kNB : 0; };
            // the next step's weights and scales, where this step's are dead
            if constexpr (wr(tt) > 0) {
                // A of step s + 1 and older copies have landed, the weights of the
                // one after may be in flight
                mem_order();
                wait_vm<(kNW - 2) * kNB>();
                if (((s + 1) & 3) == 0) read_scales();
                seq([&](auto bc) { read_w(bc, stn); }, WS_SEQ(kNB, b));
            }
            if constexpr (tt + 3 < T) read_a(std::integral_constant<int, tt + 3>{});
            // A of this strip was read three strips ago
            lds_wait<(tt + 1 < T) + (tt + 2 < T) + (tt + 3 < T) + wr(tt) + wr(tt - 1) + wr(tt - 2)>();
            lds_ready(xa[tt % 4]);
            pin();
            constexpr int kX = MF > 2 ? 2 : MF - 1;  // the strip that has them (j = 3)
            seq([&](auto bc) {
                constexpr int b = decltype(bc)::value;
                acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    frag(bq[j & 1][b]), __builtin_bit_cast(v8bf, xa[tt % 4]), acc[i][b], 0, 0, 0);
                pin();
                if constexpr (b == kNB / 2 && tt % kDStep == 0 && tt / kDStep * kDPer < L)
                    seq([&](auto qc) {
                        constexpr int q = tt / kDStep * kDPer + decltype(qc)::value;
                        if constexpr (q < AL) issue_a(q, sla, (s + 1) & 1);
                        else if constexpr (q < L) issue_w(q - AL, slw, w2);
                    }, WS_SEQ(kDPer, q));
                if constexpr (j == 3 && i == kX && b == 0) {
                    // newer reads: A issued at the strips of this sub-step so far
                    constexpr int newer = (3 < MF) + (kX >= 1 && 4 < MF) + (kX >= 2 && 5 < MF);
                    lds_wait<newer>();
                    settle_w(s + 1);
                }
                // the next sub-step's fragments (after the last: the next step's first)
                constexpr int f = j == 3 ? kX : 0;
                constexpr int slot = (i - f) * kNB + b, slots = (MF - f) * kNB;
                if constexpr (slot >= 0) {
                    constexpr int lo = slot * 16 / slots, hi = (slot + 1) * 16 / slots;
                    seq([&](auto pc) {
                        conv_b(std::integral_constant<int, (j + 1) % 4>{},
                               std::integral_constant<int, lo + decltype(pc)::value>{});
                    }, WS_SEQ(hi - lo, p));
                }
                pin();
            }, WS_SEQ(kNB, b));
        }, WS_SEQ(T, t));
        w1 = w2;
    }
    // the first K part's sums, loaded two strips ahead of their use
    v4f p0[2][kNB];
    const uint8_t *const pt = part_at();
    auto load_p0 = [&](int i) {
#pragma unroll
        for (int b = 0; b < kNB; b++) {
            p0[i & 1][b] = v4f{0.f, 0.f, 0.f, 0.f};
            if (kh > 0) p0[i & 1][b] = *(const v4f *)(pt + i * (size_t)pstride + b * 1024);
        }
    };
    if (MODE == 0) {
        load_p0(0);
        if (MF > 1) load_p0(1);
    }
    wait_vm<0>();  // the repeated copies still write this workgroup's LDS

    // ---- store: columns 4g .. 4g + 3 of a band, row r of a strip
    if (MODE == 1) {
#pragma unroll
        for (int i = 0; i < MF; i++) {
            const int row = 16 * i + r;
            if (row >= rows) continue;
#pragma unroll
            for (int b = 0; b < kNB; b++) {
                const int col = c0 + 16 * b + 4 * g;
                if (col < N)
                    *(float4 *)(p.out + (size_t)(slot0 + row) * N + col) =
                        float4{acc[i][b][0], acc[i][b][1], acc[i][b][2], acc[i][b][3]};
            }
        }
        return;
    }
    const uint64_t tab = ws_lane_exp2f_tab(lane);
    float rwt[MF];
#pragma unroll
    for (int i = 0; i < MF; i++)
        rwt[i] = p.layout_w[slot0 + (16 * i + r < rows ? 16 * i + r : 0)];
#pragma unroll
    for (int i = 0; i < MF; i++) {
        if (16 * i >= rows) continue;  // uniform
        const int row = 16 * i + r;
        float hv[2][4], m = 0.0f;
        v4f sum[kNB];
#pragma unroll
        for (int b = 0; b < kNB; b++)
#pragma unroll
            for (int v = 0; v < 4; v++) sum[b][v] = p0[i & 1][b][v] + acc[i][b][v];
        if (i + 2 < MF) load_p0(i + 2);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                float gv = sum[2 * h][v], uv = sum[2 * h + 1][v];
                if (p.limit > 0.0f) {
                    uv = rclamp(uv, -p.limit, p.limit);
                    gv = fminf(gv, p.limit);
                }
                hv[h][v] = ws_silu_lanes(gv, tab) * uv * rwt[i];
                m = fmaxf(m, __builtin_fabsf(hv[h][v]));
            }
        // the row's 1x32 block: this lane's eight values and those of the lanes
        // of the other K groups; the rule of quant_fp8_block32
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        if (!(m >= 1e-4f)) m = 1e-4f;
        const int ex = log2_ceil_div448(m);
        const float inv = block_inv_scale(ex), sc = e8m0_to_f32((uint32_t)(ex + 127) & 0xFF);
        if (row >= rows || c0 >= N) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t hb[2];
#pragma unroll
            for (int q = 0; q < 2; q++)
                hb[q] = __builtin_bit_cast(
                    uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                                  block_byte(hv[h][2 * q], inv) | (block_byte(hv[h][2 * q + 1], inv) << 8),
                                  sc, false));
            *(uint2 *)(p.hbf + (size_t)(slot0 + row) * N + c0 + 16 * h + 4 * g) = uint2{hb[0], hb[1]};
        }
    }
}

template <int MODE>
__global__ __launch_bounds__(kThreads) void moe_tile_kernel(const Args p) {
    extern __shared__ __align__(16) uint8_t m_lds[];
    int *const pre = (int *)(m_lds + kOffT);   // [kMaxE + 1] groups of the experts before e
    int *const wsum = pre + kMaxE + 1;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    int g2[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int e = 2 * t + h;
        g2[h] = e < p.n_experts ? (p.exp_cnt[e] + 16 * kStrips - 1) / (16 * kStrips) : 0;
    }
    int v = g2[0] + g2[1];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(v, off, 64);
        if (lane >= off) v += o;
    }
    if (lane == 63) wsum[w] = v;
    __syncthreads();
    int before = 0, total = 0;
    for (int k = 0; k < kWaves; k++) {
        if (k < w) before += wsum[k];
        total += wsum[k];
    }
    const int first = before + v - g2[0] - g2[1];
    pre[2 * t] = first;
    pre[2 * t + 1] = first + g2[0];
    if (t == 0) pre[kMaxE] = total;
    __syncthreads();

    // Units in (expert, column block, group) order: the groups of an expert that
    // stream the same weights are neighbours, then its column blocks, which
    // share A rows; neighbours run on one XCD (the hardware deals workgroup b to
    // XCD b % 8) and meet in its L2. (Handing units out one by one from a queue
    // per XCD instead, as they have 1 to 6 strips, changed nothing: 1383 / 1357
    // us for the gate/up step of 4096 tokens.)
    const int ncb = (p.N + (MODE == 0 ? 255 : 511)) / (MODE == 0 ? 256 : 512);
    const int G = gridDim.x, b = blockIdx.x;
    const int pb = G % 8 == 0 ? (b % 8) * (G / 8) + b / 8 : b;
    for (int u = pb; u < total * ncb; u += G) {
        __syncthreads();  // every wave has read the last unit's A
        const int grp = u / ncb;
        int lo = 0, hi = p.n_experts;  // pre[lo] <= grp < pre[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (pre[mid] <= grp) lo = mid;
            else hi = mid;
        }
        const int e = __builtin_amdgcn_readfirstlane(lo);
        // the expert's strips shared out evenly over its groups
        const int ng = __builtin_amdgcn_readfirstlane(pre[lo + 1] - pre[lo]);
        const int ue = __builtin_amdgcn_readfirstlane(u - pre[lo] * ncb);
        const int cb = ue / ng, gi = ue - cb * ng;
        const int cnt = __builtin_amdgcn_readfirstlane(p.exp_cnt[e]), ns = (cnt + 15) / 16;
        const int rel = gi * ns / ng * 16;
        const int slot0 = __builtin_amdgcn_readfirstlane(p.exp_off[e]) + rel;
        const int rows = min((gi + 1) * ns / ng * 16, cnt) - rel;
        switch ((rows + 15) / 16) {
            case 6: unit<MODE, 6>(p, m_lds, e, slot0, rows, cb); break;
            case 5: unit<MODE, 5>(p, m_lds, e, slot0, rows, cb); break;
            case 4: unit<MODE, 4>(p, m_lds, e, slot0, rows, cb); break;
            case 3: unit<MODE, 3>(p, m_lds, e, slot0, rows, cb); break;
            case 2: unit<MODE, 2>(p, m_lds, e, slot0, rows, cb); break;
            default: unit<MODE, 1>(p, m_lds, e, slot0, rows, cb); break;
        }
    }
}

}  // namespace mt

// 0: no scratch needed (one K part), 1: a slice per workgroup (48 MB, taken again
// by its next unit), 2: where those do not fit (few slots), a piece per strip and
// 32 columns; -1: neither fits.
int moe_tile_parts(size_t part_bytes, int slots, int dim, int inter) {
    if ((dim / 128 + kU - 1) / kU < 2) return 0;
    if ((size_t)cu_count() * mt::kStrips * mt::kWaves * mt::kPartPiece <= part_bytes) return 1;
    return (size_t)(slots / 16) * (inter / 32) * mt::kPartPiece <= part_bytes ? 2 : -1;
}

int moe_tile_glu(const uint16_t *xbf, const int32_t *order, const float *layout_w,
                 const int32_t *exp_off, const int32_t *exp_cnt, const uint8_t *w1,
                 const uint8_t *s1, const uint8_t *w3, const uint8_t *s3, uint16_t *hbf,
                 uint8_t *part, size_t part_bytes, int slots, int dim, int inter, int n_experts,
                 int top_k, float limit, hipStream_t stream) {
    const int mode = moe_tile_parts(part_bytes, slots, dim, inter);
    if (mode < 0) return WS_ERR_SHAPE;
    const mt::Args p{(const uint8_t *)xbf, order, layout_w, exp_off, exp_cnt, w1, s1, w3, s3, hbf,
                     nullptr, part, mode == 2, dim, inter, n_experts, top_k, limit};
    hipLaunchKernelGGL(mt::moe_tile_kernel<0>, dim3((unsigned)cu_count()), dim3(mt::kThreads),
                       mt::kLds, stream, p);
    return launch_status();
}

int moe_tile_down(const uint16_t *hbf, const int32_t *exp_off, const int32_t *exp_cnt,
                  const uint8_t *w2, const uint8_t *s2, float *out, int dim, int inter,
                  int n_experts, hipStream_t stream) {
    const mt::Args p{(const uint8_t *)hbf, nullptr, nullptr, exp_off, exp_cnt, w2, s2, nullptr,
                     nullptr, nullptr, out, nullptr, 0, inter, dim, n_experts, 1, 0.0f};
    hipLaunchKernelGGL(mt::moe_tile_kernel<1>, dim3((unsigned)cu_count()), dim3(mt::kThreads),
                       mt::kLds, stream, p);
    return launch_status();
}

}  // namespace ws
