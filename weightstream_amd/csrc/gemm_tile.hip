// Block-scaled FP8 GEMM for many rows with bf16 results (exact math): C[M,N] =
// A[M,K] . B[N,K]^T with whole-K output tiles; weight scales per 32 x 32 (UE8M0)
// or per 128 x 128 (f32).
//
// Reference semantics: weightstream-cuda/kernels/fp8_gemm_tile.cu:28-92 and
// weightstream-ref actquant.rs:110-170.
//
// What bounds it: the bf16 matrix cores. A 128-K step of a 256 x 256 tile is
// 4096 cycles of MFMA per SIMD, and everything else of the step has to fit
// beside it:
//  - the FP8 bytes of both operands go straight from global memory to LDS in
//    whole 128-byte lines, two 128-K stages deep, so the loads of a step have
//    the step before it to arrive and no register or store instruction is
//    spent on them;
//  - e4m3 -> bf16 conversions run on the vector ALU while the matrix
//    core is busy: a wave's stream alternates them with MFMAs (measured on
//    two waves per SIMD: 32 MFMAs alone 98.5, with 32 conversions between
//    them 104; grouped into blocks of one kind they add up instead). Per
//    16 x 64 strip of a 32-K sub-step a wave reads and converts the next
//    strip's A fragment and a part of the next sub-step's weight fragments;
//  - LDS reads are 8 bytes per lane and sub-step; lanes of odd K groups take
//    the upper half of their 16 bytes first, so the halves of a 16-byte bank
//    group are both in use;
//  - the weights are the first MFMA operand, so a lane holds four adjacent
//    columns of a row and stores them at once.
// One barrier per 128-K step. No split over K: partials of this size cost more
// than the step overlap they save (the split-K pipeline's reduction took 61 us
// at M = 4096, N = 4096).
// bf16 results only: one chain over the whole K rounds an f32 result more than
// the kernels that split it (2-norm error at K = 5120 1.2e-7 against 0.7e-7; sums
// beside the chain every 256 or 512 K 0.8e-7 and 0.7e-7, the latter still above
// at some shapes). Beside bf16's own rounding (1.7e-3) it cannot be seen.
#include "ws_internal.hpp"
#include "ws_kp.hpp"
#include "ws_tile.hpp"

namespace ws {
namespace tile {

template <int MF, int NB, int WM, int WN, int NS, int SMODE>
struct Geom {
    static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
    static constexpr int BM = 16 * MF * WM, BN = 16 * NB * WN;
    static constexpr int kA = BM * 128, kB = BN * 128, kStage = kA + kB;
    static constexpr int AL = kA / 1024 / kWaves, BL = kB / 1024 / kWaves;
    // weight scale rows: one per 32 weight rows, or per 128 (f32)
    static constexpr int kSDiv = SMODE == kF32s ? 128 : 32;
    static constexpr int SR = (BN + kSDiv - 1) / kSDiv;
    static constexpr int kScRows = BM + (SR + 15) / 16 * 16;
    static constexpr int kSc = kScRows * 16;     // four steps' words of every row
    static constexpr int SL = (kScRows / 16 + kWaves - 1) / kWaves;
    static constexpr int L = AL + BL;            // a wave's direct loads of a stage
    static constexpr int kLds = NS * kStage + 2 * kSc;
    static_assert(kA % (1024 * kWaves) == 0 && kB % (1024 * kWaves) == 0, "whole loads per wave");
    static_assert(kLds <= 160 * 1024, "LDS");
    static_assert(NS >= 2 && NS <= 5, "scale words are loaded four steps ahead and read one ahead");
};

struct Args {
    const uint8_t *A, *B;
    const uint8_t *SA, *SB;
    uint16_t *C;
    int M, N, K, ntm, ntn;
};

// Tile of workgroup b: the hardware deals workgroups to the 8 XCDs round
// robin, so XCD x gets a contiguous run of the tile order, and the order walks
// blocks of four row tiles column by column: the tiles that share an XCD's L2
// share their A and weight rows.
__device__ __forceinline__ void tile_of(int b, int ntm, int ntn, int &mt, int &nt) {
    const int T = ntm * ntn, q = T / 8, rem = T % 8, x = b & 7;
    const int l = x * q + min(x, rem) + (b >> 3);
    const int wide = 4 * ntn, grp = l / wide, first = grp * 4, gm = min(4, ntm - first);
    mt = first + (l - grp * wide) % gm;
    nt = (l - grp * wide) / gm;
}

template <int MF, int NB, int WM, int WN, int NS, int SMODE>
__global__ __launch_bounds__(64 * WM * WN) void gemm_tile_kernel(const Args p) {
    using G = Geom<MF, NB, WM, WN, NS, SMODE>;
    extern __shared__ __align__(16) uint8_t t_lds[];
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int wm = w % WM, wn = w / WM;
    int mt, nt;
    tile_of(blockIdx.x, p.ntm, p.ntn, mt, nt);
    const int m0 = mt * G::BM, n0 = nt * G::BN;
    const int M = p.M, N = p.N, K = p.K, n = K / 128;

    // ---- direct loads. LDS rows keep their 16-byte pieces permuted by the
    // row: piece c of row `row` sits at c ^ (row / 2 % 8). Row offsets are
    // 32-bit (host check) from a uniform base.
    uint32_t ao[G::AL], bo[G::BL], so[G::SL];
#pragma unroll
    for (int q = 0; q < G::AL; q++) {
        const int o = (w * G::AL + q) * 1024 + lane * 16, row = o >> 7, c = (o >> 4) & 7;
        ao[q] = (uint32_t)min(m0 + row, M - 1) * (uint32_t)K + (c ^ ((row >> 1) & 7)) * 16;
    }
#pragma unroll
    for (int q = 0; q < G::BL; q++) {
        const int o = (w * G::BL + q) * 1024 + lane * 16, row = o >> 7, c = (o >> 4) & 7;
        bo[q] = (uint32_t)min(n0 + row, N - 1) * (uint32_t)K + (c ^ ((row >> 1) & 7)) * 16;
    }
    // scale words of four steps: 16 rows x 4 words per instruction, rows past
    // the last one (and instructions past the last 16 rows) repeat a valid one
    const uint8_t *const ssrc[2] = {p.SA, p.SB};
    int sinst[G::SL];
#pragma unroll
    for (int q = 0; q < G::SL; q++) {
        sinst[q] = min(w * G::SL + q, G::kScRows / 16 - 1);
        const int row = sinst[q] * 16 + (lane >> 2);
        const int srow = row < G::BM ? min(m0 + row, M - 1)
                                     : min(n0 / G::kSDiv + min(row - G::BM, G::SR - 1),
                                           (N + G::kSDiv - 1) / G::kSDiv - 1);
        so[q] = (uint32_t)srow * (uint32_t)n;
    }
    // load q (of L) of a stage
    auto issue1 = [&](int q, const uint8_t *ab, const uint8_t *bb, uint8_t *base) {
        if (q < G::AL) dma16(ab + ao[q], base + (w * G::AL + q) * 1024);
        else dma16(bb + bo[q - G::AL], base + G::kA + (w * G::BL + q - G::AL) * 1024);
    };
    auto issue_scales = [&](int grp) {
        uint8_t *base = t_lds + NS * G::kStage + (grp & 1) * G::kSc;
        const int word = min(grp * 4 + (lane & 3), n - 1);
#pragma unroll
        for (int q = 0; q < G::SL; q++)
            dma4(ssrc[sinst[q] * 16 >= G::BM] + (size_t)(so[q] + word) * 4, base + sinst[q] * 256);
    };

    // ---- LDS read addresses of this lane: sub-step j (8 K values per lane)
    // is 16-byte piece 2g + j / 2 of the row, half (j + g) % 2 of it
    const uint32_t ldsb = lds_addr(t_lds);
    const uint32_t ra = ldsb + (wm * 16 * MF + r) * 128 + ((2 * g) ^ ((r >> 1) & 7)) * 16 + (g & 1) * 8;
    const uint32_t rb = ldsb + G::kA + (wn * 16 * NB + r) * 128 + ((2 * g) ^ ((r >> 1) & 7)) * 16 +
                        (g & 1) * 8;
    const uint32_t rsa = ldsb + NS * G::kStage + (wm * 16 * MF + r) * 16 + (SMODE == kUe8m0 ? g : 0);
    const uint32_t rsb = ldsb + NS * G::kStage + G::BM * 16 + (SMODE == kUe8m0 ? g : 0) +
                         wn * 16 * NB / G::kSDiv * 16;

    constexpr int kHalf = MF / 2, kRB = (NB + kHalf - 1) / kHalf;  // weight fragments per strip
    constexpr int T = 4 * MF;
    // stage loads: kDPer of them every kDStep strips, over the first half
    constexpr int kDPer = (G::L + T / 2 - 1) / (T / 2), kDStep = T / 2 * kDPer / G::L;
    // weight fragments read at strip tt (converted kHalf strips later, for the
    // next sub-step)
    auto nb_reads = [](int tt) constexpr {
        const int i = tt % MF, j = tt / MF;
        if (tt < 0 || j >= 3 || i >= kHalf) return 0;
        const int left = NB - i * kRB;
        return left < 0 ? 0 : left < kRB ? left : kRB;
    };
    // the next step's scale words are read where this step's are dead: the
    // weight words at the first strip of the last sub-step (whose weight
    // fragments are converted by then), A word q one strip after strip q's
    // last conversion, the last two at the last strip
    constexpr int kWS = (16 * NB + G::kSDiv - 1) / G::kSDiv;  // weight words
    auto sc_first = [](int tt) constexpr { return tt == 3 * MF ? MF : tt - 3 * MF - 1; };
    auto sc_reads = [](int tt) constexpr {
        return tt < 3 * MF ? 0 : tt == 3 * MF ? kWS : tt < T - 1 ? 1 : 2;
    };

    v4f acc[MF][NB], prod[SMODE == kF32s ? MF : 1][NB];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[i][b] = v4f{0.f, 0.f, 0.f, 0.f};

    issue_scales(0);
#pragma unroll
    for (int q = 0; q < NS - 1; q++) {
        const int sq = min(q, n - 1);
#pragma unroll
        for (int k = 0; k < G::L; k++)
            issue1(k, p.A + (size_t)sq * 128, p.B + (size_t)sq * 128, t_lds + q * G::kStage);
    }
    // the scales of the step: word q is A strip q, or weight word q - MF
    uint32_t sw[MF + kWS];
    float fs[MF + kWS];
    auto read_scale = [&](auto qc, uint32_t sc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (q < MF)
            sw[q] = SMODE == kUe8m0 ? rd8<q * 256>(rsa + sc) : rd32<q * 256>(rsa + sc);
        else {
            constexpr int off = (q - MF) * 16;
            sw[q] = SMODE == kUe8m0 ? rd8<off>(rsb + sc) : rd32<off>(rsb + sc);
        }
    };
    auto conv_scale = [&](auto qc) {
        constexpr int q = decltype(qc)::value;
        lds_ready(sw[q]);
        fs[q] = SMODE == kUe8m0 ? e8m0_to_f32(sw[q]) : __uint_as_float(sw[q]);
    };
    mem_order();
    wait_vm<(NS - 2) * G::L>();
    raw_barrier();
    seq([&](auto qc) { read_scale(qc, 0); }, WS_SEQ(MF + kWS, q));
    lds_wait_all();
    seq([&](auto qc) { conv_scale(qc); }, WS_SEQ(MF + kWS, q));

    int cur = 0;  // s % NS
    for (int s = 0; s < n; s++) {
        // step s is in LDS once at most the NS - 2 newer stages are in flight
        // (the scale words of a group of four steps were issued four steps ago)
        mem_order();
        wait_vm<(NS - 2) * G::L>();
        raw_barrier();  // the stage of step s - 1 has been read by every wave
        const uint32_t st = cur * G::kStage;
        const uint32_t a0 = ra + st, b0 = rb + st;
        const uint32_t scn = (((s + 1) >> 2) & 1) * G::kSc + ((s + 1) & 3) * 4;
        u32x2v xa[3], xb[NB];
        uint32_t bq[2][NB][4], aq[2][4];
        auto read_a = [&](auto tc) {
            constexpr int tt = decltype(tc)::value, i = tt % MF, j = tt / MF;
            xa[tt % 3] = rd64<i * 2048>(a0 ^ ((j >> 1) << 4) ^ ((j & 1) << 3));
        };
        auto read_b = [&](auto jc, auto bc) {
            constexpr int j = decltype(jc)::value, b = decltype(bc)::value;
            xb[b] = rd64<b * 2048>(b0 ^ ((j >> 1) << 4) ^ ((j & 1) << 3));
        };
        auto b_scale = [&](int b) {
            return SMODE == kUe8m0 ? fs[MF + 16 * b / G::kSDiv] : 1.0f;
        };
        auto conv_b = [&](auto jc, auto bc, auto pc) {
            constexpr int j = decltype(jc)::value, b = decltype(bc)::value, q = decltype(pc)::value;
            if constexpr (q == 0) lds_ready(xb[b]);
            bq[j & 1][b][q] = cvt8<q>(xb[b], b_scale(b));
        };
        auto conv_a = [&](auto tc, auto pc) {
            constexpr int tt = decltype(tc)::value, q = decltype(pc)::value;
            if constexpr (q == 0) lds_ready(xa[tt % 3]);
            aq[tt & 1][q] = cvt8<q>(xa[tt % 3], SMODE == kUe8m0 ? fs[tt % MF] : 1.0f);
        };
        auto frag = [](const uint32_t (&x)[4]) {
            return __builtin_bit_cast(v8bf, u32x4v{x[0], x[1], x[2], x[3]});
        };
        using Z = std::integral_constant<int, 0>;
        // the first strip's operands
        read_b(Z{}, Z{});
        read_a(Z{});
        seq([&](auto bc) { read_b(Z{}, std::integral_constant<int, decltype(bc)::value + 1>{}); },
            WS_SEQ(NB - 1, b));
        read_a(std::integral_constant<int, 1>{});
        read_a(std::integral_constant<int, 2>{});
        if ((s & 3) == 0 && s + 4 < n) issue_scales((s >> 2) + 1);
        const int last = cur == 0 ? NS - 1 : cur - 1;  // (s + NS - 1) % NS
        const int sl = min(s + NS - 1, n - 1);  // past the last step: repeated, not read
        const uint8_t *const ab = p.A + (size_t)sl * 128, *const bb = p.B + (size_t)sl * 128;
        uint8_t *const dst = t_lds + last * G::kStage;
        cur = cur == NS - 1 ? 0 : cur + 1;
        lds_wait<NB + 1>();
        seq([&](auto pc) { conv_a(Z{}, pc); }, WS_SEQ(4, p));
        seq([&](auto pc) { conv_b(Z{}, Z{}, pc); }, WS_SEQ(4, p));
        pin();
        seq([&](auto tc) {
            constexpr int tt = decltype(tc)::value, i = tt % MF, j = tt / MF;
            // reads: the next sub-step's weight fragments, the next step's
            // scales, A three strips ahead
            auto next_b = [&]() {
                if constexpr (nb_reads(tt) > 0)
                    seq([&](auto qc) {
                        read_b(std::integral_constant<int, j + 1>{},
                               std::integral_constant<int, i * kRB + decltype(qc)::value>{});
                    }, WS_SEQ(nb_reads(tt), q));
            };
            if constexpr (tt > 0) next_b();  // strip 0 still converts the step's first ones
            if constexpr (sc_reads(tt) > 0)
                seq([&](auto qc) {
                    read_scale(std::integral_constant<int, sc_first(tt) + decltype(qc)::value>{}, scn);
                }, WS_SEQ(sc_reads(tt), q));
            if constexpr (tt + 3 < T) read_a(std::integral_constant<int, tt + 3>{});
            pin();
            // an MFMA, then the conversions that fit beside it
            seq([&](auto bc) {
                constexpr int b = decltype(bc)::value;
                if constexpr (SMODE == kF32s) {
                    const v4f z = {0.f, 0.f, 0.f, 0.f};
                    prod[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        frag(bq[j & 1][b]), frag(aq[tt & 1]), j == 0 ? z : prod[i][b], 0, 0, 0);
                } else {
                    acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        frag(bq[j & 1][b]), frag(aq[tt & 1]), acc[i][b], 0, 0, 0);
                }
                pin();
                // a load of stage s + NS - 1, spread over the strips: issued all
                // at once they fill the memory pipe's queue and the wave waits
                if constexpr (b == NB / 2 && tt % kDStep == 0 && tt / kDStep * kDPer < G::L)
                    seq([&](auto qc) {
                        constexpr int q = tt / kDStep * kDPer + decltype(qc)::value;
                        if constexpr (q < G::L) issue1(q, ab, bb, dst);
                    }, WS_SEQ(kDPer, q));
                if constexpr (tt == 0 && b + 1 < NB) {  // the step's first weight fragments
                    lds_wait<NB - b + 1>();
                    seq([&](auto pc) {
                        conv_b(Z{}, std::integral_constant<int, b + 1>{}, pc);
                    }, WS_SEQ(4, p));
                }
                if constexpr (b == 0 && tt > 0 && tt + 1 < T)
                    // A of strip tt + 1 was read two strips ago: newer reads are A of
                    // tt + 2 and tt + 3 and the others of this strip and the last
                    lds_wait<(tt + 2 < T) + (tt + 3 < T) + nb_reads(tt) + nb_reads(tt - 1) +
                             sc_reads(tt) + sc_reads(tt - 1)>();
                if constexpr (b == NB - 1 && tt == 0) lds_wait<2>();
                constexpr int lo = 4 * b / NB, hi = 4 * (b + 1) / NB;
                if constexpr (tt + 1 < T) {
                    if constexpr (tt > 0)
                        seq([&](auto pc) {
                            conv_a(std::integral_constant<int, tt + 1>{},
                                   std::integral_constant<int, lo + decltype(pc)::value>{});
                        }, WS_SEQ(hi - lo, p));
                    else if constexpr (b == NB - 1)
                        seq([&](auto pc) { conv_a(std::integral_constant<int, 1>{}, pc); }, WS_SEQ(4, p));
                }
                if constexpr (j < 3 && i >= kHalf && nb_reads(tt - kHalf) > 0)
                    seq([&](auto qc) {
                        seq([&](auto pc) {
                            conv_b(std::integral_constant<int, j + 1>{},
                                   std::integral_constant<int, (i - kHalf) * kRB + decltype(qc)::value>{},
                                   std::integral_constant<int, lo + decltype(pc)::value>{});
                        }, WS_SEQ(hi - lo, p));
                    }, WS_SEQ(nb_reads(tt - kHalf), q));
                pin();
            }, WS_SEQ(NB, b));
            if constexpr (tt == 0) next_b();
        }, WS_SEQ(T, t));
        if constexpr (SMODE == kF32s) {
            // acc += product * (A scale * weight scale), one rounding each
#pragma unroll
            for (int i = 0; i < MF; i++) {
                const float f = fs[i] * fs[MF];
#pragma unroll
                for (int b = 0; b < NB; b++)
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        acc[i][b][v] = __builtin_fmaf(prod[i][b][v], f, acc[i][b][v]);
            }
        }
        lds_wait_all();
        seq([&](auto qc) { conv_scale(qc); }, WS_SEQ(MF + kWS, q));
    }

    wait_vm<0>();  // the repeated loads still write this workgroup's LDS

    // ---- store: columns 4g .. 4g + 3 of a band, row r of a strip
#pragma unroll
    for (int i = 0; i < MF; i++) {
        const int row = m0 + wm * 16 * MF + 16 * i + r;
        if (row >= M) continue;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int col = n0 + wn * 16 * NB + 16 * b + 4 * g;
            if (col >= N) continue;
            const size_t o = (size_t)row * N + col;
            const v4f v = acc[i][b];
            const uint32_t lo = f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
            const uint32_t hi = f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
            *(uint2 *)(p.C + o) = uint2{lo, hi};
        }
    }
}

template <int MF, int NB, int WM, int WN, int NS, int SMODE>
static int launch(const Args &a0, hipStream_t stream) {
    using G = Geom<MF, NB, WM, WN, NS, SMODE>;
    Args a = a0;
    a.ntm = (a.M + G::BM - 1) / G::BM;
    a.ntn = (a.N + G::BN - 1) / G::BN;
    hipLaunchKernelGGL((gemm_tile_kernel<MF, NB, WM, WN, NS, SMODE>),
                       dim3((unsigned)a.ntm * (unsigned)a.ntn), dim3(G::kThreads), G::kLds, stream, a);
    return launch_status();
}

enum Cfg { k256x256, k128x256, k128x128, k64x128 };

// The configuration that finishes first. Cost of one 128-K step of a round of
// workgroups, in units of 10 ns, measured at K = 1280-15360:
// 256 x 256 tiles (8 waves, one workgroup per CU) 3.08 us, 128 x 256 (8 waves)
// 1.75; 128 x 128 (4 waves) 1.13 with one workgroup per CU and 1.77 with two,
// 64 x 128 0.85 and 1.17. M = N = 4096, K = 8192: 197 / 227 / 227 / 301 us
// (1.4 PFLOP/s for the first; the split-K pipeline and its reduction 372);
// M = 4096, N = 4608, K = 5120 (a nearly empty last round of the large tiles):
// 232 / 206 / 181 / 207; M = 200, N = 8192, K = 1280: 34 / 23 / 16 / 13.
static Cfg pick_cfg(int64_t M, int64_t N, int64_t cus, bool big) {
    auto tiles = [&](int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    // rounds of `per` workgroups per CU; the last one costs less when it
    // leaves every CU at most one
    auto rounds = [&](int64_t T, int per, int full, int one) {
        const int64_t rem = T % (cus * per);
        return T / (cus * per) * full + (rem == 0 ? 0 : rem <= cus ? one : full);
    };
    const int64_t c[4] = {big ? rounds(tiles(256, 256), 1, 308, 308) : INT64_MAX,
                          rounds(tiles(128, 256), 1, 175, 175), rounds(tiles(128, 128), 2, 177, 113),
                          rounds(tiles(64, 128), 2, 117, 85)};
    int best = 0;
    for (int i = 1; i < 4; i++)
        if (c[i] < c[best]) best = i;
    return (Cfg)best;
}

template <int SMODE>
static int run(const Args &a, hipStream_t stream) {
    // the 256 x 256 tile's wave has no registers left for a step's product
    // beside the sum (f32 scales)
    constexpr bool big = SMODE != kF32s;
    switch (pick_cfg(a.M, a.N, cu_count(), big)) {
        case k256x256:
            if constexpr (big) return launch<8, 4, 2, 4, 2, SMODE>(a, stream);
            return -1;
        case k128x256: return launch<4, 4, 2, 4, 3, SMODE>(a, stream);
        case k128x128: return launch<4, 4, 2, 2, 2, SMODE>(a, stream);
        case k64x128: return launch<4, 2, 1, 4, 3, SMODE>(a, stream);
    }
    return -1;
}

}  // namespace tile

int tile_gemm_bf16(int smode, const uint8_t *a, const void *sa, const uint8_t *b, const void *sb,
                   void *out, int64_t m, int64_t n, int64_t k, hipStream_t stream) {
    using namespace tile;
    if (m * k >= (1ll << 32) || n * k >= (1ll << 32)) return -1;  // 32-bit row offsets
    if ((uintptr_t)out & 7) return -1;
    const Args p{a, b, (const uint8_t *)sa, (const uint8_t *)sb, (uint16_t *)out, (int)m, (int)n,
                 (int)k, 0, 0};
    return smode == kF32s ? run<kF32s>(p, stream) : run<kUe8m0>(p, stream);
}

}  // namespace ws
