"""GPU parity: activation/weight quantisation and the block-scaled GEMMs,
called through the C ABI (weightstream_amd.launch) and checked against the
C oracle on the same seeded inputs.

Tolerances: quantisation is integer/byte work and must be bit-exact. GEMM
outputs are f32 sums of exact fp8 x fp8 (or fp8 x fp4) products; the MFMA
accumulation order differs from the oracle's sequential per-32-block order,
so outputs are compared with max relative error <= 1e-3 (floor at 1% of the
output scale, see gpu_util.rel_err_stats); observed errors are ~1e-6.
"""
import numpy as np
import pytest
import torch

import oracle_lib as O
from gpu_util import DEV, activations, announce, assert_close, dev, host
from weightstream_amd import launch as L

pytestmark = pytest.mark.gpu

GEMM_TOL = 1e-3


@pytest.fixture(scope="module", autouse=True)
def _init():
    L.Hip.global_()


@pytest.fixture(params=["single_pass", "split_k"])
def gemm_path(request):
    """Run a GEMM test with no split-K workspace (single-pass kernels) and
    with one (M > 64, and M <= 16 when the column strips leave CUs idle,
    split K across workgroups)."""
    ws = None
    if request.param == "split_k":
        ws = torch.empty(64 << 20, dtype=torch.uint8, device=DEV)
        L.set_gemm_workspace(ws)
    yield request.param
    if ws is not None:
        torch.cuda.synchronize()
        L.set_gemm_workspace(None)


def _wide_range_acts(rng, n):
    x = rng.standard_normal(n).astype(np.float32)
    x *= np.repeat(10.0 ** rng.uniform(-7, 4, n // 32), 32).astype(np.float32)
    x[:32] = 0.0                                   # zero block -> amax floor
    x[32:64] = np.float32(15.2 / 1024) * np.sign(rng.standard_normal(32))  # carry quirk
    x[32] = 448.0                                  # scale 1: the rest sit in [15/1024, 2^-6)
    x[70] = np.float32(np.nan)
    x[100] = np.float32(1e30)
    return x


def test_emit8_and_snap8_bit_exact():
    rng = np.random.default_rng(100)
    n = 32 * 4096
    x = _wide_range_acts(rng, n)
    q_ref, s_ref = O.fp8_act_emit(x)
    announce("emit8 n=%d" % n)
    dx = dev(x)
    q = torch.empty(n, dtype=torch.uint8, device=DEV)
    s = torch.empty(n // 32, dtype=torch.uint8, device=DEV)
    L.emit8(dx, q, s, n)
    assert np.array_equal(host(q), q_ref)
    assert np.array_equal(host(s), s_ref)
    announce("snap8 n=%d" % n)
    L.snap8(dx, n)
    got = host(dx)
    want = O.fp8_snap(x)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


def test_emit8_packed_and_pack_scales():
    rng = np.random.default_rng(101)
    n = 32 * 100
    x = rng.standard_normal(n).astype(np.float32)
    q_ref, s_ref = O.fp8_act_emit(x)
    raw = n // 32
    off = (raw + 15) // 16 * 16
    announce("emit8_packed n=%d" % n)
    q = torch.empty(n, dtype=torch.uint8, device=DEV)
    s = torch.zeros(off + raw, dtype=torch.uint8, device=DEV)
    L.emit8_packed(dev(x), q, s, n)
    sh = host(s)
    assert np.array_equal(host(q), q_ref)
    assert np.array_equal(sh[:raw], s_ref) and np.array_equal(sh[off:off + raw], s_ref)
    n2 = 128 * 7
    src = rng.integers(0, 256, n2 // 32).astype(np.uint8)
    dst = torch.empty(n2 // 128, dtype=torch.int32, device=DEV)
    L.pack_scales(dev(src), dst, n2)
    assert np.array_equal(host(dst).view(np.uint32), src.view("<u4"))


def test_weight_quant_bit_exact():
    rng = np.random.default_rng(102)
    rows, cols = 200, 512
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    w[3, 5] = 7.0
    w[40:72, 64:96] = 0.0
    announce("weight_quant fp4/fp8 %dx%d" % (rows, cols))
    q4 = torch.empty((rows, cols // 2), dtype=torch.uint8, device=DEV)
    s4 = torch.empty((rows, cols // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp4(dev(w), q4, s4, rows, cols)
    q4r, s4r = O.weight_quant_fp4(w)
    assert np.array_equal(host(q4), q4r) and np.array_equal(host(s4), s4r)
    q8 = torch.empty((rows, cols), dtype=torch.uint8, device=DEV)
    s8 = torch.empty(((rows + 31) // 32, cols // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp8(dev(w), q8, s8, rows, cols)
    q8r, s8r = O.weight_quant_fp8(w)
    assert np.array_equal(host(q8), q8r) and np.array_equal(host(s8), s8r)


@pytest.mark.parametrize("n,skew", [(32, 0), (1024, 0), (2048 + 32, 0), (3 * 2048 - 32, 0),
                                    (32, 1), (2048 + 96, 1),
                                    (384 * 1024 - 32, 0), (384 * 1024, 0), (458752 - 128, 0),
                                    (458752, 0), (768 * 1024 - 32, 0), (768 * 1024, 0),
                                    (768 * 1024 + 2048 + 128, 0), (768 * 1024 + 3 * 2048 - 32, 0),
                                    (768 * 1024 + 128, 1)])
def test_act_quant_edges_and_unaligned(n, skew):
    """The four-values-per-lane kernels at the edges of their 2048-value
    workgroups, and the one- and two-value kernels that fewer values (384 K for
    bytes, 768 K in place, 448 K with f32 scales) and unaligned operands (skew
    floats and bytes off) take: bit-exact."""
    rng = np.random.default_rng(103 + n)
    x = _wide_range_acts(rng, max(n, 128))[:n].copy()
    q_ref, s_ref = O.fp8_act_emit(x)
    raw, off = n // 32, (n // 32 + 15) // 16 * 16
    announce("act quant n=%d skew=%d" % (n, skew))
    dx = torch.empty(n + skew, device=DEV)[skew:]
    dx.copy_(dev(x))
    q = torch.full((n + skew + 4,), 0xA5, dtype=torch.uint8, device=DEV)
    s = torch.zeros(off + raw, dtype=torch.uint8, device=DEV)
    L.emit8_packed(dx, q[skew:], s, n)
    sh, qh = host(s), host(q)
    assert np.array_equal(qh[skew:skew + n], q_ref) and (qh[skew + n:] == 0xA5).all()
    assert np.array_equal(sh[:raw], s_ref) and np.array_equal(sh[off:], s_ref)
    L.snap8(dx, n)
    got, want = host(dx), O.fp8_snap(x)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
    if n % 128 == 0:
        m, k = 1, n
        y = rng.standard_normal((m, k)).astype(np.float32)
        dx.copy_(dev(y.ravel()))
        aq_ref, as_ref = O.act_quant_f32s(y, 128)
        sf = torch.empty(k // 128, device=DEV)
        L.act_quant_f32s(dx, q[skew:], sf, m, k)
        assert np.array_equal(host(q)[skew:skew + n], aq_ref.ravel())
        assert np.array_equal(host(sf).view(np.uint32), as_ref.view(np.uint32).ravel())


@pytest.mark.parametrize("rows,cols,skew", [(1, 32, 0), (33, 160, 0), (31, 96, 0), (64, 384, 0),
                                            (33, 160, 1),
                                            (255, 1056, 0), (256, 1056, 0), (1023, 1024, 0),
                                            (1025, 1056, 0), (1025, 1056, 1)])
def test_weight_quant_edges_and_unaligned(rows, cols, skew):
    """The vectorised weight encoders (from 256 K values in FP4, 1 M in FP8) at
    ragged rows and columns, with FP4 values on and beside every rounding
    threshold, and the kernels for fewer values and unaligned operands:
    bit-exact."""
    rng = np.random.default_rng(104 + rows + cols)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    edges = np.array([0.25, 0.75, 1.0, 1.25, 1.75, 2.5, 3.5, 5.0, 6.0], np.float32)
    edges = np.concatenate([edges, np.nextafter(edges, np.float32(0)),
                            np.nextafter(edges[:-1], np.float32(9)), [0.0, -0.0, 1e-40]])
    edges = np.concatenate([edges, edges[:3]]).astype(np.float32)   # largest 6: scale 1
    w[0, :32] = np.where(rng.random(32) < 0.5, -edges, edges)
    w[rows - 1, cols - 32:] = np.float32(1e30) if rows > 1 else w[rows - 1, cols - 32:]
    announce("weight_quant edges %dx%d skew=%d" % (rows, cols, skew))
    dw = torch.empty(rows * cols + skew, device=DEV)[skew:]
    dw.copy_(dev(w.ravel()))
    q4 = torch.empty(rows * cols // 2 + skew, dtype=torch.uint8, device=DEV)[skew:]
    s4 = torch.empty(rows * cols // 32, dtype=torch.uint8, device=DEV)
    L.weight_quant_fp4(dw, q4, s4, rows, cols)
    q4r, s4r = O.weight_quant_fp4(w)
    assert np.array_equal(host(q4), q4r.ravel()) and np.array_equal(host(s4), s4r.ravel())
    q8 = torch.empty(rows * cols + skew, dtype=torch.uint8, device=DEV)[skew:]
    s8 = torch.empty((rows + 31) // 32 * (cols // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp8(dw, q8, s8, rows, cols)
    q8r, s8r = O.weight_quant_fp8(w)
    assert np.array_equal(host(q8), q8r.ravel()) and np.array_equal(host(s8), s8r.ravel())


def test_weight_quant_nonfinite_same_on_both_kernels():
    """Blocks with infinities, NaN, nothing else, and FLT_MAX: the vectorised
    encoders give the bytes of the general ones (which unaligned operands
    take)."""
    rows, cols = 1024, 1056
    rng = np.random.default_rng(105)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    big = np.finfo(np.float32).max
    w[0, 5], w[40, 70], w[41, 71], w[100, 1040] = np.inf, -np.inf, np.nan, np.nan
    w[200, 64:96] = np.inf
    w[224:256, 96:128] = np.nan
    w[300, 128:160] = np.nan
    w[400, 1000], w[401, 1001], w[500, 32:64] = big, -big, big
    w[600, 0:32] = 1e-42
    announce("weight_quant nonfinite %dx%d on both kernels" % (rows, cols))
    out = []
    for skew in (0, 1):
        dw = torch.empty(rows * cols + skew, device=DEV)[skew:]
        dw.copy_(dev(w.ravel()))
        q4 = torch.empty(rows * cols // 2, dtype=torch.uint8, device=DEV)
        q8 = torch.empty(rows * cols, dtype=torch.uint8, device=DEV)
        s4 = torch.empty(rows * cols // 32, dtype=torch.uint8, device=DEV)
        s8 = torch.empty(rows // 32 * (cols // 32), dtype=torch.uint8, device=DEV)
        L.weight_quant_fp4(dw, q4, s4, rows, cols)
        L.weight_quant_fp8(dw, q8, s8, rows, cols)
        out.append([host(t) for t in (q4, s4, q8, s8)])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("rows,cols", [(16, 128), (48, 1024), (2064, 1024), (32, 1152),
                                       (2048, 2048), (2064, 2048), (272, 5120), (16, 2944)])
def test_prepack_layout(rows, cols):
    """The packed layout's definition, in numpy, for the relayout by chunks
    (whole 8-step scale groups, small or one group long) and by waves; padding
    scale bytes are 127."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(rows + cols)
    announce("prepack %dx%d" % (rows, cols))
    w = torch.randint(0, 256, (rows, cols // 2), dtype=torch.uint8, device=DEV, generator=gen)
    s = torch.randint(0, 256, (rows, cols // 32), dtype=torch.uint8, device=DEV, generator=gen)
    for skew in (0, 1):
        pw = torch.full((rows * cols // 2 + 16,), 0xA5, dtype=torch.uint8, device=DEV)
        n = L.packed_fp4_scale_bytes(rows, cols)
        ps = torch.full((n + skew + 16,), 0xA5, dtype=torch.uint8, device=DEV)
        L.prepack_fp4(w, s, rows, cols, pw, ps[skew:])
        ksn = cols // 128
        # [band][step][16 g + r][16 bytes]: row 16 band + r, chunk 4 step + g
        want = host(w).reshape(rows // 16, 16, ksn, 4, 16).transpose(0, 2, 3, 1, 4)
        sc = np.full((rows // 16, (ksn + 7) // 8 * 8, 4, 16), 127, np.uint8)
        sc[:, :ksn] = host(s).reshape(rows // 16, 16, ksn, 4).transpose(0, 2, 3, 1)
        # [band][group][16 g + r][step of the group]
        sc = sc.reshape(rows // 16, -1, 8, 64).transpose(0, 1, 3, 2)
        got, gs = host(pw), host(ps)[skew:]
        assert np.array_equal(got[:-16], want.ravel()) and (got[-16:] == 0xA5).all()
        assert np.array_equal(gs[:n], sc.ravel()) and (gs[n:] == 0xA5).all()


def _quantised_case(rng, m, n, k, fp4):
    x = activations(rng, m, k)
    aq, as_ = O.fp8_act_emit(x)
    wf = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    wq, ws = O.weight_quant_fp4(wf) if fp4 else O.weight_quant_fp8(wf)
    return aq, as_, wq, ws


GEMM_SHAPES = [(1, 4096, 4096), (1, 1024, 2048), (4, 256, 512), (16, 512, 1024),
               (17, 96, 384), (64, 256, 1024), (128, 512, 4096), (130, 48, 256),
               (300, 160, 640), (65, 1024, 4096)]


@pytest.mark.parametrize("m,n,k", GEMM_SHAPES)
def test_fp8_gemm_matches_oracle(m, n, k, gemm_path):
    rng = np.random.default_rng(1000 + m + n + k)
    aq, as_, wq, ws = _quantised_case(rng, m, n, k, False)
    want = O.gemm_q(aq, as_, m, wq, ws, n, k, False)
    announce("fp8_gemm %s m=%d n=%d k=%d" % (gemm_path, m, n, k))
    out = torch.empty((m, n), dtype=torch.float32, device=DEV)
    L.fp8_gemm(dev(aq), dev(as_), dev(wq), dev(ws), out, m, n, k)
    assert_close(host(out), want, GEMM_TOL, "fp8_gemm %dx%dx%d" % (m, n, k))
    announce("fp8_gemm_bf16 m=%d n=%d k=%d" % (m, n, k))
    ob = torch.empty((m, n), dtype=torch.int16, device=DEV)
    L.fp8_gemm_bf16(dev(aq), dev(as_), dev(wq), dev(ws), ob, m, n, k)
    got = (host(ob).astype(np.uint16).astype(np.uint32) << 16).view(np.float32)
    # bf16 keeps 8 significant bits: RNE error <= 2^-8 relative; and the
    # output equals the oracle's f32 rounded to bf16 except where the two f32
    # values straddle a rounding boundary
    assert_close(got, want, 2.0 ** -8 + GEMM_TOL, "fp8_gemm_bf16 %dx%dx%d" % (m, n, k))
    want_b = np.array([O.f32_to_bf16(float(v)) for v in want.ravel()], np.uint16)
    same = np.mean(host(ob).astype(np.uint16).ravel() == want_b)
    assert same >= 0.999, same


@pytest.mark.parametrize("m", [1, 8, 64])
def test_fp8_gemm_out_projection_shape_matches_oracle(m, gemm_path):
    """The config-5 attention out-projection shape, N=4096, K=8192, at the
    block's M in {1, 8, 64}: f32 and bf16 outputs against the oracle's
    dequantise-then-f32 GEMM (or_gemm_q) on sampled rows."""
    n, k = 4096, 8192
    rng = np.random.default_rng(1500 + m)
    aq, as_, wq, ws = _quantised_case(rng, m, n, k, False)
    rows = sorted({0, m // 2, m - 1})
    want = O.gemm_q(np.ascontiguousarray(aq[rows]), np.ascontiguousarray(as_[rows]), len(rows),
                    wq, ws, n, k, False)
    announce("fp8_gemm out-projection %s m=%d" % (gemm_path, m))
    out = torch.empty((m, n), dtype=torch.float32, device=DEV)
    L.fp8_gemm(dev(aq), dev(as_), dev(wq), dev(ws), out, m, n, k)
    assert_close(host(out)[rows], want, GEMM_TOL, "fp8_gemm %dx%dx%d" % (m, n, k))
    ob = torch.empty((m, n), dtype=torch.int16, device=DEV)
    L.fp8_gemm_bf16(dev(aq), dev(as_), dev(wq), dev(ws), ob, m, n, k)
    got = (host(ob).astype(np.uint16).astype(np.uint32) << 16).view(np.float32)
    assert_close(got[rows], want, 2.0 ** -8 + GEMM_TOL, "fp8_gemm_bf16 %dx%dx%d" % (m, n, k))


@pytest.mark.parametrize("m,n,k", [(1, 2048, 4096), (8, 512, 1024), (128, 256, 2048),
                                   (33, 80, 512), (200, 192, 1024), (130, 8192, 256)])
def test_fp4_gemm_matches_oracle(m, n, k, gemm_path):
    rng = np.random.default_rng(2000 + m + n + k)
    aq, as_, wq, ws = _quantised_case(rng, m, n, k, True)
    want = O.gemm_q(aq, as_, m, wq, ws, n, k, True)
    announce("fp4_gemm %s m=%d n=%d k=%d" % (gemm_path, m, n, k))
    out = torch.empty((m, n), dtype=torch.float32, device=DEV)
    L.fp4_gemm(dev(aq), dev(as_), dev(wq), dev(ws), out, m, n, k)
    assert_close(host(out), want, GEMM_TOL, "fp4_gemm %dx%dx%d" % (m, n, k))


@pytest.mark.parametrize("m,n,k", [(1, 4096, 4096), (128, 384, 4096), (20, 256, 512),
                                   (5, 64, 1152), (257, 320, 1280), (128, 8192, 512)])  # K/128 = 9: the general kernel
def test_fp8_gemm_f32s_matches_oracle(m, n, k, gemm_path):
    rng = np.random.default_rng(3000 + m + n + k)
    x = activations(rng, m, k)
    wf = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    wq, ws = O.weight_quant_fp8_f32s(wf, 128)
    aq_ref, as_ref = O.act_quant_f32s(x, 128)
    want = O.gemm_f32s(aq_ref, as_ref, wq, ws, 128)
    announce("act_quant_f32s + fp8_gemm_f32s m=%d n=%d k=%d" % (m, n, k))
    aq = torch.empty((m, k), dtype=torch.uint8, device=DEV)
    as_ = torch.empty((m, k // 128), dtype=torch.float32, device=DEV)
    L.act_quant_f32s(dev(x), aq, as_, m, k)
    assert np.array_equal(host(aq), aq_ref)
    assert np.array_equal(host(as_).view(np.uint32), as_ref.view(np.uint32))
    out = torch.empty((m, n), dtype=torch.float32, device=DEV)
    L.fp8_gemm_f32s(aq, as_, dev(wq), dev(ws), out, m, n, k)
    assert_close(host(out), want, GEMM_TOL, "fp8_gemm_f32s %dx%dx%d" % (m, n, k))


@pytest.mark.parametrize("n", [4096, 12288, 2048])
def test_config2_fp8_gemm_f32s_full_size_matches_oracle(n, gemm_path):
    """BASELINE config 2 in its own scale scheme at full size: M=128, K=4096,
    N in {4096, 12288, 2048}; weights N(0, 0.02) quantised with 128x128 f32
    scales amax/448 (or_weight_quant_fp8_f32s), activations N(0, 1) with 1%
    outliers x20 quantised per 1x128 on the device (bit-exact with the
    oracle); f32 and bf16 outputs against the oracle's sequential
    dequantise-then-f32-accumulate GEMM (or_gemm_f32s) on every row. Runs
    with and without the split-K workspace (the line kernel takes all three
    N: 128 x 48 tiles at N = 12288, 64 x 32 at N = 4096, 32 x 32 at
    N = 2048; the split-K pipeline is covered by the model shapes below)."""
    m, k = 128, 4096
    rng = np.random.default_rng(3100 + n)
    x = activations(rng, m, k)
    wf = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    wq, ws = O.weight_quant_fp8_f32s(wf, 128)
    del wf
    aq_ref, as_ref = O.act_quant_f32s(x, 128)
    O.set_threads(16)
    try:
        want = O.gemm_f32s(aq_ref, as_ref, wq, ws, 128)
    finally:
        O.set_threads(1)
    announce("config 2 act_quant_f32s + fp8_gemm_f32s %s m=%d n=%d k=%d" % (gemm_path, m, n, k))
    aq = torch.empty((m, k), dtype=torch.uint8, device=DEV)
    as_ = torch.empty((m, k // 128), dtype=torch.float32, device=DEV)
    L.act_quant_f32s(dev(x), aq, as_, m, k)
    assert np.array_equal(host(aq), aq_ref)
    assert np.array_equal(host(as_).view(np.uint32), as_ref.view(np.uint32))
    dwq, dws = dev(wq), dev(ws)
    out = torch.empty((m, n), dtype=torch.float32, device=DEV)
    L.fp8_gemm_f32s(aq, as_, dwq, dws, out, m, n, k)
    assert_close(host(out), want, GEMM_TOL, "config 2 f32s %dx%dx%d f32 out" % (m, n, k))
    ob = torch.empty((m, n), dtype=torch.int16, device=DEV)
    L.fp8_gemm_f32s(aq, as_, dwq, dws, ob, m, n, k, out_bf16=True)
    bits = host(ob).astype(np.uint16)
    got = (bits.astype(np.uint32) << 16).view(np.float32)
    assert_close(got, want, 2.0 ** -8 + GEMM_TOL, "config 2 f32s %dx%dx%d bf16 out" % (m, n, k))
    # bf16 out is the f32 result rounded to nearest even (quant.rs:95-101):
    # equal to the oracle's f32 rounded to bf16 except at rounding boundaries
    wb = want.view(np.uint32)
    want_b = ((wb + (((wb >> 16) & 1) + 0x7FFF)) >> 16).astype(np.uint16)
    same = np.mean(bits == want_b)
    print("[config 2 bf16 n=%d] %.5f of outputs equal bf16(oracle)" % (n, same), flush=True)
    assert same >= 0.999, same


@pytest.mark.parametrize("n", [4096, 12288, 2048])
def test_fp8_gemm_full_size_vs_fp64_dequant(n, gemm_path):
    """BASELINE config 2 shapes (M=128, K=4096) against an f64 matmul of the
    dequantised operands on the device (too large for the scalar oracle)."""
    m, k = 128, 4096
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n)
    announce("fp8_gemm full %s m=%d n=%d k=%d" % (gemm_path, m, n, k))
    x = torch.randn((m, k), device=DEV, generator=gen)
    x = torch.where(torch.rand((m, k), device=DEV, generator=gen) < 0.01, x * 20, x)
    w = torch.randn((n, k), device=DEV, generator=gen) * 0.02
    aq = torch.empty((m, k), dtype=torch.uint8, device=DEV)
    as_ = torch.empty((m, k // 32), dtype=torch.uint8, device=DEV)
    L.emit8(x, aq, as_, m * k)
    wq = torch.empty((n, k), dtype=torch.uint8, device=DEV)
    ws = torch.empty((n // 32, k // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp8(w, wq, ws, n, k)
    out = torch.empty((m, n), dtype=torch.float32, device=DEV)
    L.fp8_gemm(aq, as_, wq, ws, out, m, n, k)
    table = torch.from_numpy(O.e4m3_decode_table().astype(np.float64)).to(DEV)
    pw = lambda s: torch.pow(2.0, s.to(torch.float64) - 127)
    da = table[aq.long()] * pw(as_).repeat_interleave(32, 1)
    dw = table[wq.long()] * pw(ws).repeat_interleave(32, 0).repeat_interleave(32, 1)
    want = (da @ dw.T).cpu().numpy()
    assert_close(host(out), want, GEMM_TOL, "fp8_gemm full %dx%dx%d" % (m, n, k))


# The engine's FP8 projection shapes (N, K) (weightstream-gpu engine.rs:3388-3398:
# q_a, q_b, wkv, wo_b, shared w1/w3, fused w13, shared w2, engram wkv, drafter).
MODEL_SHAPES = [(1280, 5120), (8192, 1280), (512, 5120), (5120, 2048), (2304, 5120),
                (4608, 5120), (5120, 2304), (25600, 5120), (1280, 15360)]


@pytest.mark.parametrize("n,k", MODEL_SHAPES)
@pytest.mark.parametrize("m", [1, 6, 128])
def test_fp8_gemm_model_shapes_vs_fp64_dequant(m, n, k, gemm_path):
    """The real projection shapes through the dispatch (every kernel family
    and the fallbacks for K/128 not a multiple of 4), against an f64 matmul of
    the dequantised operands on the device."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(m * 7 + n + k)
    announce("fp8_gemm model shape %s m=%d n=%d k=%d" % (gemm_path, m, n, k))
    x = torch.randn((m, k), device=DEV, generator=gen)
    w = torch.randn((n, k), device=DEV, generator=gen) * 0.02
    aq = torch.empty((m, k), dtype=torch.uint8, device=DEV)
    as_ = torch.empty((m, k // 32), dtype=torch.uint8, device=DEV)
    L.emit8(x, aq, as_, m * k)
    wq = torch.empty((n, k), dtype=torch.uint8, device=DEV)
    ws = torch.empty(((n + 31) // 32, k // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp8(w, wq, ws, n, k)
    out = torch.empty((m, n), dtype=torch.float32, device=DEV)
    L.fp8_gemm(aq, as_, wq, ws, out, m, n, k)
    table = torch.from_numpy(O.e4m3_decode_table().astype(np.float64)).to(DEV)
    pw = lambda s: torch.pow(2.0, s.to(torch.float64) - 127)
    da = table[aq.long()] * pw(as_).repeat_interleave(32, 1)
    dw = table[wq.long()] * pw(ws).repeat_interleave(32, 0)[:n].repeat_interleave(32, 1)
    want = (da @ dw.T).cpu().numpy()
    assert_close(host(out), want, GEMM_TOL, "fp8_gemm %dx%dx%d" % (m, n, k))


def test_gemm_rejects_bad_shapes():
    a = torch.zeros(256, dtype=torch.uint8, device=DEV)
    out = torch.zeros(256, dtype=torch.float32, device=DEV)
    with pytest.raises(RuntimeError, match="unsupported shape"):
        L.fp8_gemm(a, a, a, a, out, 1, 16, 100)     # K % 128 != 0
    with pytest.raises(RuntimeError, match="unsupported shape"):
        L.fp8_gemm(a, a, a, a, out, 1, 10, 128)     # N % 16 != 0


def test_split_k_is_deterministic_and_reusable():
    """Split-K tickets reset themselves: repeated calls (and a different shape
    in between) give bit-identical results."""
    rng = np.random.default_rng(4000)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=DEV)
    L.set_gemm_workspace(ws)
    try:
        outs = []
        for m, n, k in [(128, 512, 4096), (40, 192, 2048), (128, 512, 4096), (128, 512, 4096)]:
            aq, as_, wq, ws_ = _quantised_case(np.random.default_rng(4000 + m + n), m, n, k, False)
            announce("split-k repeat m=%d n=%d k=%d" % (m, n, k))
            out = torch.empty((m, n), dtype=torch.float32, device=DEV)
            L.fp8_gemm(dev(aq), dev(as_), dev(wq), dev(ws_), out, m, n, k)
            outs.append(host(out))
        assert np.array_equal(outs[0].view(np.uint32), outs[2].view(np.uint32))
        assert np.array_equal(outs[0].view(np.uint32), outs[3].view(np.uint32))
    finally:
        torch.cuda.synchronize()
        L.set_gemm_workspace(None)
    del rng


@pytest.mark.parametrize("m,n,k", [(1, 1280, 15360), (6, 512, 12288)])
def test_long_k_strip_split_matches_single_pass(m, n, k):
    """M <= 16 with few column strips and K > 8192 splits K over workgroups
    when a workspace is set: the same sums up to f32 reassociation (within
    the GEMM tolerance of the single-pass result), and repeated calls give
    the same bits."""
    aq, as_, wq, ws_ = _quantised_case(np.random.default_rng(4100 + m + n), m, n, k, False)
    announce("strip split m=%d n=%d k=%d" % (m, n, k))
    args = [dev(aq), dev(as_), dev(wq), dev(ws_)]
    single = torch.empty((m, n), dtype=torch.float32, device=DEV)
    L.fp8_gemm(*args, single, m, n, k)
    ws = torch.empty(max(L.gemm_workspace_size(m, n, k), 256), dtype=torch.uint8, device=DEV)
    L.set_gemm_workspace(ws)
    try:
        outs = []
        for _ in range(2):
            out = torch.empty((m, n), dtype=torch.float32, device=DEV)
            L.fp8_gemm(*args, out, m, n, k)
            outs.append(host(out))
    finally:
        torch.cuda.synchronize()
        L.set_gemm_workspace(None)
    assert L.gemm_workspace_size(m, n, k) > 0
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert_close(outs[0], host(single), GEMM_TOL, "strip split m=%d n=%d k=%d" % (m, n, k))


def test_workspace_registered_under_one_mode_serves_both():
    """set_gemm_workspace registers with both library builds: a NATIVE-mode
    GEMM on a stream whose workspace was set while EXACT was active takes the
    split-K path (it writes partials into the workspace) and gives the bits
    of the same NATIVE GEMM registered under NATIVE."""
    m, n, k = 128, 8192, 2304     # the split-K pipeline's shape (K not a multiple of 512)
    gen = torch.Generator(device=DEV).manual_seed(77)
    x = torch.randn((m, k), device=DEV, generator=gen)
    aq = torch.empty((m, k), dtype=torch.uint8, device=DEV)
    asc = torch.empty((m, k // 32), dtype=torch.uint8, device=DEV)
    L.emit8(x, aq, asc, m * k)
    wf = torch.randn((n, k), device=DEV, generator=gen) * 0.02
    w = torch.empty((n, k), dtype=torch.uint8, device=DEV)
    sw = torch.empty((n // 32, k // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp8(wf, w, sw, n, k)
    ws = torch.full((L.gemm_workspace_size(m, n, k),), 0xAB, dtype=torch.uint8, device=DEV)
    outs = []
    try:
        for reg_mode in (L.MATH_EXACT, L.MATH_NATIVE):
            L.set_math_mode(reg_mode)
            L.set_gemm_workspace(ws)
            ws.fill_(0xAB)
            L.set_math_mode(L.MATH_NATIVE)
            announce("native fp8_gemm after a workspace set in mode %d" % reg_mode)
            out = torch.empty((m, n), dtype=torch.float32, device=DEV)
            L.fp8_gemm(aq, asc, w, sw, out, m, n, k)
            torch.cuda.synchronize()
            assert (ws != 0xAB).any(), "the split-K path did not run"
            outs.append(out)
            L.set_gemm_workspace(None)
    finally:
        L.set_math_mode(L.MATH_EXACT)
        torch.cuda.synchronize()
        L.set_gemm_workspace(None)
    assert torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))


@pytest.mark.parametrize("m,n,k", [(100, 4096, 4096), (65, 3072, 2048), (128, 5120, 1024),
                                   (127, 3104, 4096), (100, 2048, 4096), (40, 4096, 2048),
                                   (120, 12288, 4096), (128, 9216, 768),
                                   # K > 4096, N > 4096 or few tiles
                                   (64, 4096, 8192), (96, 5120, 5120), (24, 2048, 4096),
                                   (64, 12288, 4096), (128, 1280, 8192)])
@pytest.mark.parametrize("native", [False, True])
def test_line_gemm_ragged_rows_vs_fp64_dequant(m, n, k, native):
    """The line kernel (K a multiple of 512): 64 x 32 tiles for M in 65-128
    with 192-384 workgroups, 32 x 32 tiles for 32-row blocks (n = 2048 at
    M = 100; M = 40), 128 x 48 tiles for wide N (12288; 9216 at K = 768,
    three 256-K stages); ragged last row blocks, the XCD-paired tile order and
    (n = 3104: 194 workgroups) the plain order; the other shapes it stages
    (K > 4096, N > 4096, few tiles: 32 x 32 tiles when they fit one round of
    workgroups, else 64 x 32; at most 32 rows, 32 x 32 with 64 or more
    tiles), UE8M0 and f32 scales, f32
    and bf16 outputs, against an f64 matmul of the dequantised operands.
    EXACT within 1e-3; NATIVE within its own 5e-2 (tests/test_gpu_native.py)."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(m + n + k)
    tol = 5e-2 if native else GEMM_TOL
    announce("line gemm m=%d n=%d k=%d native=%d" % (m, n, k, native))
    x = torch.randn((m, k), device=DEV, generator=gen)
    x = torch.where(torch.rand((m, k), device=DEV, generator=gen) < 0.01, x * 20, x)
    w = torch.randn((n, k), device=DEV, generator=gen) * 0.02
    aq = torch.empty((m, k), dtype=torch.uint8, device=DEV)
    as_ = torch.empty((m, k // 32), dtype=torch.uint8, device=DEV)
    L.emit8(x, aq, as_, m * k)
    wq = torch.empty((n, k), dtype=torch.uint8, device=DEV)
    ws = torch.empty((n // 32, k // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp8(w, wq, ws, n, k)
    table = torch.from_numpy(O.e4m3_decode_table().astype(np.float64)).to(DEV)
    pw = lambda s: torch.pow(2.0, s.to(torch.float64) - 127)
    da = table[aq.long()] * pw(as_).repeat_interleave(32, 1)
    dw = table[wq.long()] * pw(ws).repeat_interleave(32, 0).repeat_interleave(32, 1)
    want = (da @ dw.T).cpu().numpy()
    # f32 scales: the same codes with per-block f32 scales (128 x 128 / 1 x 128)
    af = torch.rand((m, k // 128), device=DEV, generator=gen) * 0.01 + 1e-3
    wf = torch.rand((n // 128 + (n % 128 > 0), k // 128), device=DEV, generator=gen) * 1e-4 + 1e-5
    daf = table[aq.long()] * af.double().repeat_interleave(128, 1)
    dwf = table[wq.long()] * wf.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)
    want_f = (daf @ dwf.T).cpu().numpy()
    prev = L.set_math_mode(L.MATH_NATIVE if native else L.MATH_EXACT)
    try:
        out = torch.empty((m, n), dtype=torch.float32, device=DEV)
        L.fp8_gemm(aq, as_, wq, ws, out, m, n, k)
        assert_close(host(out), want, tol, "line gemm %dx%dx%d" % (m, n, k))
        ob = torch.empty((m, n), dtype=torch.int16, device=DEV)
        L.fp8_gemm_bf16(aq, as_, wq, ws, ob, m, n, k)
        got = (host(ob).astype(np.uint16).astype(np.uint32) << 16).view(np.float32)
        assert_close(got, want, 2.0 ** -8 + tol, "line gemm bf16 %dx%dx%d" % (m, n, k))
        outf = torch.empty((m, n), dtype=torch.float32, device=DEV)
        L.fp8_gemm_f32s(aq, af, wq, wf, outf, m, n, k)
        assert_close(host(outf), want_f, tol, "line gemm f32s %dx%dx%d" % (m, n, k))
    finally:
        L.set_math_mode(prev)


@pytest.mark.parametrize("m,n,k", [(129, 400, 128), (200, 528, 256), (777, 4608, 384),
                                   (2000, 4096, 512), (4090, 4080, 640), (65, 4096, 1152),
                                   (65, 4112, 1152), (775, 4592, 640)])
def test_tile_gemm_edges_vs_fp64_dequant(m, n, k):
    """The GEMMs above 64 rows with ragged rows, columns and step counts (1, 2, 3,
    4, 5 and 9 steps, so that scale groups of four end anywhere), every weight
    format and output. bf16 results take the whole-K tile kernel (but for 65 x
    4096, whose columns make one round of 32-column strips), by its rule in 64 x
    128 tiles (129, 200 and 65 rows), 128 x 128 (777, 775), 128 x 256 (2000; f32
    scales also 4090) and 256 x 256 (4090); f32 results, FP4 and the accumulating
    output take the pipeline or the strips.

    f32 sums of at most 36 MFMAs: each rounding is at most 2^-24 of a partial sum,
    so the 2-norm error stays under sqrt(36) 2^-24 = 3.6e-7. Per value, an MFMA,
    an f32-scale fma and the scales' product each err by at most 2^-23 of the sum
    of magnitudes, and bf16 adds 2^-8 of the value."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(m + n + k)
    announce("tile gemm m=%d n=%d k=%d" % (m, n, k))
    x = torch.randn((m, k), device=DEV, generator=gen)
    w = torch.randn((n, k), device=DEV, generator=gen) * 0.02
    aq = torch.empty((m, k), dtype=torch.uint8, device=DEV)
    as_ = torch.empty((m, k // 32), dtype=torch.uint8, device=DEV)
    L.emit8(x, aq, as_, m * k)
    wq = torch.empty((n, k), dtype=torch.uint8, device=DEV)
    ws = torch.empty(((n + 31) // 32, k // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp8(w, wq, ws, n, k)
    w4 = torch.empty((n, k // 2), dtype=torch.uint8, device=DEV)
    s4 = torch.empty((n, k // 32), dtype=torch.uint8, device=DEV)
    L.weight_quant_fp4(w, w4, s4, n, k)
    table = torch.from_numpy(O.e4m3_decode_table().astype(np.float64)).to(DEV)
    pw = lambda s: torch.pow(2.0, s.to(torch.float64) - 127)
    codes, da = table[aq.long()], None
    da = codes * pw(as_).repeat_interleave(32, 1)
    dw = table[wq.long()] * pw(ws).repeat_interleave(32, 0)[:n].repeat_interleave(32, 1)

    def run(call, dtype=torch.float32, start=None):
        buf = torch.full((m * n + 64,), -7.0, dtype=torch.float32, device=DEV).to(dtype)
        if start is not None:
            buf[:m * n] = start.view(-1)
        call(buf)
        torch.cuda.synchronize()
        assert (buf[m * n:] == -7).all(), "written past the output"
        return buf[:m * n].view(m, n)

    def close(got, want, what):
        err = float((got.double() - want).norm() / want.norm())
        print("[tile %s %dx%dx%d] rel 2-norm err %.3g" % (what, m, n, k, err))
        assert err <= 3.6e-7, (what, err)

    def close_bf16(got, want, mags, what):
        roundings = k // 32 + k // 128 + 2
        bound = 2.0 ** -8 * want.abs() + roundings * 2.0 ** -23 * mags
        over = ((got.double() - want).abs() / bound).max()
        print("[tile %s %dx%dx%d] %.3g of the bound" % (what, m, n, k, float(over)))
        assert over <= 1, (what, float(over))

    out = run(lambda o: L.fp8_gemm(aq, as_, wq, ws, o, m, n, k))
    close(out, da @ dw.T, "fp8")
    ob = run(lambda o: L.fp8_gemm_bf16(aq, as_, wq, ws, o, m, n, k), torch.bfloat16)
    close_bf16(ob, da @ dw.T, da.abs() @ dw.abs().T, "fp8 bf16")
    if m > 128:  # at most 128 rows ws_fp8_gemm may take the line kernel for both
        slack = 2 * 40 * 2.0 ** -23 * (da.abs() @ dw.abs().T)
        assert ((ob.double() - out.double()).abs() <= 2.0 ** -8 * out.double().abs() + 1.01 * slack).all()
        c0 = torch.randn((m, n), device=DEV, generator=gen)
        acc = run(lambda o: L.fp8_gemm_acc(aq, as_, wq, ws, o, m, n, k), start=c0)
        assert ((acc.double() - c0.double() - out.double()).abs()
                <= 1.01 * slack + 2.0 ** -23 * (c0 + out).double().abs()).all()
    af = torch.rand((m, k // 128), device=DEV, generator=gen) * 0.01 + 1e-3
    wf = torch.rand(((n + 127) // 128, k // 128), device=DEV, generator=gen) * 1e-4 + 1e-5
    fout = run(lambda o: L.fp8_gemm_f32s(aq, af, wq, wf, o, m, n, k))
    fa = codes * af.double().repeat_interleave(128, 1)
    fw = table[wq.long()] * wf.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)
    close(fout, fa @ fw.T, "f32s")
    fob = run(lambda o: L.fp8_gemm_f32s(aq, af, wq, wf, o, m, n, k, out_bf16=True), torch.bfloat16)
    close_bf16(fob, fa @ fw.T, fa.abs() @ fw.abs().T, "f32s bf16")
    lut = torch.tensor([O.fp4_value(i) for i in range(16)], dtype=torch.float64, device=DEV)
    d4 = torch.stack((lut[(w4 & 15).long()], lut[(w4 >> 4).long()]), -1).view(n, k)
    got = run(lambda o: L.fp4_gemm(aq, as_, w4, s4, o, m, n, k))
    close(got, da @ (d4 * pw(s4).repeat_interleave(32, 1)).T, "fp4")


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,n,k", [(130, 272, 768), (130, 272, 896),        # K <= 768 (896): any
                                   (1030, 4096, 256), (1030, 4112, 256),    # more tiles than CUs
                                   (380, 400, 1280), (300, 272, 1280),      # 12 and 9 tiles
                                   (200, 1552, 1536), (150, 1424, 1536),    # 26 and 24
                                   (200, 2448, 2048), (200, 2320, 2048),    # 40 and 38
                                   (390, 3984, 2304), (380, 3984, 2304),    # 128 and 96
                                   (300, 3600, 3200), (300, 5520, 3200),    # 87 and 132
                                   (600, 4624, 3328),                       # 185
                                   (380, 4112, 4096), (450, 3088, 4096),    # 99 and 100
                                   (600, 4880, 4224), (600, 4624, 4224)])   # 195 and 185
def test_bf16_gemm_each_side_of_the_tile_rule(m, n, k, split):
    """bf16 results on both sides of each line of the rule that takes them to the whole-K tiles
    (on the tiles, on the split-K pipeline and without a workspace on its
    single pass), UE8M0 and f32 scales, against f64; per value the bound of
    test_tile_gemm_edges_vs_fp64_dequant and one rounding for each of at most 8
    partial sums."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(m + n + k)
    announce("bf16 gemm m=%d n=%d k=%d split=%d" % (m, n, k, split))
    aq = torch.randint(0, 120, (m, k), dtype=torch.uint8, device=DEV, generator=gen)
    aq |= torch.randint(0, 2, (m, k), dtype=torch.uint8, device=DEV, generator=gen) << 7
    wq = torch.randint(0, 120, (n, k), dtype=torch.uint8, device=DEV, generator=gen)
    wq |= torch.randint(0, 2, (n, k), dtype=torch.uint8, device=DEV, generator=gen) << 7
    sa = torch.randint(118, 126, (m, k // 32), dtype=torch.uint8, device=DEV, generator=gen)
    sw = torch.randint(110, 118, ((n + 31) // 32, k // 32), dtype=torch.uint8, device=DEV, generator=gen)
    fa = torch.rand((m, k // 128), device=DEV, generator=gen) + 0.1
    fw = torch.rand(((n + 127) // 128, k // 128), device=DEV, generator=gen) + 0.1
    table = torch.from_numpy(O.e4m3_decode_table().astype(np.float64)).to(DEV)
    pw = lambda s: torch.pow(2.0, s.to(torch.float64) - 127)
    ca, cw = table[aq.long()], table[wq.long()]
    ws = torch.empty(L.gemm_workspace_size(m, n, k), dtype=torch.uint8, device=DEV)
    if split and ws.numel():
        L.set_gemm_workspace(ws)
    try:
        for what in ("ue8m0", "f32s"):
            out = torch.full((m * n + 64,), -7.0, dtype=torch.bfloat16, device=DEV)
            if what == "ue8m0":
                L.fp8_gemm_bf16(aq, sa, wq, sw, out, m, n, k)
                da = ca * pw(sa).repeat_interleave(32, 1)
                dw = cw * pw(sw).repeat_interleave(32, 0)[:n].repeat_interleave(32, 1)
            else:
                L.fp8_gemm_f32s(aq, fa, wq, fw, out, m, n, k, out_bf16=True)
                da = ca * fa.double().repeat_interleave(128, 1)
                dw = cw * fw.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)
            assert (out[m * n:] == -7).all(), "written past the output"
            want = da @ dw.T
            roundings = k // 32 + k // 128 + 2 + 8
            bound = 2.0 ** -8 * want.abs() + roundings * 2.0 ** -23 * (da.abs() @ dw.abs().T)
            assert ((out[:m * n].view(m, n).double() - want).abs() <= bound).all(), what
    finally:
        L.set_gemm_workspace(None)


@pytest.mark.parametrize("m", [65, 130, 520])
def test_packed_scale_table_above_64_rows(m):
    """ws_fp8_gemm_tl above 64 rows (the column-strip kernel): per-row weight
    scale words, each row with scales of its own, against f64."""
    kind = L.TL_QB
    n, k = L.tl_gemm_shape(kind)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(m)
    announce("packed scale table m=%d" % m)
    x = torch.randn((m, k), device=DEV, generator=gen)
    aq = torch.empty((m, k), dtype=torch.uint8, device=DEV)
    as_ = torch.empty((m, k // 32), dtype=torch.uint8, device=DEV)
    L.emit8(x, aq, as_, m * k)
    wq = torch.randint(0, 120, (n, k), dtype=torch.uint8, device=DEV, generator=gen)
    ws = torch.randint(110, 124, (n, k // 32), dtype=torch.uint8, device=DEV, generator=gen)
    out = torch.empty((m, n), device=DEV)
    L.fp8_gemm_tl(kind, aq, as_, wq, ws, out, m)
    table = torch.from_numpy(O.e4m3_decode_table().astype(np.float64)).to(DEV)
    pw = lambda s: torch.pow(2.0, s.to(torch.float64) - 127)
    want = (table[aq.long()] * pw(as_).repeat_interleave(32, 1)) @ \
        (table[wq.long()] * pw(ws).repeat_interleave(32, 1)).T
    err = float((out.double() - want).norm() / want.norm())
    assert err <= 40 ** 0.5 * 2.0 ** -24, err


def test_tile_gemm_special_scales_match_strips():
    """Scale bytes 0 (2^-127) and 255 (NaN) and NaN codes: the tile kernel's
    rows against the strips that the same rows take 64 at a time."""
    m, n, k = 256, 512, 640
    rng = np.random.default_rng(77)
    aq = rng.integers(0, 256, (m, k)).astype(np.uint8)
    aq[aq % 128 == 127] = 0x30
    aq[5, 77] = 0x7F
    as_ = rng.integers(100, 130, (m, k // 32)).astype(np.uint8)
    as_[9, 3], as_[10, 4], as_[70] = 0, 255, 0
    wq = rng.integers(0, 126, (n, k)).astype(np.uint8)
    ws = rng.integers(100, 130, (n // 32, k // 32)).astype(np.uint8)
    ws[2, 1], ws[3, 2] = 0, 255
    announce("tile gemm special scales")
    a, sa, w, sw = dev(aq), dev(as_), dev(wq), dev(ws)
    got = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)  # what the tiles serve
    L.fp8_gemm_bf16(a, sa, w, sw, got, m, n, k)
    want = torch.empty((m, n), device=DEV)
    for r in range(0, m, 64):
        L.fp8_gemm(a[r:r + 64], sa[r:r + 64], w, sw, want[r:r + 64], 64, n, k)
    g, wt = host(got.float()), host(want)
    assert np.isnan(wt).any() and np.array_equal(np.isnan(g), np.isnan(wt))
    ok = ~np.isnan(wt)
    # bf16 rounds to within 2^-8 of a value, the f32 sums differ by 1e-5
    assert_close(g[ok], wt[ok], 2.0 ** -8 + 1e-5, "special scales")
