"""GPU parity of the grouped (M-token) routed MoE: the dispatch is integer
work and bit-exact with the oracle's restatement of moe_dispatch_kernel's
contract; the grouped MoE output matches the per-token CPU MoE
(weightstream-ref moe.rs:75-84,162-208) within max relative error 1e-3
(floor at 1% of the output scale), the tolerance of the decode path.

The hidden state h is re-quantised to FP8 between the two GEMMs. An element
of h whose exact value sits within f32 reassociation distance of an e4m3
rounding midpoint can land one step apart in the oracle (sequential f32 dot)
and on the GPU (MFMA accumulation); that step, times one column of w2, can
exceed the end-to-end tolerance. A row that misses the tolerance is therefore
re-checked stage by stage: every element where the GPU's h differs from the
oracle's must be such a midpoint case (adjacent e4m3 values, the oracle's f32 h within
1e-4 of the block's scale from the midpoint), and the output must then match
the oracle's down projection and expert-ordered sum of the GPU's h within the
same tolerance."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from gpu_util import DEV, announce, assert_close, dev, host, rand_fp4_weights, rel_err_stats
from weightstream_amd import launch as L

pytestmark = pytest.mark.gpu
MOE_TOL = 1e-3


@pytest.fixture(scope="module", autouse=True)
def _init():
    L.Hip.global_()


def zipf_routing(rng, m, E, k, s=1.1):
    """logits N(0,1) skewed by log Zipf(s) popularity."""
    pop = 1.0 / np.arange(1, E + 1) ** s
    bias = (rng.standard_normal(E) * 0.1).astype(np.float32)
    logits = (rng.standard_normal((m, E)) + np.log(pop)[rng.permutation(E)]).astype(np.float32)
    return logits, bias


def _dispatch_gpu(idx, w, E, tiles):
    routes = idx.size
    out = dict(order=torch.full((tiles * 32,), -7, dtype=torch.int32, device=DEV),
               layout_w=torch.full((tiles * 32,), -7.0, dtype=torch.float32, device=DEV),
               route_pos=torch.empty(routes, dtype=torch.int32, device=DEV),
               tile_expert=torch.empty(tiles, dtype=torch.int32, device=DEV),
               count=torch.empty(E, dtype=torch.int32, device=DEV),
               offset=torch.empty(E, dtype=torch.int32, device=DEV),
               psum=torch.empty(E, dtype=torch.int32, device=DEV),
               num_tiles=torch.empty(1, dtype=torch.int32, device=DEV))
    L.moe_dispatch_tl(dev(idx), dev(w), out["order"], out["layout_w"], out["route_pos"],
                      out["tile_expert"], out["count"], out["offset"], out["psum"],
                      out["num_tiles"], idx.shape[0], idx.shape[1], tiles, E)
    return {k: host(v) for k, v in out.items()}


@pytest.mark.parametrize("m,E,k", [(132, 384, 8), (1, 384, 8), (3, 16, 2), (300, 1024, 8),
                                   (700, 96, 6), (1100, 384, 8)])
def test_dispatch_bit_exact(m, E, k):
    rng = np.random.default_rng(800 + m + E)
    logits, bias = zipf_routing(rng, m, E, k)
    idx = np.argsort(-(logits + bias), axis=1, kind="stable")[:, :k].astype(np.int32)
    if m == 3:
        idx[1, 1] = -1                       # a non-local expert is dropped
    w = rng.random((m, k)).astype(np.float32)
    tiles = L.moe_tiles(m * k, E)
    announce("moe_dispatch m=%d E=%d k=%d" % (m, E, k))
    got = _dispatch_gpu(idx, w, E, tiles)
    want = O.dispatch(idx, w, E, tiles)
    nt = want["num_tiles"]
    assert got["num_tiles"][0] == nt
    for key in ("route_pos", "tile_expert", "count", "offset", "psum"):
        assert np.array_equal(got[key], want[key]), key
    used = nt * 32
    assert np.array_equal(got["order"][:used], want["order"][:used])
    assert np.array_equal(got["layout_w"][:used].view(np.uint32),
                          want["layout_w"][:used].view(np.uint32))


@pytest.mark.parametrize("m,E,k", [(512, 384, 8), (513, 384, 8), (4097, 5, 1), (900, 1024, 16)])
def test_dispatch_with_dropped_ids_around_4096_routes(m, E, k):
    """Both rankings (routes held in registers up to 4096, a run of routes per
    wave above) with ids another rank owns and one popular expert."""
    rng = np.random.default_rng(820 + m)
    idx = np.stack([rng.choice(E, k, replace=False) for _ in range(m)]).astype(np.int32)
    idx[rng.random((m, k)) < 0.2] = -1
    idx[m // 3: m // 2, 0] = 2
    idx[-1] = -1
    w = rng.random((m, k)).astype(np.float32)
    tiles = L.moe_tiles(m * k, E)
    announce("moe_dispatch with dropped ids m=%d E=%d k=%d" % (m, E, k))
    got, want = _dispatch_gpu(idx, w, E, tiles), O.dispatch(idx, w, E, tiles)
    used = want["num_tiles"] * 32
    assert got["num_tiles"][0] == want["num_tiles"]
    for key in ("route_pos", "tile_expert", "count", "offset", "psum"):
        assert np.array_equal(got[key], want[key]), key
    for key in ("order", "layout_w"):
        assert np.array_equal(got[key][:used].view(np.uint32), want[key][:used].view(np.uint32)), key


@pytest.mark.parametrize("rows", [2047, 2048])   # one row per add; groups of 4, 6 or 8
@pytest.mark.parametrize("top_k", [1, 3, 4, 5, 6, 7, 8, 9, 16])
def test_combine_adds_in_slot_order(rows, top_k):
    """The ordered sum of a row's slots, dropped ones left out, whole and ragged
    groups of loads: the bits of the same f32 adds, infinities and NaN among them."""
    dim, tiles = 132, 64
    rng = np.random.default_rng(830 + top_k)
    down = rng.standard_normal((tiles * 32, dim)).astype(np.float32)
    down[5, 3], down[9, 4], down[11, 5] = np.inf, -np.inf, np.nan
    pos = np.stack([rng.choice(tiles * 32, top_k, replace=False) for _ in range(rows)]).astype(np.int32)
    pos[rng.random(pos.shape) < 0.1] = -1
    pos[1] = -1
    out = torch.full((rows * dim + 64,), -7.0, device=DEV)
    announce("combine rows=%d top_k=%d" % (rows, top_k))
    L.moe_combine_f32(dev(down), dev(pos), out, dim, top_k, rows, tiles)
    want = np.zeros((rows, dim), np.float32)
    padded = np.concatenate([down, np.zeros((1, dim), np.float32)])
    order = np.sort(np.where(pos < 0, tiles * 32, pos), axis=1)
    for j in range(top_k):
        # a dropped slot adds nothing: the sum stays (+0 for a row of none)
        want = np.where((order[:, j] < tiles * 32)[:, None], want + padded[order[:, j]], want)
    got = host(out)
    assert (got[rows * dim:] == -7).all()
    got, nan = got[:rows * dim].reshape(rows, dim), np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


def _slabs(gen, E, dim, inter):
    """Raw (on-disk layout) expert slabs; the kernels read _packed(raw)."""
    w1, s1 = rand_fp4_weights(gen, E * inter, dim)
    w3, s3 = rand_fp4_weights(gen, E * inter, dim)
    w2, s2 = rand_fp4_weights(gen, E * dim, inter)
    return w1, s1, w3, s3, w2, s2


def _packed(raw, E, dim, inter):
    w1, s1, w3, s3, w2, s2 = raw
    p1 = L.prepack_fp4_new(w1, s1, E * inter, dim)
    p3 = L.prepack_fp4_new(w3, s3, E * inter, dim)
    p2 = L.prepack_fp4_new(w2, s2, E * dim, inter)
    return p1 + p3 + p2


def _host_experts(slabs, experts, E, dim, inter):
    shapes = [(inter, dim // 2), (inter, dim // 32), (inter, dim // 2), (inter, dim // 32),
              (dim, inter // 2), (dim, inter // 32)]
    out = []
    for t, shp in zip(slabs, shapes):
        h = np.zeros((E,) + shp, np.uint8)
        tv = t.view(E, *shp)
        for e in sorted(set(int(v) for v in experts)):
            h[e] = tv[e].cpu().numpy()
        out.append(h)
    return out


@pytest.mark.parametrize("m,E,dim,inter,k,check", [(40, 64, 1024, 512, 6, 40),
                                                    (132, 384, 4096, 2048, 8, 6),
                                                    # few tiles: the tile-streaming pair
                                                    (8, 384, 4096, 2048, 8, 8),
                                                    # the expert-stationary pair at other
                                                    # shapes (K of one ring round: 1024)
                                                    (128, 16, 2048, 1024, 4, 8),
                                                    (200, 32, 1024, 1024, 6, 8),
                                                    (400, 16, 8192, 4096, 2, 4),
                                                    (5, 16, 512, 256, 4, 5),
                                                    (96, 64, 5120, 2304, 6, 6),
                                                    (33, 8, 8192, 4096, 2, 4),
                                                    # >= 192 tiles: two bands per wave; dim
                                                    # % 256 == 128 leaves the last down unit
                                                    # half empty
                                                    (40, 256, 640, 384, 6, 10),
                                                    (64, 256, 5120, 2304, 6, 6)])
def test_moe_prefill_matches_oracle(m, E, dim, inter, k, check):
    _check_prefill(m, E, dim, inter, k, check)


def _check_prefill(m, E, dim, inter, k, check, s=1.1):
    """ws_moe_prefill against the oracle on `check` rows, popularity Zipf(s);
    returns the bodies that ran, which must be those the rules name."""
    rng = np.random.default_rng(900 + m + E)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(900 + m)
    announce("moe_prefill m=%d E=%d dim=%d inter=%d k=%d s=%.1f" % (m, E, dim, inter, k, s))
    slabs = _slabs(gen, E, dim, inter)
    logits, bias = zipf_routing(rng, m, E, k, s)
    idx = torch.empty((m, k), dtype=torch.int32, device=DEV)
    w = torch.empty((m, k), dtype=torch.float32, device=DEV)
    L.moe_topk(dev(logits), dev(bias), None, idx, w, m, E, k, O.SCORE_SIGMOID, 1.0, True, 1.0)
    x = rng.standard_normal((m, dim)).astype(np.float32)
    ws = _prefill_workspace(m, dim, inter, k, E)
    y = torch.empty((m, dim), dtype=torch.float32, device=DEV)
    L.moe_prefill(dev(x), idx, w, *_packed(slabs, E, dim, inter), y, m, dim, inter, E, k, ws)
    body = _body_ran(ws, m, dim, inter, k, E)
    print("[moe_prefill m=%d E=%d dim=%d inter=%d] %s bodies" % (m, E, dim, inter, body), flush=True)
    assert body == _body_expected(idx, E, dim, inter)
    gi, gw, gy = host(idx), host(w), host(y)
    rows = np.linspace(0, m - 1, check).astype(int)
    H = _host_experts(slabs, gi[rows].ravel(), E, dim, inter)
    staged = None
    for r in rows:
        want = O.moe_routed(*H, dim, inter, x[r], gi[r], gw[r])
        if rel_err_stats(gy[r], want)[0] <= MOE_TOL:
            assert_close(gy[r], want, MOE_TOL, "moe_prefill row %d" % r)
            continue
        if staged is None:
            staged = _staged_hidden(x, idx, w, _packed(slabs, E, dim, inter), m, E, dim, inter, k)
        _check_by_stages(gy[r], x[r], gi[r], gw[r], H, staged, r, k, dim, inter)
    return body


@pytest.mark.parametrize("m,E,dim,inter,k", [(120, 16, 768, 384, 4), (200, 32, 2304, 1152, 6),
                                             (300, 24, 1280, 640, 4), (130, 8, 256, 128, 2),
                                             (100, 64, 5120, 2432, 6)])
def test_moe_prefill_stationary_step_counts(m, E, dim, inter, k):
    """The expert-stationary pair with units of every remainder of four 128-K
    steps (6 and 3, 18 and 9, 10 and 5, 2 and 1, 40 and 19): a unit's repeated
    steps past K multiply nothing. Skewed enough that the dispatch takes it."""
    assert _check_prefill(m, E, dim, inter, k, 6) == "stationary"


@pytest.mark.parametrize("m,E,dim,inter,k", [(600, 16, 768, 384, 4), (1000, 32, 1280, 640, 4),
                                             (4600, 64, 512, 256, 8), (700, 8, 2304, 1152, 2),
                                             (260, 3, 640, 128, 3)])
def test_moe_prefill_group_tiles(m, E, dim, inter, k):
    """The 96-slot groups (96 or more routes per expert): experts with no route,
    fewer than 32, every strip count and several groups; step counts of every
    remainder of four (6 and 3, 10 and 5, 4 and 2, 18 and 9, 5 and 1); column
    blocks cut short (inter 384, 640, 1152, 128 of 256; dim 768, 1280, 2304, 640
    of 512)."""
    assert _check_prefill(m, E, dim, inter, k, 6) == "groups"


@pytest.mark.parametrize("m,E,inter,k", [(512, 128, 2048, 8), (512, 64, 1024, 8),
                                         (576, 48, 1024, 8)])
def test_moe_prefill_both_sides_of_the_group_line(m, E, inter, k):
    """The groups from 32 routes per expert on (four column blocks of 256 or more per
    CU), 64 (one or more) or 96, and the stationary pair with a token less."""
    dim = 256
    assert m * k == E * {2048: 32, 1024: 64 if E == 64 else 96}[inter]
    assert _check_prefill(m, E, dim, inter, k, 4) == "groups"
    assert _check_prefill(m - 1, E, dim, inter, k, 4) == "stationary"


@pytest.mark.parametrize("m,E,dim,inter,k,s,body",
                         [(40, 256, 1792, 384, 8, 0.0, "streaming"),    # K halves of 8 + 6
                          (40, 256, 2304, 384, 8, 0.0, "stationary"),   # 8 + 10
                          (40, 256, 3328, 384, 8, 0.0, "streaming"),    # 16 + 10
                          (40, 256, 4096, 384, 8, 0.0, "streaming"),    # 16 + 16
                          (40, 256, 4352, 384, 8, 0.0, "stationary"),   # above one pass of A
                          (40, 256, 2048, 1024, 8, 0.0, "stationary"),  # whole units
                          (300, 256, 1792, 384, 6, 0.0, "stationary"),  # tiles over 16 rows
                          (40, 256, 1792, 384, 8, 1.1, None)])          # skewed
def test_moe_prefill_choice_at_an_even_routing(m, E, dim, inter, k, s, body):
    """Padded units leave 100 or more short tiles to the tile-streaming pair where
    its K halves differ little."""
    got = _check_prefill(m, E, dim, inter, k, 4, s)
    assert body is None or got == body


@pytest.mark.parametrize("m,E,dim,inter,k,body", [(600, 1024, 512, 256, 8, "streaming"),
                                                  (1024, 1024, 512, 256, 8, "groups"),
                                                  (96, 16, 384, 256, 4, "streaming")])
def test_moe_prefill_past_the_stationary_limits(m, E, dim, inter, k, body):
    """More than 1024 tiles, under and from 8 routes per expert; dim not a multiple
    of 256."""
    assert _check_prefill(m, E, dim, inter, k, 4) == body


@pytest.mark.parametrize("m,check", [(132, 12), (300, 12), (4500, 8)])
def test_prefill_all_routes_on_k_experts(m, check):
    """Every token picks the same k experts (their bias lifts them above the
    rest; the routing weights still vary per token), so each expert holds m
    routes: ceil(m / 32) tiles, pairs of full tiles and a ragged last one in
    the expert-stationary groups (m = 132: 5 tiles per expert, groups of
    2, 2, 1; m = 300: 10 tiles, five full pairs, the last tile 12 rows). At
    m = 4500 the tile capacity exceeds what the stationary bodies take and
    the 96-slot groups run 47 of them per expert, the last two strips short."""
    E, dim, inter, k = 64, 2048, 1024, 8
    rng = np.random.default_rng(1700 + m)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1700 + m)
    announce("moe_prefill all routes on %d experts m=%d" % (k, m))
    slabs = _slabs(gen, E, dim, inter)
    hot = rng.choice(E, k, replace=False)
    bias = (rng.standard_normal(E) * 0.1).astype(np.float32)
    bias[hot] += 10.0
    logits = rng.standard_normal((m, E)).astype(np.float32)
    idx = torch.empty((m, k), dtype=torch.int32, device=DEV)
    w = torch.empty((m, k), dtype=torch.float32, device=DEV)
    L.moe_topk(dev(logits), dev(bias), None, idx, w, m, E, k, O.SCORE_SIGMOID, 1.0, True, 1.0)
    gi = host(idx)
    assert sorted(set(gi.ravel().tolist())) == sorted(hot.tolist())
    x = rng.standard_normal((m, dim)).astype(np.float32)
    ws = _prefill_workspace(m, dim, inter, k, E)
    y = torch.empty((m, dim), dtype=torch.float32, device=DEV)
    L.moe_prefill(dev(x), idx, w, *_packed(slabs, E, dim, inter), y, m, dim, inter, E, k, ws)
    body = _body_ran(ws, m, dim, inter, k, E)
    print("[all routes on k experts m=%d] %s bodies" % (m, body), flush=True)
    assert body == _body_expected(idx, E, dim, inter) == ("stationary" if m <= 300 else "groups")
    gw, gy = host(w), host(y)
    # the first and last rows (first and last tile of every expert) and
    # rows spread between them
    rows = np.linspace(0, m - 1, check).astype(int)
    H = _host_experts(slabs, hot, E, dim, inter)
    staged = None
    for r in rows:
        want = O.moe_routed(*H, dim, inter, x[r], gi[r], gw[r])
        if rel_err_stats(gy[r], want)[0] <= MOE_TOL:
            assert_close(gy[r], want, MOE_TOL, "moe_prefill row %d" % r)
            continue
        if staged is None:
            staged = _staged_hidden(x, idx, w, _packed(slabs, E, dim, inter), m, E, dim, inter, k)
        _check_by_stages(gy[r], x[r], gi[r], gw[r], H, staged, r, k, dim, inter)


def _fp4_normal_slab(gen, E, rows, cols, chunk=64):
    """E expert matrices [rows, cols] drawn N(0, 0.02) and encoded e2m1 +
    UE8M0 per 1x32 on the device (the BASELINE weight recipe)."""
    q = torch.empty((E * rows, cols // 2), dtype=torch.uint8, device=DEV)
    s = torch.empty((E * rows, cols // 32), dtype=torch.uint8, device=DEV)
    for e0 in range(0, E, chunk):
        n = min(chunk, E - e0) * rows
        wt = torch.empty((n, cols), dtype=torch.float32, device=DEV).normal_(0.0, 0.02,
                                                                            generator=gen)
        L.weight_quant_fp4(wt, q[e0 * rows:e0 * rows + n], s[e0 * rows:e0 * rows + n], n, cols)
        del wt
    return q, s


def _a256(v):
    return (v + 255) // 256 * 256


def _body_expected(idx, E, dim, inter):
    """The bodies ws_moe_prefill should take. From 32, 64 or 96 routes per
    expert on, by the expert's column blocks, or from 8 where the capacity is
    over 1024 tiles, the groups. With t_e = ceil(routes of expert e / 32) tiles, nt =
    sum t_e and ng = sum ceil(t_e / 2) groups, the stationary pair when 6 (nt
    - ng) >= nt or nt >= 96; but not on the tile count alone, from 100 tiles, when
    fewer than 1 in 128 holds over 16 rows, units are padded, dim <= 4096 and the
    first K half is the longer one and at most 8 / 13 of the whole."""
    cnt = np.bincount(host(idx).ravel(), minlength=E)
    routes, tiles = host(idx).size, L.moe_tiles(host(idx).size, E)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    blocks = E * ((inter + 255) // 256)
    steps = dim // 128
    padded = bool(steps % 8 or inter // 128 % 8)
    per = 32 if blocks >= (4 if padded else 8) * cus else 64 if blocks >= cus else 96
    if routes >= E * (8 if tiles > 1024 else per):
        return "groups"
    if dim % 256 or tiles > 1024:
        return "streaming"
    t = (cnt + 31) // 32
    nt, ng = int(t.sum()), int(((t + 1) // 2).sum())
    full = int((cnt // 32 + (cnt % 32 > 16)).sum())
    first = (steps + 7) // 8 // 2 * 8
    balanced = padded and dim <= 4096 and 2 * first >= steps and 13 * first <= 8 * steps
    if 6 * (nt - ng) >= nt:
        return "stationary"
    return "stationary" if nt >= 96 and not (balanced and nt >= 100 and 128 * full < nt) else "streaming"


_UNTOUCHED = 0x5A


def _prefill_workspace(m, dim, inter, k, E):
    return torch.full((L.moe_prefill_workspace_size(m, dim, inter, k, E),), _UNTOUCHED,
                      dtype=torch.uint8, device=DEV)


def _body_ran(ws, m, dim, inter, k, E):
    """The bodies that ws_moe_prefill took with a workspace from
    _prefill_workspace. Its regions (in order, each 256-byte aligned) are xq, xs,
    order, layout_w, route_pos, tile_expert, three per-expert arrays, the tile count
    and the dispatch's choice (int32s: 1 stationary, 0 tile-streaming), hq, hs,
    down, the bf16 tokens and the bf16 h. The groups and the plain tile-streaming
    pair make no choice; only the groups write the bf16 h."""
    routes = m * k
    slots = L.moe_tiles(routes, E) * 32
    off = (_a256(m * dim) + _a256(m * dim // 32) + 2 * _a256(slots * 4) + _a256(routes * 4) +
           _a256(slots // 32 * 4) + 3 * _a256(E * 4))
    choice = int(host(ws[off + 4:off + 8]).view(np.int32)[0])
    if choice in (0, 1):
        return "stationary" if choice else "streaming"
    assert choice == 0x01010101 * _UNTOUCHED
    hbf = ws[ws.numel() - _a256(slots * inter * 2):][:slots * inter * 2]
    return "groups" if bool((hbf != _UNTOUCHED).any()) else "streaming"


@pytest.mark.parametrize("zipf", [1.1, 0.275])
def test_config4_baseline_weights_prefill_matches_oracle(zipf):
    """BASELINE config 4 as the bench runs it: M = 132 tokens, 384 experts of
    N(0, 0.02) weights in e2m1 + UE8M0, dim 4096, inter 2048, top-8 sigmoid
    routing of N(0, 1) logits skewed by Zipf(1.1) popularity (and the bench's
    quarter-strength draw, 0.25 log Zipf(1.1) = log Zipf(0.275)), against the
    oracle on sampled rows."""
    m, E, dim, inter, k = 132, 384, 4096, 2048, 8
    rng = np.random.default_rng(4004)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(4004)
    announce("config 4: m=%d, %d experts of N(0, 0.02) weights, Zipf s=%.2f" % (m, E, zipf))
    slabs = _fp4_normal_slab(gen, E, inter, dim) + _fp4_normal_slab(gen, E, inter, dim) + \
        _fp4_normal_slab(gen, E, dim, inter)
    logits, bias = zipf_routing(rng, m, E, k, s=zipf)
    idx = torch.empty((m, k), dtype=torch.int32, device=DEV)
    w = torch.empty((m, k), dtype=torch.float32, device=DEV)
    L.moe_topk(dev(logits), dev(bias), None, idx, w, m, E, k, O.SCORE_SIGMOID, 1.0, True, 1.0)
    x = rng.standard_normal((m, dim)).astype(np.float32)
    ws = _prefill_workspace(m, dim, inter, k, E)
    y = torch.empty((m, dim), dtype=torch.float32, device=DEV)
    P = _packed(slabs, E, dim, inter)
    L.moe_prefill(dev(x), idx, w, *P, y, m, dim, inter, E, k, ws)
    # both draws run the expert-stationary bodies (the skewed one for its
    # shared groups, the mild one for its tile count)
    assert _body_ran(ws, m, dim, inter, k, E) == _body_expected(idx, E, dim, inter) == "stationary"
    gi, gw, gy = host(idx), host(w), host(y)
    H = _host_experts(slabs, gi.ravel(), E, dim, inter)
    staged = None
    ok = []
    O.set_threads(16)   # the oracle's GEMV rows in threads: the same bits
    try:
        want = np.stack([O.moe_routed(*H, dim, inter, x[r], gi[r], gw[r]) for r in range(m)])
    finally:
        O.set_threads(1)
    for r in range(m):   # every row of the benched batch
        if rel_err_stats(gy[r], want[r])[0] <= MOE_TOL:
            ok.append(r)
            continue
        if staged is None:
            staged = _staged_hidden(x, idx, w, P, m, E, dim, inter, k)
        _check_by_stages(gy[r], x[r], gi[r], gw[r], H, staged, r, k, dim, inter)
    # the distribution over all rows that met the bar directly
    print("[config 4 zipf %.3g] %d of %d rows direct, %d by stages" % (zipf, len(ok), m,
                                                                      m - len(ok)), flush=True)
    assert_close(gy[ok], want[ok], MOE_TOL, "config 4 zipf %.3g, all direct rows" % zipf)


def _staged_hidden(x, idx, w, P, m, E, dim, inter, k):
    """The GPU's re-quantised h per slot (emit8 + dispatch + grouped gate/up),
    decoded to f32, and route -> slot."""
    routes = m * k
    tiles = L.moe_tiles(routes, E)
    xq = torch.empty((m, dim), dtype=torch.uint8, device=DEV)
    xs = torch.empty((m, dim // 32), dtype=torch.uint8, device=DEV)
    L.emit8(dev(x), xq, xs, m * dim)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device=DEV)
    order, rp, te, nt = i32(tiles * 32), i32(routes), i32(tiles), i32(1)
    lw = torch.empty(tiles * 32, dtype=torch.float32, device=DEV)
    L.moe_dispatch_tl(idx, w, order, lw, rp, te, i32(E), i32(E), i32(E), nt, m, k, tiles, E)
    hq = torch.zeros((tiles * 32, inter), dtype=torch.uint8, device=DEV)
    hs = torch.zeros((tiles * 32, inter // 32), dtype=torch.uint8, device=DEV)
    L.moe_grouped_glu_quant(xq, xs, order, lw, te, nt, P[0], P[1], P[2], P[3], hq, hs, dim,
                            inter, E, k, tiles, 10.0)
    torch.cuda.synchronize()
    tab = O.e4m3_decode_table().astype(np.float64)
    h = tab[host(hq)] * np.repeat(2.0 ** (host(hs).astype(np.float64) - 127), 32, axis=1)
    return h, host(rp)


def _check_by_stages(got_row, x_row, gi, gw, H, staged, r, k, dim, inter, limit=10.0):
    h_gpu, route_pos = staged
    check_routed_by_stages(got_row, x_row, gi, gw, H, lambda j: h_gpu[route_pos[r * k + j]],
                           "moe_prefill row %d" % r, dim, inter, limit)


def check_routed_by_stages(got_row, x_row, gi, gw, H, h_of_pick, what, dim, inter, limit=10.0):
    """A routed-MoE row that missed the tolerance: every element where the
    GPU's re-quantised h (h_of_pick(j), decoded, for pick j) differs from the
    oracle's must be a rounding-midpoint case, and the output must match the
    oracle's down projection of the GPU's h. H[i][e]: expert e's w1, s1, w3,
    s3, w2, s2 as the oracle takes them."""
    y = np.zeros(dim, np.float32)
    flips = 0
    for j in np.argsort(gi, kind="stable"):  # expert order, as moe.rs:75-84 sums
        e, rw = int(gi[j]), float(gw[j])
        # the oracle's own f32 hidden state and its snap, as moe_routed computes them
        h32 = O.expert_hidden_fp4(H[0][e], H[1][e], H[2][e], H[3][e], dim, inter, x_row, rw,
                                  limit)
        h_pre = h32.astype(np.float64)
        h_or = O.fp8_snap(h32).astype(np.float64)
        hg = h_of_pick(j)
        for i in np.nonzero(hg != h_or)[0]:
            blk = np.abs(h_or[i // 32 * 32:(i // 32 + 1) * 32]).max()
            mid = 0.5 * (hg[i] + h_or[i])
            assert abs(hg[i] - h_or[i]) <= blk / 8, "%s h[%d]: not adjacent" % (what, i)
            assert abs(h_pre[i] - mid) <= 1e-4 * blk, \
                "%s h[%d]: %r vs %r, not a rounding midpoint" % (what, i, hg[i], h_or[i])
            flips += 1
        y += O.fp4_gemv(H[4][e], H[5][e], dim, inter, hg.astype(np.float32))
    print("[%s] %d h element(s) on an e4m3 rounding midpoint" % (what, flips), flush=True)
    assert flips > 0, "%s misses the tolerance with h identical to the oracle's" % what
    assert_close(got_row, y, MOE_TOL, what + " (staged)")


def test_prefill_of_one_token_matches_decode():
    rng = np.random.default_rng(950)
    E, dim, inter, k = 32, 1024, 512, 4
    gen = torch.Generator(device=DEV)
    gen.manual_seed(950)
    slabs = _packed(_slabs(gen, E, dim, inter), E, dim, inter)
    x = dev(rng.standard_normal((1, dim)).astype(np.float32))
    idx = dev(np.array([[9, 2, 30, 17]], np.int32))
    w = dev(np.array([[0.4, 0.3, 0.2, 0.1]], np.float32))
    announce("prefill(1) vs decode")
    ws = torch.empty(L.moe_prefill_workspace_size(1, dim, inter, k, E), dtype=torch.uint8,
                     device=DEV)
    y1 = torch.empty((1, dim), dtype=torch.float32, device=DEV)
    L.moe_prefill(x, idx, w, *slabs, y1, 1, dim, inter, E, k, ws)
    wsd = torch.empty(L.moe_decode_workspace_size(dim, inter, k), dtype=torch.uint8, device=DEV)
    y2 = torch.empty(dim, dtype=torch.float32, device=DEV)
    L.moe_decode(x[0], idx[0], w[0], *slabs, y2, dim, inter, E, k, wsd)
    assert_close(host(y1)[0], host(y2), MOE_TOL, "prefill(1) vs decode")


def test_moe_prefill_rejects_oversized_shapes():
    """dim above 8192 or inter above 4096 do not fit the LDS-staged A tile."""
    k, E = 2, 4
    for dim, inter in [(8320, 256), (256, 4224)]:
        ws = torch.empty(L.moe_prefill_workspace_size(4, dim, inter, k, E), dtype=torch.uint8,
                         device=DEV)
        b = torch.zeros(1 << 12, dtype=torch.uint8, device=DEV)
        f = torch.zeros(4 * dim, dtype=torch.float32, device=DEV)
        idx = torch.zeros((4, k), dtype=torch.int32, device=DEV)
        w = torch.zeros((4, k), dtype=torch.float32, device=DEV)
        with pytest.raises(RuntimeError, match="unsupported shape"):
            L.moe_prefill(f, idx, w, b, b, b, b, b, b, f, 4, dim, inter, E, k, ws)


@pytest.mark.parametrize("m,E,dim,inter,k", [(40, 64, 1024, 512, 6), (9, 16, 512, 256, 4),
                                             (40, 256, 640, 384, 6),
                                             # stationary, padded units: gate/up K parts of 8
                                             # and 10, 8 and 2, 16 and 24, 0 and 2, 0 and 6,
                                             # 16 and 16 steps
                                             (200, 32, 2304, 1152, 6), (300, 24, 1280, 640, 4),
                                             (100, 64, 5120, 2432, 6), (130, 8, 256, 128, 2),
                                             (120, 16, 768, 384, 4), (200, 48, 4096, 2176, 4),
                                             # 96-slot groups: a slice of scratch per workgroup
                                             # and (few slots, dim 1280 and 2304) per strip
                                             (1000, 32, 1280, 640, 4), (700, 8, 2304, 1152, 2),
                                             (600, 16, 768, 384, 4), (4600, 64, 512, 256, 8),
                                             (4000, 96, 2048, 1024, 6), (2000, 64, 5120, 640, 8)])
def test_prefill_stages_compose_to_moe_prefill(m, E, dim, inter, k):
    """emit8 -> dispatch -> grouped gate/up -> grouped down (every slot) ->
    combine through the public entry points gives the bits of ws_moe_prefill
    (which multiplies and writes only the slots that hold routes), on the
    tile-streaming pair and on the bodies that take its place (not on the
    stationary pair's whole units: dim and inter in 1024s)."""
    y1, y2, _ = _composed(m, E, dim, inter, k)
    assert np.array_equal(y1.view(np.uint32), y2.view(np.uint32))


def _composed(m, E, dim, inter, k, nonfinite=False):
    """y of ws_moe_prefill, y of its stages, the bodies that ws_moe_prefill took."""
    rng = np.random.default_rng(990 + m)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(990 + m)
    slabs = _slabs(gen, E, dim, inter)
    if nonfinite:  # scale bytes of NaN, 2^-127 and 2^127 in one row or another of three experts
        for j, rows in ((1, inter), (3, inter), (5, dim)):
            slabs[j].view(E, rows, -1)[0, 3, 1] = 255
            slabs[j].view(E, rows, -1)[1, 17, 0] = 0
            slabs[j].view(E, rows, -1)[2, 5, -1] = 254
    P = _packed(slabs, E, dim, inter)
    logits, bias = zipf_routing(rng, m, E, k)
    idx = torch.empty((m, k), dtype=torch.int32, device=DEV)
    w = torch.empty((m, k), dtype=torch.float32, device=DEV)
    L.moe_topk(dev(logits), dev(bias), None, idx, w, m, E, k, O.SCORE_SIGMOID, 1.0, True, 1.0)
    hx = rng.standard_normal((m, dim)).astype(np.float32)
    if nonfinite:
        hx[1, 7], hx[2, 40], hx[3, dim - 1] = np.inf, -np.inf, np.nan
        hx[4], hx[5], hx[6] = np.nan, 3e38, np.float32(1e30) * hx[6]
    x = dev(hx)
    announce("prefill stages m=%d E=%d dim=%d inter=%d k=%d" % (m, E, dim, inter, k))
    ws = _prefill_workspace(m, dim, inter, k, E)
    y1 = torch.empty((m, dim), dtype=torch.float32, device=DEV)
    L.moe_prefill(x, idx, w, *P, y1, m, dim, inter, E, k, ws)

    routes, tiles = m * k, L.moe_tiles(m * k, E)
    xq = torch.empty((m, dim), dtype=torch.uint8, device=DEV)
    xs = torch.empty((m, dim // 32), dtype=torch.uint8, device=DEV)
    L.emit8(x, xq, xs, m * dim)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device=DEV)
    order, rp, te, nt = i32(tiles * 32), i32(routes), i32(tiles), i32(1)
    lw = torch.empty(tiles * 32, dtype=torch.float32, device=DEV)
    L.moe_dispatch_tl(idx, w, order, lw, rp, te, i32(E), i32(E), i32(E), nt, m, k, tiles, E)
    hq = torch.empty((tiles * 32, inter), dtype=torch.uint8, device=DEV)
    hs = torch.empty((tiles * 32, inter // 32), dtype=torch.uint8, device=DEV)
    L.moe_grouped_glu_quant(xq, xs, order, lw, te, nt, P[0], P[1], P[2], P[3], hq, hs, dim,
                            inter, E, k, tiles, 10.0)
    down = torch.empty((tiles * 32, dim), dtype=torch.float32, device=DEV)
    L.moe_grouped_down(hq, hs, te, nt, P[4], P[5], down, dim, inter, E, tiles)
    y2 = torch.empty((m, dim), dtype=torch.float32, device=DEV)
    L.moe_combine_f32(down, rp, y2, dim, k, m, tiles)
    return host(y1), host(y2), _body_ran(ws, m, dim, inter, k, E)


@pytest.mark.parametrize("m,E,dim,inter,k,body", [(200, 32, 2304, 1152, 6, "stationary"),
                                                  (130, 8, 256, 128, 2, "stationary"),
                                                  (1000, 32, 1280, 640, 4, "groups"),
                                                  (700, 8, 2304, 1152, 2, "groups"),
                                                  (9, 16, 512, 256, 4, "streaming")])
def test_prefill_nonfinite_tokens_and_weights_compose(m, E, dim, inter, k, body):
    """Infinities, NaN and values near the type's largest in tokens, NaN and
    extreme weight scales: the same rows are NaN and the others have the same bits on
    every body."""
    y1, y2, ran = _composed(m, E, dim, inter, k, nonfinite=True)
    assert ran == body
    nan = np.isnan(y1)
    assert nan.any() and not nan.all() and np.array_equal(nan, np.isnan(y2))
    assert np.array_equal(y1[~nan].view(np.uint32), y2[~nan].view(np.uint32))
