"""GPU parity of the prefill operators behind the C ABI: the router for a token block, the
device grouping, the grouped expert FFN on the matrix cores, the token-major reduce and the
residual add. Indices, permutations, tables and the reduce are compared bit for bit; FFN
partial rows within max-abs 2e-3 / relative 1e-3 (|a-b| <= 2e-3 + 1e-3*|b|)."""
import numpy as np
import pytest

from oracle import host_logic as H
from oracle import oracle as O
from shrike_amd import capi
from shrike_amd import host as HL
from shrike_amd import synth as S
from harness import runners
from tests.helpers import Layer, assert_ffn_close, assert_rel_close, f16, ffn_rules
from tests.test_decode_gpu import DeviceLayer

pytestmark = pytest.mark.gpu
SENT = 0xFFFFFFFF


def token_rows(L: Layer, t: int, stride: int, label="prefill.x"):
    """fp16[T, stride] activations; the tail of each row past d is filler that must not be read."""
    x = S.activations_f16(L.tree, label, t * stride).reshape(t, stride).copy()
    x[:, L.d:] = 0x7E00  # NaN: any use shows
    return x.reshape(-1)


def run_router(gpu, dl, L, hidden, t, stride):
    pf = gpu.Prefill(dl.moe)
    idx, w = gpu.empty(4 * t * L.k), gpu.empty(2 * t * L.k)
    ws = gpu.empty(pf.router_workspace_bytes(t, L.ne, L.d))
    pf.encode_block(dl.router_w, dl.router_s, dl.router_b, hidden, dl.eff_scale, dl.expert_scale, dl.logit_bias,
                    idx, w, ws, t, L.ne, L.d, L.k, stride)
    gpu.synchronize()
    return pf, idx, w, ws


@pytest.mark.parametrize("router_bits,ne,d,k,t,pad", [(0, 256, 2048, 8, 48, 0), (0, 256, 2048, 8, 5, 64), (8, 32, 2880, 4, 9, 8),
                                                      (4, 64, 512, 8, 33, 0), (8, 256, 2304, 8, 1, 0)])
def test_prefill_router_bit_exact_and_equal_to_decode(gpu, router_bits, ne, d, k, t, pad):
    L = Layer(0x5EED0003 + router_bits, d, 64, ne, k, router_bits=router_bits)
    L.logit_bias = S.f32_to_bf16_bits(L.tree.key("bias").normal(ne, std=0.01))
    L.expert_scale = S.f32_to_bf16_bits(L.tree.key("escale").uniform(0.6, 1.4, ne))
    dl = DeviceLayer(gpu, L, resident=[])
    stride = d + pad
    x = token_rows(L, t, stride)
    hidden = gpu.dev(x)
    pf, idx, w, ws = run_router(gpu, dl, L, hidden, t, stride)
    ref_idx, ref_w, ref_logits = O.prefill_router(L.router_dict(), x, t, d, k, stride=stride)
    logits = ws.download(np.float32, t * ne).reshape(t, ne)
    assert np.array_equal(logits.view(np.uint32), ref_logits.view(np.uint32)), "prefill logits differ in bits"
    got_idx, got_w = idx.download(np.uint32, t * k), w.download(np.uint16, t * k)
    assert np.array_equal(got_idx, ref_idx)
    assert np.max(np.abs(f16(got_w) - f16(ref_w))) <= 1e-3
    # the decode router on the same token gives the same bytes
    for tok in sorted({0, t // 2, t - 1}):
        one = gpu.dev(np.ascontiguousarray(x[tok * stride:tok * stride + d]))
        dl.moe.encode_router(dl.router_w, dl.router_s, dl.router_b, one, dl.eff_scale, dl.expert_scale, dl.logit_bias,
                             dl.out_idx, dl.out_w, ne, d, k)
        assert np.array_equal(dl.out_idx.download(np.uint32, k), got_idx[tok * k:(tok + 1) * k])
        assert np.array_equal(dl.out_w.download(np.uint16, k), got_w[tok * k:(tok + 1) * k])


@pytest.mark.parametrize("router_bits,ne,d,t", [
    (0, 19, 64, 18), (0, 37, 2048, 61), (0, 20, 2112, 40), (0, 18, 3072, 35), (0, 18, 4096, 33),  # the fp16 instances' edges
    (8, 21, 64, 19), (8, 36, 2048, 63), (8, 19, 2112, 30), (8, 18, 3072, 37), (8, 17, 4096, 41),   # the 8-bit ones
    (4, 33, 128, 17), (4, 50, 2048, 65), (4, 19, 2176, 29), (4, 18, 4096, 31),                     # the 4-bit ones
    (8, 256, 512, 3), (0, 64, 320, 8), (0, 64, 320, 9), (0, 256, 128, 700), (8, 100, 192, 1300),   # tokens a launch, a workgroup
    # on the matrix cores: part of a lane's chunks, whole ones only, ragged tokens and experts
    (0, 200, 64, 481), (0, 250, 512, 400), (0, 241, 2112, 390), (0, 250, 4096, 391), (8, 250, 64, 300), (8, 241, 1024, 273),
    (8, 256, 2304, 258), (8, 241, 4096, 272), (4, 249, 128, 270), (4, 256, 2048, 257), (4, 241, 2176, 273), (4, 241, 4096, 258),
    (4, 250, 512, 260), (4, 241, 576, 273), (4, 256, 1088, 257), (4, 249, 1600, 270)])  # (rows without chunks for the last blocks)
def test_prefill_router_instances_bit_exact(gpu, router_bits, ne, d, t):
    k = 4
    L = Layer(0x5EED0A00 + router_bits + d, d, 64, ne, k, router_bits=router_bits)
    L.logit_bias = S.f32_to_bf16_bits(L.tree.key("bias").normal(ne, std=0.01))
    dl = DeviceLayer(gpu, L, resident=[])
    x = token_rows(L, t, d)
    _, idx, _, ws = run_router(gpu, dl, L, gpu.dev(x), t, d)
    ref_idx, _, ref_logits = O.prefill_router(L.router_dict(), x, t, d, k, stride=d)
    logits = ws.download(np.float32, t * ne).reshape(t, ne)
    assert np.array_equal(logits.view(np.uint32), ref_logits.view(np.uint32))
    assert np.array_equal(idx.download(np.uint32, t * k), ref_idx)


@pytest.mark.parametrize("router_bits,ne,d,t", [(0, 241, 2112, 390), (8, 241, 1088, 273), (4, 241, 2176, 273)])
def test_prefill_router_takes_effective_scales_at_any_element(gpu, router_bits, ne, d, t):
    """Enough tokens for the matrix cores, whose kernel loads the scales in pieces of 16 bytes where they start at one: from the first,
    the second and the fourth element on the logits are the same."""
    L = Layer(0x5EED0D00 + router_bits, d, 64, ne, 4, router_bits=router_bits)
    L.eff_scale = S.f32_to_bf16_bits(L.tree.key("eff").uniform(0.5, 1.5, d))
    dl = DeviceLayer(gpu, L, resident=[])
    x = gpu.dev(token_rows(L, t, d))
    _, _, _, ws = run_router(gpu, dl, L, x, t, d)
    want = ws.download(np.uint32, t * ne)
    for ahead in (1, 2, 4):
        moved = gpu.dev(np.concatenate([np.zeros(ahead, np.uint16), L.eff_scale]))
        dl.eff_scale = moved.ptr + 2 * ahead
        _, _, _, ws = run_router(gpu, dl, L, x, t, d)
        assert np.array_equal(ws.download(np.uint32, t * ne), want), f"{ahead} elements on"


@pytest.mark.parametrize("values", ["infinite", "subnormal", "cancelling"])
@pytest.mark.parametrize("router_bits,ne,d,t", [(0, 241, 2112, 390), (8, 241, 1088, 273), (4, 241, 2176, 273), (4, 241, 576, 273)])
def test_prefill_router_on_the_matrix_cores_takes_any_values(gpu, router_bits, ne, d, t, values):
    """Rows that end inside a walk of chunks, on the matrix cores: an infinite effective scale, products and sums down to
    fp32's smallest subnormals, neighbours that cancel to their last bit."""
    L = Layer(0x5EED0B00 + router_bits, d, 64, ne, 4, router_bits=router_bits)
    rows = f16(token_rows(L, t, d)).reshape(t, d)
    rng = np.random.default_rng(9)
    eff = np.ones(d, np.float32)
    if values == "infinite":
        eff[0] = np.inf
        if router_bits:  # biases of the scales' sign: an infinite product keeps its sign through scale and bias
            L.router_b = L.router_b & np.uint16(0x7FFF)
    elif values == "subnormal":
        eff = np.exp2(rng.integers(-126, -99, d)).astype(np.float32)
        rows = rows * np.exp2(-(np.arange(t) % 24.0))[:, None]
    else:
        eff = np.repeat(np.exp2(rng.integers(-8, 9, d // 2)), 2).astype(np.float32)
        rows[:, 1::2] = -rows[:, ::2]
        if router_bits == 4:
            low = L.router_w & 0x0F
            L.router_w = low | (low ^ rng.integers(0, 2, low.shape).astype(np.uint8)) << 4
        else:
            L.router_w[:, 1::2] = L.router_w[:, ::2] ^ rng.integers(0, 2, L.router_w[:, ::2].shape).astype(L.router_w.dtype)
    L.eff_scale = S.f32_to_bf16_bits(eff)
    x = S.f32_to_f16_bits(rows.astype(np.float32)).reshape(-1)
    dl = DeviceLayer(gpu, L, resident=[])
    _, _, _, ws = run_router(gpu, dl, L, gpu.dev(x), t, d)
    logits = ws.download(np.float32, t * ne).reshape(t, ne)
    want = np.stack([O.router_logits(L.router_w, L.router_s, L.router_b, router_bits, x[i * d:(i + 1) * d], L.eff_scale, ne, d, meta=L.meta)
                     for i in range(t)])
    ordinary = ~np.isnan(want)
    assert np.array_equal(np.isnan(logits), ~ordinary)
    assert np.array_equal(logits[ordinary].view(np.uint32), want[ordinary].view(np.uint32))
    smallest = np.finfo(np.float32).smallest_normal
    assert {"infinite": np.isinf(want).any(), "subnormal": ((want != 0) & (np.abs(want) < smallest)).any(), "cancelling": True}[values]


@pytest.mark.parametrize("router_bits,ne,d,f,k,t,pad,bits", [
    (0, 64, 2048, 512, 8, 70, 0, 4),     # the fp16 logits kernel with four packed rows a wave forms the sums itself
    (0, 24, 2880, 384, 4, 21, 8, 8),     # the instance for longer rows; an odd token count, padded rows
    (0, 16, 192, 320, 3, 50, 24, 4),     # a row shorter than one wave load
    (8, 32, 512, 256, 4, 40, 0, 4),      # an affine router: the sums come from the pass of their own
    (0, 16, 512, 128, 2, 3, 0, 4)])      # a handful of tokens: the decode router's kernel, and the pass of their own
def test_router_with_group_sums_feeds_the_presummed_ffn(gpu, router_bits, ne, d, f, k, t, pad, bits):
    """shrike_hip_prefill_router_with_group_sums + shrike_hip_prefill_grouped_ffn_presummed against the two calls that
    each read `hidden` for themselves: the same logits, routes and weights, the same group sums at the head of the FFN's
    workspace, and the same partial rows, all bit for bit."""
    L = Layer(0x5EED0610 + router_bits + t, d, f, ne, k, bits=bits, router_bits=router_bits)
    L.logit_bias = S.f32_to_bf16_bits(L.tree.key("bias").normal(ne, std=0.01))
    dl = DeviceLayer(gpu, L)
    stride = d + pad
    x = token_rows(L, t, stride)
    hidden = gpu.dev(x)
    pf, idx, w, logits = run_router(gpu, dl, L, hidden, t, stride)
    routes = gpu.GroupedRoutesDevice(t * k, ne)
    pf.group_pairs(idx, w, t, k, ne, routes, residency=dl.pool.table)
    ws_bytes = pf.ffn_workspace_bytes(t, routes.max_row_tiles)
    ws, ws2 = gpu.empty(ws_bytes).fill(0xA5), gpu.empty(ws_bytes).fill(0x5A)
    partials, partials2 = (gpu.dev(np.full(t * k * d, 0xD4D0, np.uint16)) for _ in range(2))
    pf.encode_grouped_expert_gemms(dl.pool, dl.off, routes, hidden, stride, partials, ws, t, k)
    gpu.synchronize()
    # the fused pair, into buffers of its own
    idx2, w2 = gpu.empty(4 * t * k).fill(0xA5), gpu.empty(2 * t * k).fill(0xA5)
    logits2 = gpu.empty(pf.router_workspace_bytes(t, ne, d)).fill(0xA5)
    pf.encode_block(dl.router_w, dl.router_s, dl.router_b, hidden, dl.eff_scale, dl.expert_scale, dl.logit_bias,
                    idx2, w2, logits2, t, ne, d, k, stride, ffn_workspace=ws2)
    gpu.synchronize()
    assert np.array_equal(logits2.download(np.uint32, t * ne), logits.download(np.uint32, t * ne))
    assert np.array_equal(idx2.download(np.uint32, t * k), idx.download(np.uint32, t * k))
    assert np.array_equal(w2.download(np.uint16, t * k), w.download(np.uint16, t * k))
    sums = t * (d // 64)
    assert np.array_equal(ws2.download(np.uint32, sums), ws.download(np.uint32, sums)), "group sums differ from the FFN's own pass"
    pf.encode_grouped_expert_gemms(dl.pool, dl.off, routes, hidden, stride, partials2, ws2, t, k, presummed=True)
    gpu.synchronize()
    assert np.array_equal(partials2.download(np.uint16, t * k * d), partials.download(np.uint16, t * k * d))
    # what the entry point refuses
    lib = capi.load()
    assert lib.shrike_hip_prefill_router_with_group_sums(dl.moe.handle, None, dl.router_w.ptr, None, None, hidden.ptr, dl.eff_scale.ptr,
                                                         dl.expert_scale.ptr, dl.logit_bias.ptr, idx2.ptr, w2.ptr, logits2.ptr,
                                                         t, ne, d, k, stride, None) != 0
    assert "workspace" in capi.last_error()


def random_routes(seed, t, k, ne, skew=1.2):
    rng = np.random.default_rng(seed)
    p = 1.0 / np.arange(1, ne + 1) ** skew
    p = rng.permutation(p / p.sum())
    idx = np.concatenate([rng.choice(ne, size=k, replace=False, p=p) for _ in range(t)]).astype(np.uint32) if t else np.zeros(0, np.uint32)
    w = rng.integers(0, 0x3C00, size=t * k).astype(np.uint16)
    return idx, w


def expected_row_tiles(groups, cell_of):
    tiles = []
    for e, start, count in groups:
        for j in range(0, count, 64):
            tiles.append((cell_of(e), start + j, min(64, count - j), e))
    return tiles


@pytest.mark.parametrize("t,k,ne,mode", [(512, 8, 256, "plain"), (512, 8, 256, "keys"), (37, 3, 17, "plain"), (64, 4, 32, "residency"),
                                         (1, 8, 256, "plain"), (300, 2, 4, "keys"), (0, 8, 16, "plain"),
                                         (200, 1, 32, "plain"), (5000, 1, 7, "keys")])  # one expert a token: the token index is the pair index
def test_device_grouping_equals_host_grouping(gpu, t, k, ne, mode):
    idx, w = random_routes(t * 131 + k, t, k, ne)
    keys = None
    residency = None
    cell_of = lambda e: e
    if mode == "keys":
        order = np.random.default_rng(9).permutation(ne)[: max(1, ne // 2)].astype(np.uint32)
        keys = HL.expert_sort_keys(order, ne)
    if mode == "residency":
        words = np.array([H.residency_word(H.RESIDENT, 100 + e) if e % 3 else H.residency_word(H.LOADING if e % 2 else H.EMPTY, e)
                          for e in range(ne)], np.uint64)
        residency = gpu.dev(words)
        cell_of = lambda e: 100 + e if e % 3 else SENT
    routes = gpu.GroupedRoutesDevice(t * k, ne)
    pf = gpu.Prefill(gpu.MoE(64, 64, ne, min(k, 8)))
    pf.group_pairs(gpu.dev(idx) if t else None, gpu.dev(w) if t else None, t, k, ne, routes,
                   expert_sort_keys=None if keys is None else gpu.dev(keys), residency=residency)
    gpu.synchronize()
    got = routes.download()
    pairs = HL.make_token_expert_pairs(idx, w, t, k)
    host = HL.group_token_expert_pairs(pairs, t, k, ne, 16, keys)
    ref = H.group_token_expert_pairs(H.make_token_expert_pairs(idx, w, t, k), t, k, ne, 16, None if keys is None else keys.tolist())
    assert got["counts"].tolist() == ref.per_expert_counts == host.per_expert_counts.tolist()
    assert got["offsets"].tolist() == ref.per_expert_offsets == host.per_expert_offsets.tolist()
    assert [tuple(r) for r in got["sorted_pairs"].tolist()] == [p.as_tuple() for p in ref.sorted_pairs]
    assert [tuple(r) for r in got["row_tiles"].tolist()] == expected_row_tiles(ref.groups, cell_of)
    assert got["row_tile_count"] <= routes.max_row_tiles


@pytest.mark.parametrize("t,k,ne,mode", [(683, 3, 256, "plain"), (685, 3, 250, "residency"),  # the most pairs of one run, and four uneven ones
                                         (7001, 8, 64, "plain"), (18001, 8, 64, "keys")])     # ids without weights in LDS, and neither
def test_device_grouping_of_many_pairs(gpu, t, k, ne, mode):
    test_device_grouping_equals_host_grouping(gpu, t, k, ne, mode)


def check_pair_stagewise(L: Layer, blob, x_row, dev_act, got_row, what, act=O.ACT_SILU):
    """Stage by stage, so that each comparison holds one rounding: the activations against the
    oracle's, the partial row against the oracle's down projection of the device's own
    activations; then the whole chain in the reference's relative-error metric."""
    off = L.oracle_offsets()
    dev_act = np.ascontiguousarray(dev_act)
    assert_ffn_close(dev_act, O.moe_phase1([blob], off, x_row, L.d, L.f, L.bits, L.meta, act, L.additive), f"{what}: activations")
    one, zero = np.array([0x3C00], np.uint16), np.zeros(L.d, np.uint16)
    assert_ffn_close(got_row, O.moe_phase2([blob], off, dev_act, one, zero, L.d, L.f, L.bits, L.meta, L.additive),
                     f"{what}: partial row from the device's activations")
    whole = O.prefill_pair_partial(blob, off, x_row, L.d, L.f, L.bits, L.meta, act, L.additive)
    assert_rel_close(got_row, whole, f"{what}: whole chain")


class WorkspaceActs:
    """The pairs' fp16 activation rows as the grouped FFN left them in its workspace: row tile j keeps rows
    [64 j, 64 j + 64), a pair sits at its place in the sorted pairs."""

    def __init__(self, routes, ws, t, d, f):
        self.tables = routes.download()
        act_off = (t * (d // 64) * 4 + 255) & ~255
        rows = routes.max_row_tiles * 64
        self.act = ws.download(np.uint16, rows * f, offset=act_off).reshape(rows, f)
        self.pos = {(int(r[0]), int(r[2])): i for i, r in enumerate(self.tables["sorted_pairs"])}

    def row(self, tok, rank):
        at = self.pos[(tok, rank)]
        for j, (cell, start, rows, expert) in enumerate(self.tables["row_tiles"].tolist()):
            if start <= at < start + rows:
                return self.act[j * 64 + at - start]
        raise AssertionError("pair not covered by a row tile")


class PrefillCase:
    def __init__(self, gpu, L: Layer, t, stride_pad=0, idx=None, moe_kwargs=None, resident=None, scale=1.0):
        self.gpu, self.L, self.t = gpu, L, t
        self.dl = DeviceLayer(gpu, L, moe_kwargs=moe_kwargs, resident=resident)
        self.stride = L.d + stride_pad
        self.x = token_rows(L, t, self.stride)
        if scale != 1.0:
            self.x = S.f32_to_f16_bits(f16(self.x) * np.float32(scale))
        self.hidden = gpu.dev(self.x)
        self.pf = gpu.Prefill(self.dl.moe)
        if idx is None:
            idx, w = random_routes(t + L.ne, t, L.k, L.ne)
        else:
            w = np.random.default_rng(1).integers(0x3000, 0x3C00, size=t * L.k).astype(np.uint16)
        self.idx, self.w = idx, w
        self.routes = gpu.GroupedRoutesDevice(t * L.k, L.ne)
        self.d_idx, self.d_w = gpu.dev(idx), gpu.dev(w)
        self.pf.group_pairs(self.d_idx, self.d_w, t, L.k, L.ne, self.routes, residency=self.dl.pool.table)
        self.partials = gpu.dev(np.full(t * L.k * L.d, 0xD4D0, np.uint16))  # -77: rows nobody writes keep it
        self.ws = gpu.empty(self.pf.ffn_workspace_bytes(t, self.routes.max_row_tiles))

    def run(self):
        self.pf.encode_grouped_expert_gemms(self.dl.pool, self.dl.off, self.routes, self.hidden, self.stride, self.partials,
                                            self.ws, self.t, self.L.k)
        self.gpu.synchronize()
        return self.partials.download(np.uint16, self.t * self.L.k * self.L.d).reshape(self.t, self.L.k, self.L.d)

    def device_act(self, tok, rank):
        if not hasattr(self, "_acts"):
            self._acts = WorkspaceActs(self.routes, self.ws, self.t, self.L.d, self.L.f)
        return self._acts.row(tok, rank)

    def check_pair(self, got, tok, rank, what, act=O.ACT_SILU):
        L = self.L
        x = np.ascontiguousarray(self.x[tok * self.stride:tok * self.stride + L.d])
        check_pair_stagewise(L, L.blobs[int(self.idx[tok * L.k + rank])], x, self.device_act(tok, rank), got[tok, rank], what, act)


FFN_CASES = [
    # name, d, f, experts, k, tokens, bits, meta, stride pad
    ("small-int4", 512, 256, 16, 4, 40, 4, S.META_BF16, 0),
    ("small-int8-f16meta", 512, 256, 16, 4, 40, 8, S.META_F16, 8),
    ("q-shape-int4-f16meta", 2048, 512, 24, 8, 20, 4, S.META_F16, 0),
    ("q-shape-int8", 2048, 512, 12, 4, 12, 8, S.META_BF16, 0),
    ("long-experts-two-tiles", 256, 128, 3, 2, 110, 4, S.META_BF16, 0),
    ("ragged-k-192x320", 192, 320, 8, 3, 50, 4, S.META_F16, 0),
    ("kimi-shape-int8", 2304, 1024, 8, 2, 6, 8, S.META_BF16, 0),
]


@pytest.mark.parametrize("case", FFN_CASES, ids=[c[0] for c in FFN_CASES])
def test_grouped_ffn_against_oracle(gpu, case):
    name, d, f, ne, k, t, bits, meta, pad = case
    L = Layer(0x5EED0003, d, f, ne, k, bits=bits, meta=meta)
    pc = PrefillCase(gpu, L, t, stride_pad=pad)
    got = pc.run()
    rng = np.random.default_rng(4)
    sample = [(int(a), int(b)) for a, b in zip(rng.integers(0, t, 40), rng.integers(0, k, 40))] if t * k > 48 else \
        [(a, b) for a in range(t) for b in range(k)]
    for tok, rank in sample:
        pc.check_pair(got, tok, rank, f"{name} token {tok} rank {rank}")
    assert not np.any(np.all(got == 0xD4D0, axis=-1)), "a pair's partial row was left unwritten"


def _swept_ffn_cases():
    """Sixty chunks drawn once from a fixed seed: hidden and intermediate sizes any multiple of 64 up to 1,536 (column blocks
    that end inside a workgroup's 128 or 256 columns, k that ends inside a staged chunk of 256, group counts that are not
    multiples of four), 1 to 150 tokens over 2 to 20 experts (row tiles of one row, of 32, of 33, of 64 and more)."""
    rng = np.random.default_rng(0x5EEDFF)
    out = []
    for i in range(60):
        d, f = (int(64 * rng.integers(1, 25)) for _ in range(2))
        ne = int(rng.integers(2, 21))
        k = int(rng.integers(1, min(ne, 8) + 1))
        out.append((f"sweep-{i}-d{d}-f{f}", d, f, ne, k, int(rng.integers(1, 151)), int(rng.choice([4, 8])),
                    int(rng.choice([S.META_BF16, S.META_F16])), int(rng.choice([0, 8, 24]))))
    return out


@pytest.mark.parametrize("case", _swept_ffn_cases(), ids=[c[0] for c in _swept_ffn_cases()])
def test_grouped_ffn_shape_sweep(gpu, case):
    name, d, f, ne, k, t, bits, meta, pad = case
    L = Layer(0x5EED0300 + d + f, d, f, ne, k, bits=bits, meta=meta)
    pc = PrefillCase(gpu, L, t, stride_pad=pad)
    got = pc.run()
    rng = np.random.default_rng(5)
    sample = [(int(a), int(b)) for a, b in zip(rng.integers(0, t, 24), rng.integers(0, k, 24))] if t * k > 24 else \
        [(a, b) for a in range(t) for b in range(k)]
    for tok, rank in sample:
        pc.check_pair(got, tok, rank, f"{name} token {tok} rank {rank}")
    assert not np.any(np.all(got == 0xD4D0, axis=-1)), "a pair's partial row was left unwritten"


def check_pair_ranges(gpu, pc):
    """Ranges that start and end inside row tiles, one of a single pair and one to the chunk's end: their pairs' rows are the whole
    call's bytes, and no others are written."""
    t, d, k = pc.t, pc.L.d, pc.L.k
    want = pc.run()
    order = pc.routes.download()["sorted_pairs"].astype(int)  # token, expert, rank, weight
    at = order[:, 0] * k + order[:, 2]
    for lo, count in ((37, 203), (t * k - 90, 90), (130, 1)):
        pc.partials = gpu.dev(np.full(t * k * d, 0xD4D0, np.uint16))
        pc.pf.encode_streamed_batched(pc.dl.pool, pc.dl.off, pc.routes, pc.hidden, pc.stride, pc.partials, pc.ws, t, k, lo, count)
        gpu.synchronize()
        got = pc.partials.download(np.uint16, t * k * d).reshape(t * k, d)
        inside = np.zeros(t * k, bool)
        inside[at[lo:lo + count]] = True
        assert np.array_equal(got[inside], want.reshape(t * k, d)[inside]), f"pairs {lo} to {lo + count}"
        assert np.all(got[~inside] == 0xD4D0), f"pairs {lo} to {lo + count}: a row of another pair was written"


def row_scale(d, f):
    """Of rows so long that N(0, 1) inputs make outputs of 75: a partial row is then a sum of products that come to 4,000 to 5,000
    in magnitude, of which fp32 keeps 2^-24 = 3e-4 a step, and where it cancels, two orders of addition differ by more than the
    2e-3 that is stated for outputs of order 1. An eighth of the inputs gives those (gate, up and so their product: a 64th)."""
    return 0.125 if d >= 2048 and f >= 1152 else 1.0


# The cases name the shape that the FFN's products take, which ffn_rules.h chooses (test_ffn_rules.py asks it).
SHAPE_CASES = [  # d, f, experts, k, tokens, bits, meta, shape
    # k over the waves: one group and one stage in all, a quarter without any, 9 to 16 rows and two pieces of a row tile,
    # groups that no quarter shares evenly
    (64, 64, 3, 2, 20, 4, S.META_BF16, "split"), (128, 192, 2, 1, 45, 8, S.META_F16, "split"), (2880, 64, 4, 2, 50, 4, S.META_F16, "split"),
    # one row tile a workgroup: fewer than eight groups and more than sixty-four, both odd
    (192, 4160, 6, 2, 70, 4, S.META_BF16, "tile"), (192, 1088, 24, 4, 120, 8, S.META_F16, "deep"),
    # the same with more groups ahead: one group, two, and odd many
    (64, 4096, 9, 2, 12, 8, S.META_BF16, "deep"), (128, 4096, 9, 2, 70, 8, S.META_F16, "deep"), (4032, 1088, 40, 3, 33, 8, S.META_F16, "deep"),
    (960, 832, 24, 4, 300, 8, S.META_BF16, "deep"), (4032, 1152, 40, 3, 33, 4, S.META_F16, "deep"), (64, 5184, 9, 2, 70, 4, S.META_BF16, "deep"),
    # two row tiles of an expert a workgroup: 128 rows and what is left over, odd groups, column blocks that end inside it
    (128, 8192, 6, 4, 360, 4, S.META_BF16, "wide"), (576, 3008, 8, 4, 960, 4, S.META_F16, "wide"), (960, 832, 24, 4, 1050, 8, S.META_BF16, "wide"),
    (192, 1344, 24, 4, 700, 8, S.META_F16, "wide")]


@pytest.mark.parametrize("d,f,ne,k,t,bits,meta", [c[:-1] for c in SHAPE_CASES])
def test_grouped_ffn_shapes_of_a_workgroup(gpu, d, f, ne, k, t, bits, meta):
    L = Layer(0x5EED0400 + d + f, d, f, ne, k, bits=bits, meta=meta)
    pc = PrefillCase(gpu, L, t, stride_pad=8, resident=[e for e in range(ne) if e != 1], scale=row_scale(d, f))
    got = pc.run()
    here = pc.idx.reshape(t, k) != 1
    assert np.all(got[~here] == 0xD4D0), "an absent expert's row was written"
    assert not np.any(np.all(got[here] == 0xD4D0, axis=-1)), "a pair's partial row was left unwritten"
    order = np.argwhere(here)
    for tok, rank in order[np.random.default_rng(6).choice(len(order), min(len(order), 40), replace=False)]:
        pc.check_pair(got, int(tok), int(rank), f"token {tok} rank {rank}")


# Groups of 64 in k around the four that the loop takes at once and the places of each shape's rings, of both products; experts of
# up to 32 rows, up to 64 and, where two tiles are one workgroup's, more; more than 64 tiles, or too many workgroups, so that none
# is cut in two.
RING_CASES = [  # d, f, experts, tokens, bits, shape
    (448, 576, 70, 700, 4, "tile"), (512, 704, 70, 700, 4, "tile"), (832, 1408, 70, 700, 4, "tile"),
    (576, 1600, 70, 700, 4, "tile"), (704, 1536, 70, 700, 4, "tile"), (768, 1664, 70, 700, 4, "tile"),
    (448, 576, 70, 700, 8, "deep"), (512, 704, 70, 700, 8, "deep"), (832, 768, 70, 700, 8, "deep"), (448, 576, 70, 1000, 8, "deep"),
    (2816, 2304, 8, 450, 4, "deep"), (2624, 2496, 8, 450, 4, "deep"), (2688, 2432, 8, 450, 4, "deep"),
    (576, 4672, 8, 160, 4, "deep"), (448, 4800, 8, 160, 4, "deep"),
    (704, 1408, 70, 1000, 8, "wide"), (512, 1024, 20, 920, 8, "wide"), (832, 704, 20, 1200, 8, "wide"), (576, 960, 20, 920, 8, "wide"),
    (512, 4096, 30, 500, 4, "wide"), (832, 3136, 16, 480, 4, "wide"), (1472, 1600, 20, 1190, 4, "wide"), (640, 2880, 16, 620, 4, "wide")]


@pytest.mark.parametrize("d,f,ne,t,bits", [c[:-1] for c in RING_CASES])
def test_grouped_ffn_rings(gpu, d, f, ne, t, bits):
    L = Layer(0x5EED0700 + d + f, d, f, ne, 4, bits=bits, meta=S.META_F16 if f % 128 else S.META_BF16)
    pc = PrefillCase(gpu, L, t, scale=row_scale(d, f))
    got = pc.run()
    assert not np.any(np.all(got == 0xD4D0, axis=-1)), "a pair's partial row was left unwritten"
    for pair in np.random.default_rng(12).choice(t * 4, 40, replace=False):
        pc.check_pair(got, int(pair) // 4, int(pair) % 4, f"pair {pair}")


# Units of two groups, one in all and around the ring of three places; experts of up to 32 rows, up to 64 and more; enough workgroups
# for whole tiles, few enough tiles for their second halves to be workgroups of their own (the 12 experts). The experts in use are more
# than the memory-side cache holds, but for the last: the hint is then left out.
LINE_CASES = [  # d, f, experts, tokens, meta, experts that may be in use, whether the lines carry the hint
    (128, 4096, 220, 800, S.META_F16, 220, True), (256, 2176, 210, 900, S.META_BF16, 210, True), (384, 1152, 250, 1000, S.META_F16, 250, True),
    (512, 1024, 220, 1200, S.META_BF16, 220, True), (640, 768, 230, 1100, S.META_F16, 230, True), (768, 640, 230, 1100, S.META_BF16, 230, True),
    (1152, 896, 110, 600, S.META_F16, 110, True), (2304, 1024, 50, 250, S.META_BF16, 50, True), (2048, 4096, 12, 60, S.META_BF16, 12, True),
    (512, 1024, 190, 300, S.META_BF16, 9, False)]


class LineCase(PrefillCase):
    """Experts that together are more than the memory-side cache holds, sixteen of them made. `beside` is the pool whose cells hold
    the same blobs 16 bytes further on, where no row starts with a line: its codes come as half lines."""

    def __init__(self, gpu, d, f, ne, t, meta, in_use, hint, **layer_and_case):
        layer = {n: layer_and_case.pop(n) for n in ("additive_biases",) if n in layer_and_case}
        L = Layer(0x5EED0C00 + d + f, d, f, ne, 4, bits=8, meta=meta, distinct=min(ne, 16, max(3, (48 << 20) // (3 * d * f))), **layer)
        idx = random_routes(t + ne, t, 4, in_use, skew=0.7)[0]
        super().__init__(gpu, L, t, idx=idx, scale=row_scale(d, f), **layer_and_case)
        o = self.dl.off
        align = self.dl.pool.stride | o.gate_w_off | o.up_w_off | o.down_w_off
        for base in self.dl.pool.bases.contents.base:
            align |= base or 0
        assert ffn_rules().takes_lines(4 * t, ne, d, f, 8, align | d | f)
        rows = np.bincount(idx, minlength=ne)
        tiles = [min(64, n - at) for n in rows for at in range(0, n, 64)]  # the table's, in its order
        last = sum(n < 64 for n in tiles[:256])
        assert ffn_rules().past_the_cache(last, d, f, 8) == hint and max(rows) > 32

    def beside(self):
        L = self.L
        pool, off = self.gpu.ExpertPool(L.ne, L.stride + 16, L.ne), capi.ExpertOffsets()
        for name, _ in off._fields_:
            setattr(off, name, getattr(self.dl.off, name) + 16)
        for e, cell in self.dl.cell_of.items():
            pool.upload(cell, np.concatenate([np.zeros(16, np.uint8), L.blobs[e]]))
            pool.publish(e, cell, capi.RESIDENT)
        assert not ffn_rules().takes_lines(4 * self.t, L.ne, L.d, L.f, 8, off.gate_w_off)
        return pool, off

    def check(self, got, act=O.ACT_SILU):
        for pair in np.random.default_rng(13).choice(self.t * 4, 12, replace=False):
            self.check_pair(got, int(pair) // 4, int(pair) % 4, f"pair {pair}", act)


@pytest.mark.parametrize("d,f,ne,t,meta,in_use,hint", LINE_CASES)
def test_grouped_ffn_of_codes_past_the_caches(gpu, d, f, ne, t, meta, in_use, hint):
    """Codes as whole lines: the oracle's rows, and the bytes that the same experts give where their codes come as half lines."""
    pc = LineCase(gpu, d, f, ne, t, meta, in_use, hint, stride_pad=8)
    got = pc.run()
    pc.check(got)
    pc.dl.pool, pc.dl.off = pc.beside()
    pc.pf.group_pairs(pc.d_idx, pc.d_w, t, 4, ne, pc.routes, residency=pc.dl.pool.table)
    pc.partials = gpu.dev(np.full(t * 4 * d, 0xD4D0, np.uint16))
    assert np.array_equal(pc.run(), got)


@pytest.mark.parametrize("d,f,ne,t", [(1152, 896, 110, 600), (2048, 4096, 12, 60)])
def test_gpt_oss_epilogues_of_codes_past_the_caches(gpu, d, f, ne, t):
    pc = LineCase(gpu, d, f, ne, t, S.META_BF16, ne, True, additive_biases=True, moe_kwargs=dict(activation=capi.ACT_CLAMPED_SWIGLU, additive_biases=True))
    got = pc.run()
    assert not np.any(np.all(got == 0xD4D0, axis=-1)), "a pair's partial row was left unwritten"
    pc.check(got, O.ACT_CLAMPED_SWIGLU)


def test_codes_past_the_caches_of_absent_experts(gpu):
    absent = [0, 1, 17, 63, 108]
    pc = LineCase(gpu, 1152, 896, 110, 600, S.META_F16, 110, True, resident=[e for e in range(110) if e not in absent])
    got = pc.run()
    there = ~np.isin(pc.idx, absent).reshape(pc.t, 4)
    assert np.all(got[~there] == 0xD4D0), "an absent expert's row was written"
    assert not np.any(np.all(got[there] == 0xD4D0, axis=-1)), "a pair's partial row was left unwritten"
    for tok, rank in np.argwhere(there)[::131]:
        pc.check_pair(got, int(tok), int(rank), f"token {tok} rank {rank}")


@pytest.mark.parametrize("d,f,ne,t", [(384, 1152, 250, 1000), (2048, 4096, 12, 60)])
def test_pair_ranges_of_codes_past_the_caches_equal_the_whole_chunk(gpu, d, f, ne, t):
    check_pair_ranges(gpu, LineCase(gpu, d, f, ne, t, S.META_BF16, ne, True))


@pytest.mark.parametrize("d,f,bits,meta", [(320, 640, 4, S.META_BF16), (1088, 704, 8, S.META_F16)])
def test_grouped_ffn_of_few_larger_tiles(gpu, d, f, bits, meta):
    """Experts of 0, 1, 32, 33, 64 and more rows, few enough for a tile's rows past 32 to be a workgroup's of their own."""
    counts = [33, 64, 65, 96, 97, 32, 1, 0] + [20] * 32
    idx = np.random.default_rng(8).permutation(np.repeat(np.arange(40), counts)).astype(np.uint32)
    pc = PrefillCase(gpu, Layer(0x5EED0500 + d, d, f, 40, 1, bits=bits, meta=meta), len(idx), idx=idx)
    got = pc.run()
    assert not np.any(np.all(got == 0xD4D0, axis=-1)), "a pair's partial row was left unwritten"
    for e in range(6):  # an expert's pairs lie in token order: the first and last row of each part of a tile
        tokens = np.flatnonzero(idx == e)
        for r in sorted({r for r in (0, 31, 32, 63, 64, 95, 96, len(tokens) - 1) if r < len(tokens)}):
            pc.check_pair(got, int(tokens[r]), 0, f"expert {e} row {r}")


HOLE_CASES = [  # pairs of each expert, tiles left out of the table, d, f, bits, shape
    ([200, 330] + [30] * 22, [1, 6], 192, 896, 8, "deep"), ([4200, 200, 300, 100], [68], 192, 896, 8, "deep"),
    ([200, 330] + [170] * 22, [1, 6], 640, 896, 8, "wide"), ([4200, 200, 300, 100], [68], 640, 896, 8, "wide"),
    # an expert's first tile, its last, two neighbours and every second one; 4-bit codes
    ([700, 130, 260, 70, 500, 1] + [190] * 6, [0, 10, 15, 16, 22, 24, 26], 448, 2944, 4, "wide"),
    # over 64 tiles an XCD, experts that run from one XCD's into the next and over several 64s of records, in odd and even numbers
    ([9000, 64, 129, 65, 63] + [128, 1, 193, 33] * 40 + [12345, 100, 20, 6400], [70, 150, 151, 500], 128, 1408, 8, "wide")]


@pytest.mark.parametrize("counts,out,d,f,bits", [c[:-1] for c in HOLE_CASES], ids=[f"{c[5]}-{len(c[0])}-{c[4]}" for c in HOLE_CASES])
def test_grouped_ffn_takes_a_table_that_leaves_tiles_out(gpu, counts, out, d, f, bits):
    """Two row tiles a workgroup are two that continue each other, not any two neighbours of the table: tiles inside an expert's
    left out; an expert of more tiles than a wave reads at once."""
    ne = len(counts)
    idx = np.random.default_rng(10).permutation(np.repeat(np.arange(ne), counts)).astype(np.uint32)
    pc = PrefillCase(gpu, Layer(0x5EED0600, d, f, ne, 1, bits=bits, meta=S.META_BF16), len(idx), idx=idx)
    table = pc.routes.download()["row_tiles"]
    kept = np.delete(table, out, axis=0)
    pc.routes.row_tiles.upload(np.ascontiguousarray(kept))
    pc.routes.row_tile_count.upload(np.array([len(kept)], np.uint32))
    got = pc.run()[:, 0]
    pair_tokens = pc.routes.download()["sorted_pairs"][:, 0]
    for i, (_, start, rows, expert) in enumerate(table):
        tokens = pair_tokens[start:start + rows]
        written = ~np.all(got[tokens] == 0xD4D0, axis=-1)
        assert np.all(written == (i not in out)), f"tile {i} of expert {expert}: {written.sum()} of {rows} rows written"
        if i not in out and (i < 10 or 60 < i < 70 or min(abs(i - o) for o in out) <= 2):
            for tok in tokens[[0, -1]]:
                pc.check_pair(got[:, None], int(tok), 0, f"tile {i} token {tok}")


TABLE_CASES = [  # d, f, experts, tokens, bits, shape; up to 64 tiles, and more
    (192, 2048, 16, 40, 4, "tile"), (512, 512, 200, 60, 8, "deep")]


@pytest.mark.parametrize("d,f,ne,t,bits", [c[:-1] for c in TABLE_CASES])
def test_grouped_ffn_of_a_table_shorter_than_the_bound(gpu, d, f, ne, t, bits):
    """One bound and one workspace for several chunks: this chunk's table has room for its own tiles only, at the end of its memory."""
    k = 2
    L = Layer(0x5EED0900 + ne, d, f, ne, k, bits=bits)
    pc = PrefillCase(gpu, L, t)
    want = pc.run()
    records = pc.routes.row_tiles.download(np.uint32, 4 * pc.routes.max_row_tiles)
    memory = gpu.empty(1 << 21)
    table_at = memory.ptr + (1 << 21) - records.nbytes
    memory.upload(records.view(np.uint8), offset=(1 << 21) - records.nbytes)
    routes = capi.HipGroupedRoutes.from_buffer_copy(pc.routes.c)
    routes.row_tiles = table_at
    bound = 4 * pc.routes.max_row_tiles
    pc.routes.c = routes
    pc.partials = gpu.dev(np.full(t * k * d, 0xD4D0, np.uint16))
    pc.ws = gpu.empty(pc.pf.ffn_workspace_bytes(t, bound))
    pc.pf.encode_grouped_expert_gemms(pc.dl.pool, pc.dl.off, pc.routes, pc.hidden, pc.stride, pc.partials, pc.ws, t, k, max_row_tiles=bound)
    gpu.synchronize()
    assert np.array_equal(pc.partials.download(np.uint16, t * k * d).reshape(t, k, d), want)


CHUNK_CASES = [  # d, f, experts, bits, tokens and their shape
    (512, 4096, 12, 4, {90: "tile", 400: "tile", 2900: "wide"}), (512, 1024, 40, 8, {150: "deep", 1000: "deep", 2000: "deep", 3700: "wide"}),
    (512, 512, 12, 4, {13: "split", 40: "split"}), (512, 2048, 12, 4, {40: "split", 400: "tile"})]


@pytest.mark.parametrize("d,f,ne,bits,chunks", CHUNK_CASES)
def test_a_row_of_the_ffn_over_chunks_of_different_lengths(gpu, d, f, ne, bits, chunks):
    """The same bytes where in both chunks one wave sums all of k, or four waves a quarter each; else the end-to-end bound (the
    sums' rounding moves fp16 activations by their last place)."""
    first = min(chunks)
    L = Layer(0x5EED0800, d, f, ne, 1, bits=bits, meta=S.META_BF16)
    x = token_rows(L, max(chunks), d)
    idx = np.random.default_rng(11).integers(0, ne, max(chunks)).astype(np.uint32)
    rows = {}
    for t in chunks:
        pc = PrefillCase(gpu, L, t, idx=idx[:t])
        pc.hidden = gpu.dev(x[:t * d])
        rows[t] = pc.run()[:first, 0]
    for t in chunks:
        if (chunks[t] == "split") == (chunks[first] == "split"):
            assert np.array_equal(rows[t], rows[first]), f"{t} tokens against {first}"
        else:
            assert_rel_close(rows[t].reshape(-1), rows[first].reshape(-1), f"{t} tokens against {first}")


@pytest.mark.parametrize("d,last", [(384, 1), (768, 7)])  # the last group of a wave's share of k, which ends inside a chunk of four
def test_grouped_ffn_with_an_infinite_bias(gpu, d, last):
    """An infinite bias against a sum that is not zero is an infinite gate, whatever the group's place in a wave's share of k."""
    L = Layer(0x5EED0700 + d, d, 64, 2, 1, bits=4, meta=S.META_F16)
    for blob in L.blobs:
        at = L.off["gate_b"] + 2 * last
        blob[at:at + 2].view(np.uint16)[0] = 0x7C00
    t = 20
    pc = PrefillCase(gpu, L, t)
    x = pc.x.reshape(t, d)
    x[:, 64 * last:64 * last + 64] = 0
    for half in (0, 32):  # each half's sum needs both of its fp16 parts, of one sign
        x[:, 64 * last + half], x[:, 64 * last + half + 1] = 0x3C00, 0x0800  # 1 and 2^-13
    pc.hidden = gpu.dev(pc.x)
    pc.run()
    for tok in range(t):
        act = pc.device_act(tok, 0)
        want = O.moe_phase1([L.blobs[int(pc.idx[tok])]], L.oracle_offsets(), np.ascontiguousarray(x[tok]), d, 64, 4, S.META_F16, O.ACT_SILU, False)
        assert np.isinf(f16(want[:1]))[0] and act[0] == want.reshape(-1)[0], f"token {tok}: {f16(act[:1])} vs {f16(want.reshape(-1)[:1])}"
        assert_ffn_close(act[1:], want.reshape(-1)[1:], f"token {tok}")


def test_grouped_ffn_gpt_oss_epilogues(gpu):
    # additive biases + clamped SwiGLU at the gpt-oss shape (moe.metal:257-288), 45 groups per row
    d = f = 2880
    L = Layer(0x5EED0004, d, f, 3, 2, bits=4, additive_biases=True)
    pc = PrefillCase(gpu, L, 5, moe_kwargs=dict(activation=capi.ACT_CLAMPED_SWIGLU, additive_biases=True))
    got = pc.run()
    for tok in range(5):
        for rank in range(2):
            pc.check_pair(got, tok, rank, f"gpt-oss token {tok} rank {rank}", O.ACT_CLAMPED_SWIGLU)


EPILOGUE_CASES = [  # d, f, experts, tokens, bits, shape; the additive biases stand in each shape's own order of a tile's columns
    (2880, 2880, 8, 370, 4, "wide"), (960, 832, 24, 1050, 8, "wide"),
    (832, 1408, 70, 700, 4, "tile"), (2880, 2880, 8, 160, 4, "deep"), (832, 768, 70, 700, 8, "deep")]


@pytest.mark.parametrize("d,f,ne,t,bits", [c[:-1] for c in EPILOGUE_CASES])
def test_grouped_ffn_gpt_oss_epilogues_of_each_shape(gpu, d, f, ne, t, bits):
    L = Layer(0x5EED0A04, d, f, ne, 4, bits=bits, additive_biases=True)
    pc = PrefillCase(gpu, L, t, moe_kwargs=dict(activation=capi.ACT_CLAMPED_SWIGLU, additive_biases=True), scale=row_scale(d, f))
    got = pc.run()
    assert not np.any(np.all(got == 0xD4D0, axis=-1)), "a pair's partial row was left unwritten"
    for pair in np.random.default_rng(13).choice(t * 4, 24, replace=False):
        pc.check_pair(got, int(pair) // 4, int(pair) % 4, f"pair {pair}", O.ACT_CLAMPED_SWIGLU)


@pytest.mark.parametrize("d,f,ne,k,t,bits", [(512, 256, 6, 2, 70, 4), (320, 192, 5, 3, 21, 8)])
def test_grouped_ffn_gelu_tanh(gpu, d, f, ne, k, t, bits):
    # the GELU-tanh GLU of moe.metal:98-105 through the grouped kernels (prefill.metal:318-363): one- and two-tile
    # row tiles, both code widths
    L = Layer(0x5EED0009, d, f, ne, k, bits=bits, meta=S.META_F16)
    pc = PrefillCase(gpu, L, t, moe_kwargs=dict(activation=capi.ACT_GELU_TANH))
    got = pc.run()
    rng = np.random.default_rng(8)
    for tok, rank in {(int(a), int(b)) for a, b in zip(rng.integers(0, t, 30), rng.integers(0, k, 30))}:
        pc.check_pair(got, tok, rank, f"gelu token {tok} rank {rank}", O.ACT_GELU_TANH)
    # and it is not the SiLU result: the activation switch reached the kernel
    silu = PrefillCase(gpu, L, t).run()
    assert not np.array_equal(silu, got)


def test_grouped_ffn_skips_absent_experts(gpu):
    L = Layer(0x5EED0005, 256, 128, 8, 2, bits=4)
    pc = PrefillCase(gpu, L, 30, resident=[0, 1, 2, 4, 5, 7])
    got = pc.run()
    for tok in range(30):
        for rank in range(2):
            e = int(pc.idx[tok * 2 + rank])
            if e in (3, 6):
                assert np.all(got[tok, rank] == 0xD4D0)
            elif tok % 5 == 0:
                pc.check_pair(got, tok, rank, f"token {tok} rank {rank}")
            else:
                assert not np.all(got[tok, rank] == 0xD4D0)


def test_one_pair_expert_leaves_other_rows_alone(gpu):
    # PrefillGroupedRoutedMoETests+Execution.swift:657-763: a single 1-pair expert; the padded
    # rows of its tile must not leave the staging block
    L = Layer(0x5EED0006, 512, 512, 8, 1, bits=4)
    pc = PrefillCase(gpu, L, 1, idx=np.array([5], np.uint32))
    guard = pc.gpu.dev(np.full(64 * 512, 0xD4D0, np.uint16))
    got = pc.run()
    pc.check_pair(got, 0, 0, "single pair")
    assert np.all(guard.download(np.uint16, 64 * 512) == 0xD4D0)


@pytest.mark.parametrize("bits,tile_experts", [(4, 3), (8, 16), (4, 1)])
def test_streamed_batched_over_pair_ranges_equals_the_whole_chunk(gpu, bits, tile_experts):
    """encodeStreamedBatched: the chunk's routed tiles (pair ranges of groupTokenExpertPairs' tiles) one call
    each, against a residency table that holds the tile's experts only, give the partial rows of the one-pass
    grouped FFN byte for byte, each call writing its own pairs' rows and no others; then a range cut through
    an expert's rows."""
    d, f, ne, k, t = 256, 128, 12, 3, 90
    L = Layer(0x5EED0007 + bits, d, f, ne, k, bits=bits)
    whole = PrefillCase(gpu, L, t)
    want = whole.run()
    pc = PrefillCase(gpu, L, t)
    pairs = H.make_token_expert_pairs(pc.idx, pc.w, t, k)
    grouped = H.group_token_expert_pairs(pairs, t, k, ne, tile_expert_count=tile_experts)
    order = {(p.token, p.rank): i for i, p in enumerate(grouped.sorted_pairs)}
    cells = pc.dl.cell_of
    written = np.zeros((t, k), bool)
    for group_start, group_count, pair_start, pair_count in grouped.tiles:
        live = [g[0] for g in grouped.groups[group_start:group_start + group_count]]
        table = np.full(ne, capi.EMPTY << 32 | 0xFFFFFFFF, np.uint64)
        for e in live:
            table[e] = capi.RESIDENT << 32 | cells[e]
        batches = pc.pf.encode_streamed_batched(pc.dl.pool, pc.dl.off, pc.routes, pc.hidden, pc.stride, pc.partials, pc.ws,
                                                t, k, pair_start, pair_count, residency=gpu.dev(table))
        assert batches == -(-pair_count // 32)  # PrefillGroupedRoutedMoE.swift:864-921: microbatches of 32 pairs
        gpu.synchronize()
        got = pc.partials.download(np.uint16, t * k * d).reshape(t, k, d)
        for (tok, rank), at in order.items():
            if pair_start <= at < pair_start + pair_count:
                written[tok, rank] = True
        assert np.array_equal(got[written], want[written]), "a tile's rows differ from the one-pass result"
        assert np.all(got[~written] == 0xD4D0), "a call wrote rows of pairs outside its range"
    assert written.all()
    # a range that starts and ends inside experts' rows, against the grouping's own cells
    cut = PrefillCase(gpu, L, t)
    lo, count = 17, 101
    assert cut.pf.encode_streamed_batched(cut.dl.pool, cut.dl.off, cut.routes, cut.hidden, cut.stride, cut.partials, cut.ws,
                                          t, k, lo, count, pair_microbatch_rows=8) == 13
    gpu.synchronize()
    got = cut.partials.download(np.uint16, t * k * d).reshape(t, k, d)
    inside = np.zeros((t, k), bool)
    for (tok, rank), at in order.items():
        inside[tok, rank] = lo <= at < lo + count
    assert np.array_equal(got[inside], want[inside]) and np.all(got[~inside] == 0xD4D0)
    # nothing to do is not an error; a range past the chunk is
    assert cut.pf.encode_streamed_batched(cut.dl.pool, cut.dl.off, cut.routes, cut.hidden, cut.stride, cut.partials, cut.ws,
                                          t, k, 5, 0) == 0
    with pytest.raises(capi.ShrikeError):
        cut.pf.encode_streamed_batched(cut.dl.pool, cut.dl.off, cut.routes, cut.hidden, cut.stride, cut.partials, cut.ws,
                                       t, k, t * k - 3, 4)


RANGE_CASES = [  # d, f, experts, tokens, bits, shape
    (448, 576, 70, 700, 4, "tile"), (576, 4672, 8, 160, 4, "deep"), (448, 576, 70, 700, 8, "deep"), (640, 2880, 16, 620, 4, "wide"),
    (576, 960, 20, 920, 8, "wide")]


@pytest.mark.parametrize("d,f,ne,t,bits", [c[:-1] for c in RANGE_CASES])
def test_pair_ranges_of_each_shape_equal_the_whole_chunk(gpu, d, f, ne, t, bits):
    check_pair_ranges(gpu, PrefillCase(gpu, Layer(0x5EED0B00 + d, d, f, ne, 4, bits=bits), t, scale=row_scale(d, f)))


def test_reduce_and_residual_bit_exact(gpu):
    rng = np.random.default_rng(12)
    for t, k, d in ((7, 8, 2048), (33, 4, 2880), (1, 1, 64)):
        partials = S.f32_to_f16_bits(rng.standard_normal(t * k * d).astype(np.float32))
        weights = S.f32_to_f16_bits(rng.random(t * k).astype(np.float32))
        pf = gpu.Prefill(gpu.MoE(64, 64, 8, 1))
        h2 = gpu.empty(2 * t * d)
        pf.encode_reduce_token_major(gpu.dev(partials), gpu.dev(weights), h2, t, k, d)
        gpu.synchronize()
        ref = O.prefill_reduce(partials, weights, t, k, d)
        assert np.array_equal(h2.download(np.uint16, t * d), ref)
        hidden = S.f32_to_f16_bits(rng.standard_normal(t * d).astype(np.float32))
        dh = gpu.dev(hidden)
        pf.residual_add(dh, h2, t * d)
        gpu.synchronize()
        assert np.array_equal(dh.download(np.uint16, t * d), O.residual_add_f16(hidden.copy(), ref))


def test_prefill_layer_at_full_size_agrees_with_the_decode_kernels(gpu):
    """T = 512 tokens, 256 experts, top 8 at the 35B-A3B int4 shape with the Zipf(1.1) skew: the routes of all
    512 tokens equal the oracle's router bit for bit (logits, indices), the grouping is a permutation with the
    host function's tables, 24 sampled pairs' activation and partial rows are held to the oracle stage by stage,
    the reduced rows equal the oracle's reduce of the device's partial rows, and sampled tokens' h2 agree with
    the decode kernels' y for that token alone (no shared expert, residual 0)."""
    d, f, ne, k, t = 2048, 512, 256, 8, 512
    L = Layer(0x5EED0003, d, f, ne, k, bits=4, meta=S.META_F16)
    # Zipf skew through the logit bias operand, over a seeded permutation
    perm = np.argsort(L.tree.key("zipf.perm").next(ne))
    bias = np.zeros(ne, np.float32)
    bias[perm] = -1.1 * np.log(np.arange(ne) + 1.0)
    L.logit_bias = S.f32_to_bf16_bits(bias)
    dl = DeviceLayer(gpu, L)
    x = token_rows(L, t, d)
    hidden = gpu.dev(x)
    pf, idx, w, ws = run_router(gpu, dl, L, hidden, t, d)
    routes = gpu.GroupedRoutesDevice(t * k, ne)
    pf.group_pairs(idx, w, t, k, ne, routes, residency=dl.pool.table)
    partials = gpu.dev(np.full(t * k * d, 0xD4D0, np.uint16))
    work = gpu.empty(pf.ffn_workspace_bytes(t, routes.max_row_tiles))
    pf.encode_grouped_expert_gemms(dl.pool, dl.off, routes, hidden, d, partials, work, t, k)
    h2 = gpu.empty(2 * t * d)
    pf.encode_reduce_token_major(partials, w, h2, t, k, d)
    gpu.synchronize()
    h_idx, h_w = idx.download(np.uint32, t * k), w.download(np.uint16, t * k)
    # every token's routes against the oracle's router, bit for bit
    ref_idx, ref_w, ref_logits = O.prefill_router(L.router_dict(), x, t, d, k)
    assert np.array_equal(ws.download(np.float32, t * ne).view(np.uint32), ref_logits.reshape(-1).view(np.uint32))
    assert np.array_equal(h_idx, ref_idx), "a token's routing indices differ from the oracle's"
    assert np.max(np.abs(f16(h_w) - f16(ref_w))) <= 1e-3
    counts = np.bincount(h_idx, minlength=ne)
    assert counts.max() > 64 and np.count_nonzero(counts) < ne, "the skew should give long experts and leave some without a pair"
    got = routes.download()
    host = HL.group_token_expert_pairs(HL.make_token_expert_pairs(h_idx, h_w, t, k), t, k, ne)
    assert got["counts"].tolist() == host.per_expert_counts.tolist() and int(got["counts"].sum()) == t * k
    assert got["offsets"].tolist() == host.per_expert_offsets.tolist()
    assert np.array_equal(got["sorted_pairs"], host.sorted_pairs.view(np.uint32).reshape(-1, 4))
    out = h2.download(np.uint16, t * d).reshape(t, d)
    rows = partials.download(np.uint16, t * k * d).reshape(t, k, d)
    assert not np.any(np.all(rows.reshape(t * k, d) == 0xD4D0, axis=-1))
    # sampled pairs against the oracle, stage by stage: pairs of the longest expert (two MFMA row tiles, several row
    # tiles), of an expert with a single pair if the routes have one, and 20 drawn over the chunk
    acts = WorkspaceActs(routes, work, t, d, f)
    rng = np.random.default_rng(6)
    sample = {(int(a), int(b)) for a, b in zip(rng.integers(0, t, 20), rng.integers(0, k, 20))}
    by_expert = {}
    for i, e in enumerate(h_idx.tolist()):
        by_expert.setdefault(e, []).append((i // k, i % k))
    longest = by_expert[int(np.argmax(counts))]
    sample.update([longest[0], longest[len(longest) // 2], longest[-1]])
    sample.add(by_expert[min(by_expert, key=lambda e: len(by_expert[e]))][0])
    for tok, rank in sorted(sample):
        check_pair_stagewise(L, L.blobs[int(h_idx[tok * k + rank])], np.ascontiguousarray(x[tok * d:(tok + 1) * d]),
                             acts.row(tok, rank), rows[tok, rank], f"full-size chunk token {tok} rank {rank}")
    assert np.array_equal(out.reshape(-1), O.prefill_reduce(rows.reshape(-1), h_w, t, k, d)), "reduce differs from the oracle's"
    zero = gpu.dev(np.zeros(d, np.uint16))
    for tok in (0, 1, 77, 255, 256, 511):
        one = gpu.dev(np.ascontiguousarray(x[tok * d:(tok + 1) * d]))
        dl.moe.encode_router(dl.router_w, None, None, one, dl.eff_scale, dl.expert_scale, dl.logit_bias, dl.out_idx, dl.out_w, ne, d, k)
        assert np.array_equal(dl.out_idx.download(np.uint32, k), h_idx[tok * k:(tok + 1) * k])
        cells = np.array([dl.cell_of[int(e)] for e in h_idx[tok * k:(tok + 1) * k]], np.uint32)
        dl.moe.encode_spec_phase1(dl.pool, gpu.dev(cells), dl.off, one, dl.acts, d, f, k)
        hid = gpu.dev(np.zeros(d, np.uint16))
        dl.moe.encode_spec_phase2(dl.pool, gpu.dev(cells), dl.off, dl.acts, dl.out_w, zero, dl.y, hid, d, f, k)
        gpu.synchronize()
        # The decode kernel rounds the fp32 sum over the experts once; prefill rounds each of the
        # eight partial rows to fp16 first (as the reference does), so single elements of a
        # cancelling sum move by a few fp16 steps of the largest partial: compared in the
        # reference's relative-error metric.
        assert_rel_close(out[tok], dl.y.download(np.uint16, d), f"token {tok}: prefill h2 vs decode y", tol=2e-3)


@pytest.mark.parametrize("rows", [2047, 2048, 2049, 2051])
def test_scalar_gate_of_many_rows(gpu, rows):
    # four rows a workgroup from 2,048 on, the last ones short of four; rows of nine groups, one more than the half-waves
    d, stride = 576, 584
    L = Layer(0x5EED0009, d, 64, 4, 2)
    x = token_rows(L, rows, stride)
    row = S.affine_matrix(L.tree.key("shared.scalar_gate"), 1, d, 8, L.meta)
    gates = gpu.dev(np.full(rows + 1, 0xD4D0, np.uint16))
    pf = gpu.Prefill(DeviceLayer(gpu, L, resident=[]).moe)
    pf.encode_scalar_gate_rows(tuple(gpu.dev(a) for a in row), gpu.dev(x), stride, gates, rows, d)
    gpu.synchronize()
    got = gates.download(np.uint16, rows + 1)
    assert np.array_equal(got[:rows], O.shared_scalar_gate_rows(row, x, rows, d, x_stride=stride, meta=L.meta)) and got[rows] == 0xD4D0


@pytest.mark.parametrize("d,fs,bits,t,gated", [(2048, 512, 4, 20, False), (2048, 512, 4, 70, True), (2304, 1024, 8, 16, True),
                                              (192, 320, 4, 70, False), (128, 64, 8, 1, True)])
def test_shared_expert_for_a_token_block(gpu, d, fs, bits, t, gated):
    """The chunk's shared expert with ONE SCALAR GATE A TOKEN (RealForwardRunner.swift:4438-4456): the gate row's
    GEMV for every token (moe.metal:1154-1193) bit for bit against the oracle, then h1[t] = shared(x_t) * sigmoid(gate[t])
    against the oracle token by token; the two-launch form (ungated block, then sigmoid_scalar_mul_rows) gives the same."""
    L = Layer(0x5EED0007, d, 64, 4, 2, bits=bits, shared_f=fs, shared_bits=bits)
    dl = DeviceLayer(gpu, L, resident=[])
    pf = gpu.Prefill(dl.moe)
    stride = d + 8
    x = token_rows(L, t, stride)
    dx = gpu.dev(x)
    h1 = gpu.dev(np.full(t * d, 0xD4D0, np.uint16))
    gates = None
    d_gates = None
    if gated:
        gate_row = S.affine_matrix(L.tree.key("shared.scalar_gate"), 1, d, 8, L.meta)
        d_gates = gpu.empty(2 * t).fill(0xFF)
        pf.encode_scalar_gate_rows(tuple(gpu.dev(a) for a in gate_row), dx, stride, d_gates, t, d)
        gates = d_gates.download(np.uint16, t)
        want_gates = O.shared_scalar_gate_rows(gate_row, x, t, d, x_stride=stride, meta=L.meta)
        assert np.array_equal(gates, want_gates), "the per-row gate differs from the oracle in bits"
        assert t == 1 or len(set(gates.tolist())) > 1
    pf.encode_shared_expert(dl.shared["gate"], dl.shared["up"], dl.shared["down"], bits, dx, stride, h1, t, fs,
                            scalar_gate=d_gates)
    gpu.synchronize()
    got = h1.download(np.uint16, t * d).reshape(t, d)
    for tok in range(t):
        xt = np.ascontiguousarray(x[tok * stride:tok * stride + d])
        gate_bits = gates[tok:tok + 1].copy() if gated else None
        ref = O.shared_expert(L.shared["gate"], L.shared["up"], L.shared["down"], xt, d, fs, bits=bits, meta=L.meta,
                              scalar_gate_f16=gate_bits)
        # gate/up -> fp16 -> act -> fp16 -> down -> fp16 (-> gate -> fp16): whole chain, the reference's metric
        assert_rel_close(got[tok], ref, f"token {tok}", tol=2e-3 if gated else 1e-3)
        # and equal to the single-token operator on the same token
        if tok in (0, t - 1):
            one = gpu.empty(2 * d)
            dl.moe.encode_shared_expert(dl.shared["gate"], dl.shared["up"], dl.shared["down"], bits, gpu.dev(xt), dl.shared_scratch,
                                        one, d, fs, scalar_gate=gpu.dev(gate_bits) if gated else None)
            gpu.synchronize()
            assert_rel_close(got[tok], one.download(np.uint16, d), f"token {tok} vs the decode operator", tol=2e-3 if gated else 1e-3)
    if gated:
        # the reference's two kernels: the ungated block, then y[t, :] *= sigmoid(gate[t]) in place
        plain = gpu.dev(np.full(t * d, 0xD4D0, np.uint16))
        pf.encode_shared_expert(dl.shared["gate"], dl.shared["up"], dl.shared["down"], bits, dx, stride, plain, t, fs)
        ungated = plain.download(np.uint16, t * d)
        pf.encode_sigmoid_scalar_mul_rows(plain, d_gates, d, t)
        gpu.synchronize()
        assert np.array_equal(plain.download(np.uint16, t * d).reshape(t, d), got), "fused and two-launch gating differ"
        # the elementwise kernel against the oracle: the device's exp may differ from libm's in the last bit
        assert_ffn_close(plain.download(np.uint16, t * d), O.sigmoid_scalar_mul_rows(ungated.copy(), gates, d, t), "sigmoid rows")


@pytest.mark.parametrize("d,fs,bits,t,gated", [(128, 4032, 4, 290, True), (192, 4096, 8, 265, False)])
def test_shared_expert_for_many_rows(gpu, d, fs, bits, t, gated):
    # a row tile a workgroup: more than two pieces of k_ffn_split's for each of its workgroups
    test_shared_expert_for_a_token_block(gpu, d, fs, bits, t, gated)


@pytest.mark.parametrize("d,f,ne,k,t,bits,slots,slru", [
    (256, 128, 48, 4, 12, 8, 16, None), (256, 128, 48, 4, 12, 4, 8, 0.5),
    (2304, 1024, 256, 8, 16, 8, 64, None),  # config 5 as it is stated: Kimi-Linear shape, 16 sequences, 64 of 256 cells
])
def test_batched_decode_through_a_pool_smaller_than_the_expert_set(gpu, d, f, ne, k, t, bits, slots, slru):
    """Config 5: several sequences, one token each, through a pool smaller than the expert set; the experts
    stream from pinned host memory in passes. Routes are bit-exact, every partial row matches the
    oracle stage by stage, the statistics (and so the miss rate) equal the slot-cache restatement's over the
    same plans, and a second step hits the cache."""
    L = Layer(0x5EED0005, d, f, ne, k, bits=bits)
    dl = DeviceLayer(gpu, L, cells=slots, resident=[])
    dl.moe.stream = gpu.Stream()
    cache = HL.SlotCache(slots, ne, slru_share=slru)
    store = gpu.PinnedBuffer(ne * L.stride)
    for e in range(ne):
        store.array[e * L.stride:(e + 1) * L.stride] = L.blobs[e]
    layer = runners.BatchedDecodeLayer(dl.moe, dl.pool, cache, dl.off, store, L.stride, L.stride, t)
    x = token_rows(L, t, d)
    hidden = gpu.dev(x)
    router = dict(weights=dl.router_w, eff_scale=dl.eff_scale, expert_scale=dl.expert_scale, bias=dl.logit_bias)
    h2 = layer.run(router, hidden, t, d)
    dl.moe.stream.synchronize()
    ref_idx, ref_w, _ = O.prefill_router(L.router_dict(), x, t, d, k)
    idx, w = layer.idx.download(np.uint32, t * k), layer.w.download(np.uint16, t * k)
    assert np.array_equal(idx, ref_idx)
    used = len(set(idx.tolist()))
    assert layer.passes == -(-used // slots) and layer.passes >= 2
    partials = layer.partials.download(np.uint16, t * k * d).reshape(t, k, d)
    # every pair stage by stage (the passes share one grouping, so a pair's activation row stays where the pass that
    # served its expert left it)
    acts = WorkspaceActs(layer.routes, layer.ffn_ws, t, d, f)
    for tok in range(t):
        xt = np.ascontiguousarray(x[tok * d:(tok + 1) * d])
        for rank in range(k):
            check_pair_stagewise(L, L.blobs[int(idx[tok * k + rank])], xt, acts.row(tok, rank), partials[tok, rank],
                                 f"token {tok} rank {rank}")
    assert np.array_equal(h2.download(np.uint16, t * d), O.prefill_reduce(partials.reshape(-1), w, t, k, d))
    st = cache.statistics(L.stride)
    assert (st.plans, st.requested_experts, st.misses, st.hits) == (layer.passes, used, used, 0)
    assert st.bytes_read == used * L.stride and st.loading_slots == 0 and st.resident_slots == min(slots, used)
    # every device residency word equals the cache's own
    assert [dl.pool.entry(e) for e in range(ne)] == [cache.entry(e) for e in range(ne)]
    # a second step over the same tokens: the experts of the last pass are still resident
    before = cache.statistics().hits
    layer.run(router, hidden, t, d)
    dl.moe.stream.synchronize()
    assert cache.statistics().hits > before
    # the miss rate over both steps is the slot-cache restatement's over the same plans
    twin = H.SlotCache(slots, ne, slru_share=slru)
    for batch in layer.plan_log:
        twin.load(batch)
    st, ts = cache.statistics(L.stride), twin.stats
    assert (st.plans, st.requested_experts, st.hits, st.misses, st.evictions, st.reloads) == tuple(
        ts[n] for n in ("plans", "requested", "hits", "misses", "evictions", "reloads"))
    assert [cache.entry(e) for e in range(ne)] == list(twin.words)
    miss_rate = st.misses / st.requested_experts
    print(f"\n[config 5] d={d} f={f} E={ne} K={k} tokens={t} cells={slots}: {used} distinct experts a step, "
          f"{layer.passes} passes, miss rate over two steps {miss_rate:.3f}")
    assert 0.0 < miss_rate < 1.0
    again = layer.partials.download(np.uint16, t * k * d)
    assert np.array_equal(again, partials.reshape(-1))  # same bytes whatever cell an expert landed in


@pytest.mark.parametrize("d,rows", [(2048, 1), (2304, 1), (2880, 3), (64, 5), (4096, 2), (2048, 512)])
def test_residual_add_rmsnorm_bit_exact(gpu, d, rows):
    """The producer of the path's input (rmsnorm.metal:96-130) against the oracle: the updated hidden rows
    and the normalised rows bit for bit, with and without the residual add."""
    tree = S.SeedTree(0x5EED0052)
    eps = 1e-6
    hidden = S.activations_f16(tree, "hidden", rows * d)
    delta = S.f32_to_f16_bits(tree.key("delta").normal(rows * d, std=0.5))
    weight = S.f32_to_bf16_bits(tree.key("weight").uniform(0.5, 1.5, d))
    for with_delta in (True, False):
        d_hidden, d_delta, d_weight, d_out = gpu.dev(hidden), gpu.dev(delta), gpu.dev(weight), gpu.empty(2 * rows * d)
        gpu.residual_add_rmsnorm_bf16w(d_hidden, d_delta if with_delta else None, d_weight, d_out, d, eps, rows)
        got_hidden, got_out = d_hidden.download(np.uint16, rows * d), d_out.download(np.uint16, rows * d)
        for r in range(rows if rows <= 8 else 4):
            h = hidden[r * d:(r + 1) * d].copy()
            want = O.residual_add_rmsnorm_bf16w(h, delta[r * d:(r + 1) * d] if with_delta else None, weight, eps)
            assert np.array_equal(got_hidden[r * d:(r + 1) * d], h)
            assert np.array_equal(got_out[r * d:(r + 1) * d], want), f"row {r} of d={d}"
    for bad_d in (20, 8192):  # not a multiple of 8; past the kernels' hidden-size ceiling
        with pytest.raises(capi.ShrikeError, match="multiple of 8"):
            gpu.residual_add_rmsnorm_bf16w(d_hidden, None, d_weight, d_out, bad_d, eps)
