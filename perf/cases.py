"""The work that a user of the library has it do, as cases to time: a MoE layer's decode step for one sequence and for
several, a prefill chunk from a few tokens to thousands, a step whose experts stream through a pool smaller than the
expert set, and the experts a host keeps in its own memory.

Shapes are those of the benchmark's five configurations (bench.py) and, for drawn cases, generic ones
inside the operators' documented limits. Weights follow the benchmark's definition: uniform codes, scales |N(0, 0.02)|
(a sixteenth of that at 8 bits), biases minus half the code range times the scale, router rows N(0, 0.02), activations
N(0, 1) in fp16; `skew` is the exponent of a Zipf skew over the experts, injected through the router's logit bias.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from shrike_amd import capi, host, synth
from shrike_amd import runtime as rt

GROUP = 64
Q35B = dict(d=2048, f=512, experts=256, top_k=8)      # 35B-A3B: configurations 1, 2 and 3
GPTOSS = dict(d=2880, f=2880, experts=32, top_k=4)    # gpt-oss-20B: configuration 4
KIMI = dict(d=2304, f=1024, experts=256, top_k=8)     # Kimi-Linear-48B: configuration 5
LARGEST_FLOPS = 2048 * 4 * 6 * 2880 * 2880            # no drawn case multiplies more than the largest listed one


def _case(kind, shape, **more):
    case = dict(kind=kind, bits=4, meta="f16", router_bits=0, shared_f=0, gated=False, act="silu", expert_biases=False,
                sigmoid=False, skew=0.0, tokens=1, layers=1)
    case.update(shape)
    case.update(more)
    return case


def listed():
    return [
        # the smallest call: one token through one layer of a small model, a call at a time (latency, launches, host path)
        dict(_case("decode", dict(d=512, f=256, experts=32, top_k=4), meta="bf16", shared_f=256), name="decode_small_int4"),
        # configuration 2: one token of the 35B-A3B shape through a run of layers, one fused call a layer
        dict(_case("decode", Q35B, shared_f=512, layers=8), name="decode_q35b_int4"),
        # one token of a gpt-oss-shape model at 8 bits: additive biases, clamped SwiGLU, rows of 2,880
        dict(_case("decode", GPTOSS, bits=8, meta="bf16", act="clamped", expert_biases=True, layers=4), name="decode_gptoss_int8"),
        # configuration 4: four sequences, one token each
        dict(_case("batch", GPTOSS, tokens=4, act="clamped", expert_biases=True, layers=4), name="batch4_gptoss_int4"),
        # configuration 5 with every expert resident: sixteen sequences at 8 bits, sigmoid scores, a shared expert
        dict(_case("batch", KIMI, bits=8, meta="bf16", tokens=16, shared_f=1024, sigmoid=True, router_bits=8), name="batch16_kimi_int8"),
        # a short prompt, or the ragged last chunk of a longer one: an odd handful of rows over many experts
        dict(_case("prefill", Q35B, tokens=37, shared_f=512, gated=True, skew=1.1), name="prefill_q35b_int4_t37"),
        # configuration 3: the 512-token chunk, with the model's shared expert and its scalar gate
        dict(_case("prefill", Q35B, tokens=512, shared_f=512, gated=True, skew=1.1), name="prefill_q35b_int4_t512"),
        # a long prompt in one chunk, experts evenly loaded
        dict(_case("prefill", Q35B, meta="bf16", tokens=4096, shared_f=512, gated=True), name="prefill_q35b_int4_t4096"),
        # 8-bit experts and an affine 8-bit router over a ragged chunk
        dict(_case("prefill", KIMI, bits=8, meta="bf16", tokens=1000, shared_f=1024, sigmoid=True, router_bits=8), name="prefill_kimi_int8_t1000"),
        # the largest products: gpt-oss rows and epilogues, many rows an expert
        dict(_case("prefill", GPTOSS, meta="bf16", tokens=2048, act="clamped", expert_biases=True), name="prefill_gptoss_int4_t2048"),
        # a step under a memory budget: the routed experts pass through a pool that holds a quarter of them
        dict(_case("streamed", Q35B, tokens=8, cells=32), name="streamed_q35b_int4_t8"),
        # configuration 1: the experts a host keeps in CPU memory, one token's eight on one core
        dict(_case("cpu", dict(d=2048, f=512, experts=8, top_k=8), meta="bf16"), name="cpu_experts_q35b_int4"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "batch", "prefill", "prefill", "prefill", "prefill", "streamed", "cpu"])
    if kind not in ("streamed", "cpu") and rng.random() < 0.4:
        shape = dict(rng.choice([Q35B, GPTOSS, KIMI]))
    else:
        shape = dict(d=GROUP * rng.randint(8, 48), f=GROUP * rng.randint(3, 32), experts=rng.choice([16, 48, 64, 100, 128, 200, 256]))
        shape["top_k"] = rng.randint(2, 8)
    d, f, k = shape["d"], shape["f"], shape["top_k"]
    bits, meta = rng.choice([4, 4, 8]), rng.choice(["f16", "bf16"])
    if kind == "cpu":
        k = max(1, min(k, 8 * 2048 * 512 // (d * f)))
        return _case("cpu", dict(d=d, f=f, experts=k, top_k=k), meta="bf16")
    if kind == "streamed":  # no more bytes over the link than the listed case may need
        most = max(1, min(12, 8 * 8 * 2048 * 512 // (k * d * f)))
        return _case("streamed", shape, meta=meta, tokens=rng.randint(1, most), cells=max(k, shape["experts"] // rng.choice([4, 8])))
    biases = rng.random() < 0.3
    more = dict(bits=bits, meta=meta, router_bits=rng.choice([0, 0, 8]), act="clamped" if biases else "silu", expert_biases=biases,
                sigmoid=rng.random() < 0.3, shared_f=0 if biases else rng.choice([0, f]))
    if more["shared_f"] > 2048:
        more["shared_f"] = 0
    if kind == "decode":
        return _case("decode", shape, layers=rng.randint(1, 4), **more)
    if kind == "batch":
        return _case("batch", shape, tokens=rng.randint(2, 16), layers=rng.randint(1, 2), **more)
    most = min(4096, LARGEST_FLOPS // ((k * f + more["shared_f"]) * 6 * d))
    more["gated"] = more["shared_f"] > 0 and rng.random() < 0.5
    return _case("prefill", shape, tokens=_log_int(rng, 5, most), skew=rng.choice([0.0, 1.1]), **more)


# ---------------------------------------------------------------------------------------------- inputs

def _meta16(v, meta):
    """fp32 -> the 16-bit type of scales and biases, as raw int16 words."""
    return v.to(torch.float16 if meta == "f16" else torch.bfloat16).view(torch.int16)


def _bf16(v):
    return v.to(torch.bfloat16).contiguous()


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=g.device) * std


def _codes(g, count):
    """`count` uniform random bytes (count a multiple of 8)."""
    return torch.randint(-2**63, 2**63 - 1, (count // 8,), dtype=torch.int64, generator=g, device=g.device).view(torch.uint8)


def _scales_and_biases(g, rows, n, bits, meta, lead=()):
    scale = _normal(g, *lead, rows * (n // GROUP), std=0.02 if bits == 4 else 0.02 / 16).abs_()
    s = _meta16(scale, meta)
    back = s.view(torch.float16 if meta == "f16" else torch.bfloat16).float()
    return s, _meta16(back * -(8.0 if bits == 4 else 128.0), meta)


def _projection(g, rows, n, bits, meta):
    s, b = _scales_and_biases(g, rows, n, bits, meta)
    return _codes(g, rows * n * bits // 8), s, b


def _expert_blobs(g, c, count, row_bytes):
    """`count` packed expert blobs, one every `row_bytes` bytes."""
    d, f, bits, meta = c["d"], c["f"], c["bits"], c["meta"]
    off, _ = synth.expert_offsets(d, f, bits, c["expert_biases"])
    blobs = _codes(g, count * row_bytes).view(count, row_bytes)

    def put(at, words):
        raw = words.contiguous().view(torch.uint8).view(count, -1)
        blobs[:, at:at + raw.shape[1]] = raw
    for name, rows, n in (("gate", f, d), ("up", f, d), ("down", d, f)):
        s, b = _scales_and_biases(g, rows, n, bits, meta, (count,))
        put(off[name + "_s"], s)
        put(off[name + "_b"], b)
    if c["expert_biases"]:
        for name, n in (("gate_ab", f), ("up_ab", f), ("down_ab", d)):
            put(off[name], _bf16(_normal(g, count, n, std=0.1)).view(torch.int16))
    return blobs


def _pool(g, c):
    """A pool that holds every expert of one layer, expert e in cell e."""
    _, stride = rt.expert_offsets(c["d"], c["f"], c["bits"], c["expert_biases"])
    pool = rt.ExpertPool(c["experts"], stride, c["experts"])
    blobs = _expert_blobs(g, c, c["experts"], pool.stride)
    capi.check(capi.load().shrike_hip_memcpy_d2d(pool.cell_ptr(0), blobs.data_ptr(), blobs.numel()), "memcpy_d2d")
    for e in range(c["experts"]):
        pool.publish(e, e, capi.RESIDENT)
    rt.synchronize()  # the blobs go back to torch
    return pool


def _router(g, c):
    d, e = c["d"], c["experts"]
    bias = torch.zeros(e, device=g.device)
    if c["skew"]:
        rank = torch.randperm(e, generator=g, device=g.device)
        bias[rank] = -c["skew"] * torch.log(torch.arange(1, e + 1, device=g.device, dtype=torch.float32))
    r = dict(effective_scale=_bf16(torch.ones(d, device=g.device)), per_expert_scale=_bf16(torch.ones(e, device=g.device)),
             logit_bias=_bf16(bias), scales=None, biases=None)
    if c["router_bits"] == 0:
        r["weights"] = _normal(g, e, d, std=0.02).to(torch.float16).contiguous()
    else:  # group-affine rows of the same spread: codes uniform over 256 levels
        s = _meta16((_normal(g, e * (d // GROUP), std=0.0002).abs_() + 0.0001), c["meta"])
        back = s.view(torch.float16 if c["meta"] == "f16" else torch.bfloat16).float()
        r["weights"], r["scales"], r["biases"] = _codes(g, e * d * c["router_bits"] // 8), s, _meta16(back * -127.5, c["meta"])
    return r


def _at(t):
    return None if t is None else t.data_ptr()


def _moe(c):
    act = {"silu": capi.ACT_SILU, "clamped": capi.ACT_CLAMPED_SWIGLU}[c["act"]]
    return rt.MoE(c["d"], c["f"], c["experts"], c["top_k"], routed_bits=c["bits"], router_bits=c["router_bits"],
                  meta=capi.META_F16 if c["meta"] == "f16" else capi.META_BF16, activation=act,
                  additive_biases=c["expert_biases"], sigmoid=c["sigmoid"], scaling=2.5 if c["sigmoid"] else 1.0)


def _shared(g, c):
    d, fs = c["d"], c["shared_f"]
    if not fs:
        return None
    return [_projection(g, rows, n, c["bits"], c["meta"]) for rows, n in ((fs, d), (fs, d), (d, fs))]


def _ptrs(projection):
    return tuple(t.data_ptr() for t in projection)


def _decode_layer(g, c, shared_scratch):
    """One layer's weights, inputs and argument block for the fused decode call (one token, or a batch of them)."""
    d, t, k = c["d"], c["tokens"], c["top_k"]
    new = lambda n, dtype: torch.zeros(n, dtype=dtype, device=g.device)  # noqa: E731
    lay = dict(pool=_pool(g, c), router=_router(g, c), shared=_shared(g, c),
               x=_normal(g, t, d).to(torch.float16), hidden=_normal(g, t, d).to(torch.float16),
               y=new((t, d), torch.float16), idx=new((t, k), torch.int32), w=new((t, k), torch.float16), h1=new((t, d), torch.float16))
    off, _ = rt.expert_offsets(d, c["f"], c["bits"], c["expert_biases"])
    r, p, s = lay["router"], lay["pool"], shared_scratch
    a = capi.DecodeLayerArgs()
    a.router_weights, a.router_scales, a.router_biases = _at(r["weights"]), _at(r["scales"]), _at(r["biases"])
    a.effective_scale, a.per_expert_scale, a.logit_bias = _at(r["effective_scale"]), _at(r["per_expert_scale"]), _at(r["logit_bias"])
    a.pool, a.pool_slot_stride, a.residency, a.offsets = p.bases, p.stride, p.table, off
    a.x, a.hidden, a.y = _at(lay["x"]), _at(lay["hidden"]), _at(lay["y"])
    a.out_indices, a.out_weights = _at(lay["idx"]), _at(lay["w"])
    a.resolved_slots, a.acts = _at(s["resolved"]), _at(s["acts"])
    if c["kind"] == "decode":
        a.hit_count, a.hit_positions, a.miss_count = _at(s["hit_count"]), _at(s["hit_positions"]), _at(s["miss_count"])
        a.miss_positions, a.miss_experts = _at(s["miss_positions"]), _at(s["miss_experts"])
        if lay["shared"]:
            for name, proj in zip(("gate", "up", "down"), lay["shared"]):
                setattr(a, "shared_" + name, capi.Projection(*_ptrs(proj)))
            a.shared_bits, a.shared_f, a.shared_scratch, a.h1 = c["bits"], c["shared_f"], _at(s["shared"]), _at(lay["h1"])
    lay["args"] = a
    return lay


def _prepare_decode(g, c):
    d, f, t, k = c["d"], c["f"], c["tokens"], c["top_k"]
    new = lambda n, dtype: torch.zeros(n, dtype=dtype, device=g.device)  # noqa: E731
    scratch = {n: new(8 * t, torch.int32) for n in ("resolved", "hit_count", "hit_positions", "miss_count", "miss_positions", "miss_experts")}
    scratch["acts"], scratch["shared"] = new(t * k * f, torch.float16), new(2 * max(1, c["shared_f"]), torch.float16)
    st = dict(c=c, moe=_moe(c), scratch=scratch, layers=[_decode_layer(g, c, scratch) for _ in range(c["layers"])])
    if c["kind"] == "batch":
        st["pf"] = rt.Prefill(st["moe"])
        if c["shared_f"]:
            st["shared_ws"] = rt.empty(capi.load().shrike_hip_prefill_shared_expert_workspace_bytes(t, d, c["shared_f"]))
    return st


def _prepare_prefill(g, c):
    d, t, k, e = c["d"], c["tokens"], c["top_k"], c["experts"]
    moe = _moe(c)
    pf = rt.Prefill(moe)
    new = lambda n, dtype: torch.zeros(n, dtype=dtype, device=g.device)  # noqa: E731
    st = dict(c=c, moe=moe, pf=pf, router=_router(g, c), shared=_shared(g, c), hidden=_normal(g, t, d).to(torch.float16),
              idx=new((t, k), torch.int32), w=new((t, k), torch.float16), y=new((t, d), torch.float16), h1=new((t, d), torch.float16),
              gate=new(t, torch.float16), partials=new((t * k, d), torch.float16))
    st["off"], st["stride"] = rt.expert_offsets(d, c["f"], c["bits"], c["expert_biases"])
    st["routes"] = rt.GroupedRoutesDevice(t * k, e)
    st["router_ws"] = rt.empty(pf.router_workspace_bytes(t, e, d))
    st["ffn_ws"] = rt.empty(pf.ffn_workspace_bytes(t, st["routes"].max_row_tiles))
    if c["shared_f"]:
        st["shared_ws"] = rt.empty(capi.load().shrike_hip_prefill_shared_expert_workspace_bytes(t, d, c["shared_f"]))
    if c["gated"]:
        st["gate_row"] = _projection(g, 1, d, 8, c["meta"])
    if c["kind"] == "prefill":
        st["pool"] = _pool(g, c)
    else:  # the experts live in pinned host memory; the pool and its slot cache hold some of them
        store = rt.PinnedBuffer(e * st["stride"])
        blobs = _expert_blobs(g, c, e, st["stride"])
        capi.check(capi.load().shrike_hip_memcpy_d2h(store.ptr, blobs.data_ptr(), blobs.numel()), "memcpy_d2h")
        st.update(store=store, pool=rt.ExpertPool(c["cells"], st["stride"], e), cache=host.SlotCache(c["cells"], e), table=rt.empty(8 * e))
    return st


def _prepare_cpu(seed, c):
    d, f = c["d"], c["f"]
    g = torch.Generator("cpu").manual_seed(seed)
    off, stride = rt.expert_offsets(d, f, 4)
    return dict(c=c, off=off, blobs=[b for b in _expert_blobs(g, c, c["experts"], stride).numpy()], x=_normal(g, d).numpy(),
                weights=torch.softmax(_normal(g, c["experts"]), 0).tolist(), scratch=np.empty(2 * f + d, np.float32),
                out=np.zeros(d, np.float32))


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "cpu":
        return _prepare_cpu(seed, c)
    g = torch.Generator("cuda").manual_seed(seed)
    st = _prepare_decode(g, c) if c["kind"] in ("decode", "batch") else _prepare_prefill(g, c)
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------------------------------------- one pass

def _run_decode(st):
    c, moe = st["c"], st["moe"]
    for lay in st["layers"]:
        if c["kind"] == "decode":
            moe.encode_decode_layer(lay["args"])
            continue
        moe.encode_decode_layer_batch(lay["args"], c["tokens"], c["d"])
        if c["shared_f"]:
            gate, up, down = (_ptrs(p) for p in lay["shared"])
            st["pf"].encode_shared_expert(gate, up, down, c["bits"], _at(lay["x"]), c["d"], _at(lay["h1"]), c["tokens"], c["shared_f"],
                                          workspace=st["shared_ws"])
            st["pf"].residual_add(_at(lay["hidden"]), _at(lay["h1"]), c["tokens"] * c["d"])
    return [[lay[n] for n in ("idx", "w", "y", "hidden")] for lay in st["layers"]]


def _run_prefill(st):
    c, pf, r = st["c"], st["pf"], st["router"]
    d, t, k, e = c["d"], c["tokens"], c["top_k"], c["experts"]
    x, idx, w = _at(st["hidden"]), _at(st["idx"]), _at(st["w"])
    pf.encode_block(_at(r["weights"]), _at(r["scales"]), _at(r["biases"]), x, _at(r["effective_scale"]), _at(r["per_expert_scale"]),
                    _at(r["logit_bias"]), idx, w, st["router_ws"], t, e, d, k, d, ffn_workspace=st["ffn_ws"])
    pf.group_pairs(idx, w, t, k, e, st["routes"], residency=st["pool"].table)
    pf.encode_grouped_expert_gemms(st["pool"], st["off"], st["routes"], x, d, _at(st["partials"]), st["ffn_ws"], t, k, presummed=True)
    pf.encode_reduce_token_major(_at(st["partials"]), w, _at(st["y"]), t, k, d)
    if c["shared_f"]:
        if c["gated"]:
            pf.encode_scalar_gate_rows(_ptrs(st["gate_row"]), x, d, _at(st["gate"]), t, d)
        gate, up, down = (_ptrs(p) for p in st["shared"])
        pf.encode_shared_expert(gate, up, down, c["bits"], x, d, _at(st["h1"]), t, c["shared_f"], workspace=st["shared_ws"],
                                scalar_gate=_at(st["gate"]) if c["gated"] else None)
        pf.residual_add(_at(st["y"]), _at(st["h1"]), t * d)
    return [st["idx"], st["w"], st["y"]]


def _run_streamed(st):
    """The runner's loop: routes back to the host, then passes of as many experts as the pool takes, residents first."""
    c, pf, r, cache, pool = st["c"], st["pf"], st["router"], st["cache"], st["pool"]
    d, t, k, e = c["d"], c["tokens"], c["top_k"], c["experts"]
    x, idx, w = _at(st["hidden"]), _at(st["idx"]), _at(st["w"])
    pf.encode_block(_at(r["weights"]), _at(r["scales"]), _at(r["biases"]), x, _at(r["effective_scale"]), _at(r["per_expert_scale"]),
                    _at(r["logit_bias"]), idx, w, st["router_ws"], t, e, d, k, d)
    ids = st["idx"].cpu().numpy().reshape(-1).tolist()  # the router's readback
    rows, last = {}, {}
    for i, expert in enumerate(ids):
        rows[expert] = rows.get(expert, 0) + 1
        last[expert] = i // k
    resident = np.zeros(e, np.uint8)
    resident[cache.resident_experts()] = 1
    todo = host.resident_first_balanced(rows, last, resident, cache.slot_count, min(16, cache.slot_count))
    while todo:
        experts, todo = todo[:cache.slot_count], todo[cache.slot_count:]
        plan = cache.plan(experts)
        pool.execute_plan(cache, plan, st["store"], st["stride"], st["stride"])
        table = np.full(e, (capi.EMPTY << 32) | capi.SENTINEL, np.uint64)  # this pass's experts alone count as resident
        for expert in experts:
            table[expert] = cache.entry(expert)
        st["table"].upload(table)
        pf.group_pairs(idx, w, t, k, e, st["routes"], residency=st["table"])
        pf.encode_grouped_expert_gemms(pool, st["off"], st["routes"], x, d, _at(st["partials"]), st["ffn_ws"], t, k)
    pf.encode_reduce_token_major(_at(st["partials"]), w, _at(st["y"]), t, k, d)
    return [st["idx"], st["w"], st["y"]]


def _run_cpu(st):
    c, out = st["c"], st["out"]
    out.fill(0.0)
    for blob, weight in zip(st["blobs"], st["weights"]):
        host.cpu_expert_ffn_accumulate(blob, st["off"], st["x"], c["d"], c["f"], weight, out, st["scratch"])
    return out


def run(state):
    return {"decode": _run_decode, "batch": _run_decode, "prefill": _run_prefill, "streamed": _run_streamed, "cpu": _run_cpu}[state["c"]["kind"]](state)


# ---------------------------------------------------------------------------------------------- what a pass cannot do without

def _experts_used(c):
    """Distinct experts of a pass: the router's logits are normal with the spread of N(0, 0.02) rows against N(0, 1), plus the skew."""
    t, e, k = c["tokens"], c["experts"], c["top_k"]
    if c["skew"] == 0.0:  # every expert as likely as any other
        return e * (1.0 - (1.0 - k / e) ** t)
    rng = np.random.default_rng(0)
    logits = rng.standard_normal((t, e), dtype=np.float32) * 0.02 * math.sqrt(c["d"])
    logits -= c["skew"] * np.log(np.arange(1, e + 1, dtype=np.float32))
    return len(np.unique(np.argpartition(-logits, k - 1, axis=1)[:, :k]))


def work(case):
    c = dict(case)
    d, f, t, k, e = c["d"], c["f"], c["tokens"], c["top_k"], c["experts"]
    _, stride = synth.expert_offsets(d, f, c["bits"], c["expert_biases"])
    if c["kind"] == "cpu":
        return {"bytes": e * stride + 8.0 * d, "flops": 6.0 * e * d * f}
    router = e * d * (2 if c["router_bits"] == 0 else c["router_bits"] / 8 + 4 / GROUP)
    shared = 3 * d * c["shared_f"] * (c["bits"] / 8 + 4 / GROUP)
    rows = t * d * 2 * (4 if c["kind"] in ("decode", "batch") else 2)
    return {"bytes": c["layers"] * (_experts_used(c) * stride + router + shared + rows + t * k * 6),
            "flops": c["layers"] * t * (6.0 * d * (k * f + c["shared_f"]) + 2.0 * e * d)}


def tolerance(case):
    if case["kind"] == "cpu":
        return {"rel": 1e-5}  # fp32 sums
    return {"rel": 1e-3}      # fp16 results and fp16 roundings between the stages; routes are whole numbers and exact
