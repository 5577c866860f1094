"""Timed cases of the quantized KV-cache path, from single calls to whole layers.

A program that uses this package does five things with it, and a case is one of them:

* ``call``    one function-style decode call (``decode_attn_int8``, ``decode_attn_int4``,
              ``decode_attn_int4_asym`` over the KIVI layout) over a cache it has in hand;
* ``plan``    the decode attention of several layers, each a prepared ``DecodePlan`` over its
              layer's cache, as a serving loop launches them;
* ``prefill`` the hand-off of a prompt's K / V to a cache engine, layer by layer (``clear``, then
              ``append``: the buffers stay from the prompt before);
* ``turn``    a new engine, a prompt, then decode steps through it (``append``, then
              ``append_decode_attn`` per layer and token), as generation drives it;
* ``dequant`` ``get_kv`` of an engine's layers, the hand-over to a model's own attention.

Sizes: the head counts of the benchmark configurations (12/2, 28/4 and 40/8 query / KV heads,
head dimension 128), prompts and contexts from a short question to 64k tokens, batches 1 to 16.
K ~ N(0, 1) with 4 channels per head scaled x20, V and q ~ N(0, 1), as the benchmark draws them.
"""
import math

import torch

import llm_kvcache_quantization_amd as kvq
from llm_kvcache_quantization_amd import _capi as abi
from llm_kvcache_quantization_amd import kernels

D = 128
DEV = "cuda"
HEADS = ((12, 2), (28, 4), (40, 8))
SM = 1.0 / math.sqrt(D)

# largest number of (row, KV head, token) triples over all layers of a drawn case
MAX_CELLS = 1 << 20


def listed():
    return [
        # the smallest call: one sequence, a short chat context, INT8 with one scale per token
        dict(name="call_int8_short", op="call", fmt="int8", group=128, batch=1, q_heads=12, kv_heads=2,
             tokens=517, layers=1, ragged=False),
        # a small serving batch of uneven lengths through the INT4 drop-in call
        dict(name="call_int4_ragged", op="call", fmt="int4", group=32, batch=6, q_heads=28, kv_heads=4,
             tokens=7999, layers=1, ragged=True),
        # one decode step's attention over 8 layers, static INT8 tables, 4 sequences of 8k
        dict(name="plan_int8_8k", op="plan", fmt="int8_static", group=32, batch=4, q_heads=12, kv_heads=2,
             tokens=8192, layers=8, ragged=False),
        # the headline shape: asymmetric INT4 with fp16 outlier channels, 8 sequences of 32k
        dict(name="plan_asym_32k", op="plan", fmt="asym", group=32, batch=8, q_heads=28, kv_heads=4,
             tokens=32768, layers=2, ragged=False),
        # K INT8 / V INT4 over a ragged batch of long documents
        dict(name="plan_k8v4_ragged", op="plan", fmt="k8v4", group=32, batch=8, q_heads=40, kv_heads=8,
             tokens=65536, layers=1, ragged=True),
        # one chat turn: a 2k prompt, then an answer, KIVI at its default 8 bits
        dict(name="turn_kivi8", op="turn", fmt="kivi8", group=128, pct=100.0, batch=1, q_heads=28,
             kv_heads=4, tokens=1999, layers=2, steps=14),
        # the same for two longer prompts with calibrated INT4 scales and the group rescue
        dict(name="turn_int4_rescue", op="turn", fmt="int4_rescue", group=16, pct=100.0, batch=2,
             q_heads=28, kv_heads=4, tokens=4096, layers=2, steps=14),
        # prompt hand-off, dynamic INT8 scales at the default clip percentile
        dict(name="prefill_int8", op="prefill", fmt="int8", group=128, pct=99.9, batch=1, q_heads=12,
             kv_heads=2, tokens=4096, layers=4),
        # the largest hand-off: 8 prompts of 32k into one layer of the headline format
        dict(name="prefill_asym_32k", op="prefill", fmt="asym", group=32, pct=100.0, batch=8, q_heads=28,
             kv_heads=4, tokens=32768, layers=1),
        # prompt hand-off to the KIVI layout with calibrated clipping of both sides
        dict(name="prefill_kivi4_clip", op="prefill", fmt="kivi4", group=32, pct=99.9, batch=1,
             q_heads=28, kv_heads=4, tokens=8191, layers=2),
        # prompt hand-off, K INT8 / V INT4 with dynamic scales, a batch of short prompts
        dict(name="prefill_mixed_short", op="prefill", fmt="mixed", group=128, pct=99.9, batch=4,
             q_heads=40, kv_heads=8, tokens=333, layers=2),
        # the cache handed to a model's own attention as fp16
        dict(name="dequant_int4", op="dequant", fmt="int4", group=32, pct=99.9, batch=2, q_heads=28,
             kv_heads=4, tokens=6001, layers=2),
    ]


# formats a drawn case takes, per kind: every quantizer of the engines, every decode entry
_CALL = ("int8", "int4", "kivi4")
_PLAN = ("int8_static", "asym", "k8v4")
_ENGINE = ("int8", "int8_static", "int4", "int4_rescue", "kivi8", "kivi4", "mixed", "asym", "k8v4")
_DEQUANT = ("int8", "int8_static", "int4", "int4_rescue", "kivi8", "kivi4", "mixed")


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("call", "plan", "prefill", "prefill", "turn", "dequant"))
    q_heads, kv_heads = rng.choice(HEADS)
    batch = rng.choice((1, 1, 2, 3, 4, 6, 8, 16))
    layers = 1 if op == "call" else rng.choice((1, 2, 4))
    lo, hi = {"call": (64, 65536), "plan": (256, 65536), "prefill": (24, 32768), "turn": (64, 8192),
              "dequant": (64, 16384)}[op]
    # a turn reads its cache again at every step
    cells = MAX_CELLS // 4 if op == "turn" else MAX_CELLS
    tokens = _log_uniform(rng, lo, min(hi, cells // (batch * kv_heads * layers)))
    case = dict(op=op, batch=batch, q_heads=q_heads, kv_heads=kv_heads, tokens=tokens, layers=layers)
    if op == "call":
        fmt = rng.choice(_CALL)
        group = 32 if fmt == "kivi4" else rng.choice((16, 32, 64, 128))
        case.update(fmt=fmt, group=group, ragged=batch > 1 and rng.random() < 0.5)
    elif op == "plan":
        fmt = rng.choice(_PLAN)
        case.update(fmt=fmt, group=rng.choice((16, 32, 64)) if fmt == "int8_static" else 32,
                    ragged=batch > 1 and rng.random() < 0.5)
    else:
        fmt = rng.choice(_DEQUANT if op == "dequant" else _ENGINE)
        group = {"int8": rng.choice((32, 64, 128)), "int8_static": rng.choice((16, 32)),
                 "int4": rng.choice((16, 32, 64)), "int4_rescue": 16,
                 "mixed": rng.choice((64, 128))}.get(fmt, 32)
        pct = rng.choice((100.0, 99.9, 99.9)) if fmt in ("int8", "int4", "kivi8", "kivi4", "mixed") else 100.0
        case.update(fmt=fmt, group=group, pct=pct)
        if op == "turn":
            case["steps"] = max(1, min(rng.choice((3, 6, 12)), 48 // layers))
    return case


# ---------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + 17)


def _kv(case, tokens, g):
    """fp16 K, V [B, Hkv, tokens, 128]."""
    shape = (case["batch"], case["kv_heads"], tokens, D)
    k = torch.randn(shape, generator=g, device=DEV).half()
    for h, ch in enumerate(_outliers(case)):
        k[:, h, :, ch] *= 20
    v = torch.randn(shape, generator=g, device=DEV).half()
    return k, v


def _outliers(case):
    """The 4 scaled K channels of each KV head."""
    g = torch.Generator().manual_seed(case["kv_heads"])
    return [torch.randperm(D, generator=g)[:4].tolist() for _ in range(case["kv_heads"])]


def _q(case, g):
    return torch.randn(case["batch"], case["q_heads"], D, generator=g, device=DEV).half()


def _tau(case, g):
    return (0.8 + 0.4 * torch.rand(case["q_heads"], generator=g, device=DEV)).half()


def _contexts(case, g):
    """Row lengths: all `tokens`, or ragged with the longest at `tokens`."""
    n, B = case["tokens"], case["batch"]
    if not case.get("ragged"):
        return [n] * B
    lens = torch.randint(max(1, n // 16), n + 1, (B,), generator=g, device=DEV).tolist()
    lens[B // 2] = n
    return lens


def _per_group(case, qmax, g):
    """Calibrated static scales [Hkv, G]: the absmax of 512 tokens over qmax, per group."""
    sample = dict(case, batch=1)
    out = []
    for x in _kv(sample, 512, g):
        a = x[0].float().abs().view(case["kv_heads"], 512, D // case["group"], case["group"])
        out.append(a.amax(dim=(1, 3)) / qmax)
    return out


def _asym_tables(case, g):
    """Calibrated scale / zero-point [Hkv, 4] of K (its outlier channels left out) and V."""
    sample = dict(case, batch=1)
    k, v = _kv(sample, 512, g)
    for h, ch in enumerate(_outliers(case)):
        k[:, h, :, ch] = 0
    out = []
    for x in (k, v):
        x = x[0].float().view(case["kv_heads"], 512, 4, 32)
        lo, hi = x.amin(dim=(1, 3)), x.amax(dim=(1, 3))
        s = ((hi - lo) / 15).clamp(min=1e-4).half()
        out += [s, (lo + 8 * s.float()).half()]
    return out


def _codes(shape, qmin, qmax, spread, g):
    return (torch.randn(shape, generator=g, device=DEV) * spread).round_().clamp_(qmin, qmax).to(torch.int8)


def _pack(c):
    """Two 4-bit codes a byte, the even channel in the high nibble, offset 8."""
    u = (c + 8).view(torch.uint8)
    return (u[..., 0::2] << 4) | u[..., 1::2]


def _layer_cache(case, g):
    """One layer's quantized cache as codes and parameters (a cache the program has in hand)."""
    B, H, n, fmt, gs = case["batch"], case["kv_heads"], case["tokens"], case["fmt"], case["group"]
    shape, G = (B, H, n, D), D // gs
    c = {}
    if fmt in ("int8", "int4", "int8_static"):
        qmax, spread = (7, 2.2) if fmt == "int4" else (127, 34.0)
        c["k"], c["v"] = (_codes(shape, -qmax, qmax, spread, g) for _ in range(2))
        for side in ("ks", "vs"):
            sshape = (H, G) if fmt == "int8_static" else (B, H, n, G)
            s = (0.6 + 0.8 * torch.rand(sshape, generator=g, device=DEV)) / spread
            if side == "ks":  # the head's outlier group is the wide one
                s[..., 0] *= 6
            c[side] = s.half()
    elif fmt == "kivi4":
        c["k"], c["v"] = (_codes(shape, -8, 7, 2.8, g) for _ in range(2))
        c["ks"] = (0.3 + 0.2 * torch.rand(B, H, D, generator=g, device=DEV))
        for h, ch in enumerate(_outliers(case)):
            c["ks"][:, h, ch] *= 12
        c["kz"] = 0.1 * torch.randn(B, H, D, generator=g, device=DEV)
        c["vs"] = 0.3 + 0.1 * torch.rand(B, H, n, generator=g, device=DEV)
        c["vz"] = 0.1 * torch.randn(B, H, n, generator=g, device=DEV)
    else:
        c["k"] = _codes(shape, -127, 127, 34.0, g) if fmt == "k8v4" else _codes(shape, -8, 7, 2.8, g)
        c["v"] = _codes(shape, -8, 7, 2.8, g)
        if fmt == "k8v4":
            c["ks"] = ((0.6 + 0.8 * torch.rand(H, 4, generator=g, device=DEV)) / 34.0).half()
        else:
            c["ks"] = (0.3 + 0.1 * torch.rand(H, 4, generator=g, device=DEV)).half()
            c["kz"] = (0.1 * torch.randn(H, 4, generator=g, device=DEV)).half()
            c["oi"] = torch.tensor(_outliers(case), dtype=torch.int32, device=DEV)
            c["ov"] = (20 * torch.randn(B, H, n, 4, generator=g, device=DEV)).half()
        c["vs"] = (0.3 + 0.1 * torch.rand(H, 4, generator=g, device=DEV)).half()
        c["vz"] = (0.1 * torch.randn(H, 4, generator=g, device=DEV)).half()
    return c


def _caches(case, seed):
    """(per layer: cache, q, inv_tau), row lengths."""
    g = _gen(seed)
    lens = _contexts(case, g)
    return [(_layer_cache(case, g), _q(case, g), _tau(case, g)) for _ in range(case["layers"])], lens


# ---------------------------------------------------------------- engines


def _engine(case, tables, cap):
    fmt, gs, n, pct = case["fmt"], case["group"], case["layers"], case["pct"]
    if fmt == "int8":
        return kvq.INT8KVCache(n, DEV, clip_percentile=pct, group_size=gs, max_seq_len=cap)
    if fmt == "int4":
        return kvq.INT4KVCache(n, DEV, clip_percentile=pct, group_size=gs, max_seq_len=cap)
    if fmt == "int8_static":
        return kvq.INT8KVCache(n, DEV, group_size=gs, max_seq_len=cap, static_k_scale=tables["ks"],
                               static_v_scale=tables["vs"])
    if fmt == "int4_rescue":
        return kvq.INT4KVCache(n, DEV, group_size=gs, max_seq_len=cap, static_k_scale=tables["ks"],
                               static_v_scale=tables["vs"], outlier_rescue_ratio=0.01)
    if fmt in ("kivi8", "kivi4"):
        return kvq.KIVIStyleKVCache(n, DEV, max_seq_len=cap, quant_bits=int(fmt[-1]), k_percentile=pct,
                                    v_percentile=pct)
    if fmt == "mixed":
        return kvq.MixedKVCache(n, DEV, max_seq_len=cap, k_group_size=gs, k_clip_percentile=pct,
                                v_percentile=pct)
    if fmt == "asym":
        return kvq.INT4AsymKVCache(n, tables["ks"], tables["kz"], tables["vs"], tables["vz"], device=DEV,
                                   max_seq_len=cap, k_outlier_idx=tables["oi"])
    return kvq.K8V4KVCache(n, tables["ks"], tables["vs"], tables["vz"], device=DEV, max_seq_len=cap)


def _tables(case, g):
    L = case["layers"]
    if case["fmt"] in ("int8_static", "int4_rescue"):
        ks, vs = _per_group(case, 127.0 if case["fmt"] == "int8_static" else 7.0, g)
        if case["fmt"] == "int8_static":
            ks, vs = ks.half(), vs.half()
        return {"ks": ks[None].repeat(L, 1, 1), "vs": vs[None].repeat(L, 1, 1)}
    if case["fmt"] in ("asym", "k8v4"):
        ks, kz, vs, vz = (t[None].repeat(L, 1, 1) for t in _asym_tables(case, g))
        if case["fmt"] == "k8v4":
            ks = (_per_group(case, 127.0, g)[0]).half()[None].repeat(L, 1, 1)
        oi = torch.tensor(_outliers(case), dtype=torch.int32)[None].repeat(L, 1, 1)
        return {"ks": ks, "kz": kz, "vs": vs, "vz": vz, "oi": oi}
    return {}


def _prompt(case, seed):
    """Tables, and per layer the prompt's K / V and every decode step's q, k, v."""
    g = _gen(seed)
    tables = _tables(case, g)
    layers = []
    for _ in range(case["layers"]):
        k, v = _kv(case, case["tokens"], g)
        steps = [(_q(case, g),) + _kv(case, 1, g) for _ in range(case.get("steps", 0))]
        layers.append((k, v, steps))
    return tables, layers, _tau(case, g)


def _stored(case, eng, layer):
    """What the engine holds of a layer: codes and parameters."""
    fmt = case["fmt"]
    if fmt in ("int8", "int8_static"):
        kc, vc, ks, vs = eng.get_int8_tensors(layer)
        return [kc, vc] if fmt == "int8_static" else [kc, vc, ks, vs]
    if fmt in ("int4", "int4_rescue"):
        return list(eng.get_int4_tensors(layer))
    if fmt in ("kivi8", "kivi4"):
        return list(eng.get_kivi_tensors(layer))
    if fmt == "mixed":
        return list(eng.get_mixed_tensors(layer))
    if fmt == "asym":
        t = eng.get_int4_g32_tensors(layer)
        return [t[0], t[1], t[7]]
    t = eng.get_k8v4_tensors(layer)
    return [t[0], t[2]]


# ---------------------------------------------------------------- the cases' functions


def prepare(case, seed):
    op, fmt = case["op"], case["fmt"]
    if op in ("call", "plan"):
        layers, lens = _caches(case, seed)
        ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
        st = {"case": case, "ctx": ctx}
        if op == "call":
            c, q, _ = layers[0]
            if fmt in ("int4", "kivi4"):
                c["k"], c["v"] = _pack(c["k"]).view(torch.int8), _pack(c["v"]).view(torch.int8)
            st.update(c=c, q=q)
            return st
        B, H, n = case["batch"], case["kv_heads"], case["tokens"]
        # uniform batches pass their length by value, ragged ones their lengths' tensor
        where = ctx if case["ragged"] else n
        plans = []
        for c, q, tau in layers:
            if fmt == "int8_static":
                k, v = (kernels.kv_view_tok(c[x], c[x + "s"][None, :, None].expand(B, H, n, D // case["group"]))
                        for x in "kv")
                kf = vf = abi.KVQ_FMT_INT8_SYM
            else:
                vf = abi.KVQ_FMT_INT4_ASYM
                v = kernels.kv_view_static(kvq.tile_v(_pack(c["v"])), c["vs"], c["vz"])
                if fmt == "asym":
                    kf = abi.KVQ_FMT_INT4_ASYM
                    k = kernels.kv_view_static(_pack(c["k"]), c["ks"], c["kz"], c["oi"], c["ov"])
                else:
                    kf = abi.KVQ_FMT_INT8_SYM
                    k = kernels.kv_view_tok(c["k"], c["ks"][None, :, None].expand(B, H, n, 4))
            plans.append(kvq.DecodePlan(q, kf, k, vf, v, where, H, n, SM, case["group"], inv_tau=tau,
                                        keepalive=(c,)))
        st["plans"] = plans
        return st
    tables, layers, tau = _prompt(case, seed)
    if op == "turn":
        return {"case": case, "tables": tables, "layers": layers, "tau": tau}
    cap = -(-case["tokens"] // 32) * 32
    eng = _engine(case, tables, cap)
    # the engine has served a prompt of full length before: its buffers are there
    zk = torch.zeros(case["batch"], case["kv_heads"], cap, D, dtype=torch.float16, device=DEV)
    for i in range(case["layers"]):
        eng.append(i, zk, zk)
    eng.clear()
    st = {"case": case, "eng": eng, "layers": layers}
    if op == "dequant":
        for i, (k, v, _) in enumerate(layers):
            eng.append(i, k, v)
    return st


def run(state):
    case = state["case"]
    op, fmt = case["op"], case["fmt"]
    if op == "call":
        c, q, ctx = state["c"], state["q"], state["ctx"]
        if fmt == "int8":
            return kvq.decode_attn_int8(q, c["k"], c["v"], c["ks"], c["vs"], ctx, SM)
        if fmt == "int4":
            return kvq.decode_attn_int4(q, c["k"], c["v"], c["ks"], c["vs"], ctx, SM)
        return kvq.decode_attn_int4_asym(q, c["k"], c["v"], c["ks"], c["kz"], c["vs"], c["vz"], ctx, SM)
    if op == "plan":
        return [p.launch() for p in state["plans"]]
    L = case["layers"]
    if op == "dequant":
        return [state["eng"].get_kv(i) for i in range(L)]
    if op == "turn":
        eng = _engine(case, state["tables"], case["tokens"] + case["steps"])
    else:
        eng = state["eng"]
        eng.clear()
    for i, (k, v, _) in enumerate(state["layers"]):
        eng.append(i, k, v)
    if op == "prefill":
        return [_stored(case, eng, i) for i in range(L)]
    out = []
    for s in range(case["steps"]):
        for i in range(L):
            q, k, v = state["layers"][i][2][s]
            out.append(eng.append_decode_attn(i, q, k, v, SM, inv_tau=state["tau"]))
    return out


def _cell_bytes(case):
    """(code bytes, parameter bytes) one (row, KV head, token) takes in the cache, K and V."""
    fmt, G = case["fmt"], D // case["group"]
    return {"int8": (256, 4 * G), "int8_static": (256, 0), "int4": (128, 8 * G), "int4_rescue": (128, 8 * G),
            "kivi8": (256, 8), "kivi4": (128, 8), "mixed": (192, 2 * G + 8), "asym": (128, 8),
            "k8v4": (192, 0)}[fmt]


def work(case):
    op, B, H, L = case["op"], case["batch"], case["kv_heads"], case["layers"]
    code, par = _cell_bytes(case)
    if op == "call" and case["fmt"] == "int4":
        par //= 2  # the call takes fp16 scales
    cell = code + par
    if op in ("call", "plan"):
        # ragged rows hold (tokens / 16 .. tokens) uniformly, the longest at `tokens`
        n = case["tokens"]
        total = B * n if not case["ragged"] else n + (B - 1) * n * 17 // 32
        return {"bytes": L * (H * total * cell + 4 * B * case["q_heads"] * D),
                "flops": L * 4.0 * total * case["q_heads"] * D}
    cells = L * B * H * case["tokens"]
    fill = cells * (2 * 2 * D + cell)
    if op == "prefill":
        return {"bytes": fill, "flops": 0}
    if op == "dequant":
        return {"bytes": cells * (cell + 2 * 2 * D), "flops": 0}
    S = case["steps"]
    seen = L * B * (S * case["tokens"] + S * (S + 1) // 2)
    return {"bytes": fill + seen * H * cell + L * S * B * (4 * case["q_heads"] * D + H * (4 * D + cell)),
            "flops": 4.0 * seen * case["q_heads"] * D}


def tolerance(case):
    if case["op"] == "prefill":
        return "exact"  # codes and scales are the reference quantizer's bits
    if case["op"] == "dequant":
        return "exact"  # one rounding to fp16 of an fp32 product (and sum)
    # fp16 outputs; over splits of 256 to 16384 tokens a work-group they differ from each other by
    # rel 8e-5 and, in single values, one ulp (max 9.8e-4): four times that
    return {"rel": 4e-4, "max": 4e-3}


# ---------------------------------------------------------------- 64-bit results


def _attend(q, k, v):
    """softmax(q k^T / sqrt(128)) v in 64 bits: q [Hq, 128], k / v [Hkv, n, 128]."""
    Hkv = k.shape[0]
    qg = q.double().view(Hkv, -1, D)
    p = torch.softmax(torch.matmul(qg, k.transpose(1, 2).contiguous()) * SM, dim=-1)
    return torch.matmul(p, v).reshape(-1, D)


def _exact_caches(case, seed):
    layers, lens = _caches(case, seed)
    B, H, fmt, gs = case["batch"], case["kv_heads"], case["fmt"], case["group"]
    outs = []
    for c, q, tau in layers:
        if case["op"] == "plan":
            q = q * tau.view(1, -1, 1)  # the scaled query is fp16 by definition
        rows = []
        for b in range(B):
            n = lens[b]

            def side(x):
                z = c[x][b, :, :n].double()
                s = c[x + "s"].double()
                if fmt in ("int8", "int4"):
                    return (z.view(H, n, D // gs, gs) * s[b, :, :n, :, None]).view(H, n, D)
                if fmt == "kivi4":
                    zp = c[x + "z"].double()
                    if x == "k":
                        return z * s[b][:, None] + zp[b][:, None]
                    return z * s[b, :, :n, None] + zp[b, :, :n, None]
                r = z.view(H, n, D // gs, gs) * s[:, None, :, None]
                if x + "z" in c:
                    r = r + c[x + "z"].double()[:, None, :, None]
                return r.view(H, n, D)

            k, v = side("k"), side("v")
            if fmt == "asym":
                for h in range(H):
                    k[h][:, c["oi"][h].long()] = c["ov"][b, h, :n].double()
            rows.append(_attend(q[b], k, v))
        outs.append(torch.stack(rows))
    return outs[0] if case["op"] == "call" else outs


def _level(x, p, dim):
    """Quantile p / 100 of x along dim in 64 bits, between the two nearest ranks."""
    s = torch.sort(x.double(), dim=dim).values
    r = p / 100.0 * (x.shape[dim] - 1)
    lo = int(math.floor(r))
    hi = min(lo + 1, x.shape[dim] - 1)
    a, b = s.select(dim, lo), s.select(dim, hi)
    return a + (r - lo) * (b - a)


def _range(x, pct, span, dim):
    """Scale and zero-point of an asymmetric range over dim (codes from -(span + 1) / 2)."""
    if pct < 100.0:
        lo, hi = _level(x, 100.0 - pct, dim), _level(x, pct, dim)
    else:
        lo, hi = x.double().amin(dim), x.double().amax(dim)
    s = (hi - lo).clamp(min=span * 2.0 ** -14) / span
    return s, lo + (span + 1) / 2 * s


def _quantized(case, x, side, tables, layer, frozen=None):
    """(dequantised values, parameters) of rows x [B, H, S, 128] in 64 bits."""
    fmt, gs = case["fmt"], case["group"]
    B, H, S, _ = x.shape
    xd = x.double()
    if fmt in ("kivi8", "kivi4") or (fmt == "mixed" and side == "v"):
        span = 255.0 if fmt == "kivi8" else 15.0
        if side == "k":
            s, z = frozen if frozen is not None else _range(xd, case["pct"], span, 2)
            se, ze = s[:, :, None], z[:, :, None]
        else:
            s, z = _range(xd, case["pct"], span, 3)
            se, ze = s[..., None], z[..., None]
        half = (span + 1) / 2
        return ((xd - ze) / se).round().clamp(-half, half - 1) * se + ze, (s, z)
    xg = xd.view(B, H, S, D // gs, gs)
    if fmt in ("asym", "k8v4") and not (fmt == "k8v4" and side == "k"):
        s, z = (tables[side + n][layer].to(DEV).double()[None, :, None, :, None] for n in "sz")
        y = (((xg - z) / s).round().clamp(-8, 7) * s + z).view(B, H, S, D)
        if side == "k":
            for h, ch in enumerate(_outliers(case)):
                y[:, h, :, ch] = xd[:, h, :, ch]
        return y, ()
    int8 = fmt in ("int8", "int8_static", "mixed", "k8v4")
    qmax = 127.0 if int8 else 7.0
    if fmt in ("int8_static", "k8v4"):
        s = tables[side + "s"][layer].to(DEV).double()[None, :, None].expand(B, H, S, D // gs)
    else:
        a = xg.abs()
        am = _level(a, case["pct"], 4) if case["pct"] < 100.0 else a.amax(4)
        s = am.clamp(min=1e-5) / qmax
        if fmt == "int4_rescue":
            st = tables[side + "s"][layer].to(DEV).double()[None, :, None].expand_as(s)
            s = torch.where(s >= _level(s.reshape(-1), 99.0, 0), torch.maximum(st, s), st)
    # the codes are whole numbers by definition: INT8 scales are fp16 and the quotient too
    if int8:
        am16 = s.half() if fmt in ("int8_static", "k8v4") else am.half() / torch.full_like(am, 127).half()
        c = (x.view(xg.shape) / am16[..., None]).round().clamp(-127, 127).double()
        y = c * am16.double()[..., None]
    else:
        c = (xg.float() / s.float()[..., None]).round().clamp(-7, 7).double()
        # decode attention reads INT4 scales as fp16 (as the reference's does), get_kv as fp32
        y = c * (s.half() if case["op"] == "turn" else s.float()).double()[..., None]
    return y.view(B, H, S, D), (s,)


def exact(case, seed):
    if case["op"] in ("call", "plan"):
        return _exact_caches(case, seed)
    op, fmt = case["op"], case["fmt"]
    tables, layers, tau = _prompt(case, seed)
    per_layer = []
    for i, (k, v, steps) in enumerate(layers):
        yk, pk = _quantized(case, k, "k", tables, i)
        yv, pv = _quantized(case, v, "v", tables, i)
        if op == "dequant":
            per_layer.append((yk, yv))
        elif op == "prefill":
            # the engine's order: codes (whole numbers, left out), then parameters
            if fmt in ("int8", "int4", "int4_rescue"):
                per_layer.append([None, None, pk[0], pv[0]])
            elif fmt in ("kivi8", "kivi4"):
                per_layer.append([None, None, *pk, *pv])
            elif fmt == "mixed":
                per_layer.append([None, pk[0], None, *pv])
            elif fmt == "asym":  # the outlier channels' values, as they come
                per_layer.append([None, None, torch.stack(
                    [k[:, h][..., ch] for h, ch in enumerate(_outliers(case))], 1).double()])
            else:
                return None  # codes alone
        else:
            outs = []
            for q, k1, v1 in steps:
                yk = torch.cat([yk, _quantized(case, k1, "k", tables, i, pk)[0]], 2)
                yv = torch.cat([yv, _quantized(case, v1, "v", tables, i)[0]], 2)
                qs = q * tau.view(1, -1, 1)
                outs.append(torch.stack([_attend(qs[b], yk[b], yv[b]) for b in range(case["batch"])]))
            per_layer.append(outs)
    if op == "turn":
        return [per_layer[i][s] for s in range(case["steps"]) for i in range(case["layers"])]
    return per_layer
