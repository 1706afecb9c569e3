"""The work that users of this package run, as measurable cases.

A case is a dict of plain values. Its ``kind`` names the entry point:

  step    one decode token of one layer, called eagerly: ``append_and_attend``
          of a ``QuantizedKVCache`` (the token is then dropped again with
          ``crop``, as assisted decoding does with a rejected draft)
  token   one decode token through every layer, replayed as a HIP graph of
          ``ops.decode_step`` launches (how ``bench.py`` and the graph decoder
          run decoding)
  paged   one decode token of a ragged batch over a paged cache, one layer
  append  a prompt's K and V quantized into a fresh ``QuantizedKVCache``
  codec   ``quantize_int4`` and ``dequantize_int4`` on a tensor
  attend  attention of a query block over the packed cache
          (``attention_forward_quant_gqa`` / ``attention_forward_quant``):
          whole prompts, prompt chunks after cached tokens, speculative blocks
  model   one decode token of a Llama model with swapped attention modules,
          called through Hugging Face's forward

Shapes are those of the repository's own benchmark workloads (GPT-2 small and
XL, Llama-3.1-8B, the 70B shape) or of the same ranges, with odd and ragged
sizes among them. Weights and activations are random; keys carry eight
outlier channels, as trained models' keys do.
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (_ROOT, os.path.join(_ROOT, "kv-cache-triton_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _size(dtype):
    return 4 if dtype == "f32" else 2


def listed():
    return [
        # the smallest call: GPT-2 small in fp32, one layer of one decode token (latency and launches)
        dict(name="gpt2-step-1k", kind="step", family="gpt2", dtype="f32", B=1, Hq=12, Hkv=12, D=64, G=32, ctx=1024),
        # the ordinary case: Llama-3.1-8B at 16K context, one token through 32 layers
        dict(name="llama8b-token-16k", kind="token", dtype="bf16", B=1, Hq=32, Hkv=8, D=128, G=32, ctx=16384,
             layers=32, ragged=False),
        # large batched decoding: the 70B shape, batch 8 at 32K context (four of its layers)
        dict(name="llama70b-token-b8-32k", kind="token", dtype="bf16", B=8, Hq=64, Hkv=8, D=128, G=32, ctx=32768,
             layers=4, ragged=False),
        # GPT-2 XL in fp16, a ragged batch of 16 short sequences, one token through 48 layers
        dict(name="gpt2xl-token-ragged-b16", kind="token", dtype="f16", B=16, Hq=25, Hkv=25, D=64, G=32, ctx=1024,
             layers=48, ragged=True),
        # serving: a ragged batch of 32 sequences of very different lengths over a paged cache
        dict(name="llama8b-paged-ragged-b32", kind="paged", dtype="bf16", B=32, Hq=32, Hkv=8, D=128, G=32, ctx=16384,
             page=64),
        # a 16K prompt's K and V going into the cache (one layer)
        dict(name="llama8b-append-16k", kind="append", family="llama3", dtype="bf16", B=1, Hkv=8, D=128, G=32, S=16384),
        # the quantizer and dequantizer on a head dim that the group size does not divide, an odd row count
        dict(name="codec-d80-odd", kind="codec", family="llama3", dtype="bf16", B=2, H=32, S=3001, D=80, G=32),
        # a whole 16K prompt's attention (the largest)
        dict(name="llama8b-prompt-16k", kind="attend", family="llama3", dtype="bf16", B=1, Hq=32, Hkv=8, D=128, G=32,
             Sq=16384, Sk=16384, causal=True),
        # a prompt chunk of odd length after odd cached tokens, fp16
        dict(name="llama8b-chunk-odd-f16", kind="attend", family="llama3", dtype="f16", B=1, Hq=32, Hkv=8, D=128, G=32,
             Sq=777, Sk=9001, causal=True),
        # a speculative block of 8 tokens
        dict(name="llama8b-spec8-8k", kind="attend", family="llama3", dtype="bf16", B=1, Hq=32, Hkv=8, D=128, G=32,
             Sq=8, Sk=8200, causal=True),
        # a whole GPT-2 small prompt in fp32
        dict(name="gpt2-prompt-1k-f32", kind="attend", family="gpt2", dtype="f32", B=1, Hq=12, Hkv=12, D=64, G=32,
             Sq=1000, Sk=1000, causal=True),
        # a whole call: one eager decode token of a 4-layer Llama of the 8B widths at 4K context, logits out
        dict(name="llama-model-token-4k", kind="model", dtype="bf16", layers=4, hidden=4096, inter=14336, Hq=32, Hkv=8,
             D=128, G=32, vocab=32000, ctx=4096),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["step", "token", "token", "paged", "append", "codec", "attend", "attend", "attend", "model"])
    if kind == "step":
        if rng.random() < 0.5:
            return dict(kind=kind, family="gpt2", dtype=rng.choice(["f32", "f16"]), B=rng.randint(1, 4), Hq=12, Hkv=12,
                        D=64, G=32, ctx=_log(rng, 32, 1023))
        ratio = rng.choice([1, 4, 8])
        return dict(kind=kind, family="llama3", dtype=rng.choice(["bf16", "f16"]), B=rng.randint(1, 4), Hq=8 * ratio,
                    Hkv=8, D=128, G=rng.choice([32, 64, 128]), ctx=_log(rng, 64, 16384))
    if kind == "token":
        if rng.random() < 0.25:
            return dict(kind=kind, dtype="f16", B=_log(rng, 1, 24), Hq=25, Hkv=25, D=64, G=32, ctx=_log(rng, 128, 1023),
                        layers=rng.randint(12, 48), ragged=rng.random() < 0.7)
        B = _log(rng, 1, 32)
        ctx = _log(rng, 512, min(32768, 262144 // B))
        layers = rng.randint(2, max(2, min(32, (1 << 19) // (B * ctx))))
        return dict(kind=kind, dtype="bf16", B=B, Hq=rng.choice([32, 64]), Hkv=8, D=128, G=32, ctx=ctx, layers=layers,
                    ragged=B > 1 and rng.random() < 0.4)
    if kind == "paged":
        return dict(kind=kind, dtype=rng.choice(["bf16", "f16"]), B=_log(rng, 2, 48), Hq=rng.choice([32, 64]), Hkv=8,
                    D=128, G=32, ctx=_log(rng, 512, 16384), page=rng.choice([64, 128, 256]))
    if kind == "append":
        B = rng.randint(1, 4)
        return dict(kind=kind, family="llama3", dtype=rng.choice(["bf16", "f16"]), B=B, Hkv=8, D=128,
                    G=rng.choice([32, 64, 128]), S=_log(rng, 8, 32768 // B))
    if kind == "codec":
        family = rng.choice(["llama3", "gpt2"])
        return dict(kind=kind, family=family, dtype=rng.choice(["bf16", "f16", "f32"]), B=rng.randint(1, 3),
                    H=rng.choice([8, 12, 32]), S=_log(rng, 5, 6000), D=rng.choice([64, 80, 96, 120, 128]),
                    G=rng.choice([16, 32, 64]))
    if kind == "model":
        return dict(kind=kind, dtype="bf16", layers=rng.randint(2, 4), hidden=rng.choice([2048, 4096]), inter=8192,
                    Hq=32, Hkv=8, D=128, G=32, vocab=32000, ctx=_log(rng, 128, 8192))
    if rng.random() < 0.2:
        S = _log(rng, 32, 1024)
        return dict(kind=kind, family="gpt2", dtype=rng.choice(["f32", "f16"]), B=rng.randint(1, 2), Hq=12, Hkv=12,
                    D=64, G=32, Sq=S, Sk=S, causal=True)
    Sk = _log(rng, 512, 16384)
    Sq = Sk if rng.random() < 0.25 else _log(rng, 2, min(Sk, 4096))
    Hq = rng.choice([32, 64]) if Sq < 8192 else 32
    return dict(kind=kind, family="llama3", dtype=rng.choice(["bf16", "bf16", "f16"]), B=1, Hq=Hq, Hkv=8,
                D=128, G=rng.choice([32, 32, 64, 128]), Sq=Sq, Sk=Sk, causal=True)


# ---------------------------------------------------------------------------
# inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _randn(g, *shape, dtype):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(DT[dtype])


def _keys(g, *shape, dtype):
    """Key rows with eight outlier channels of eight times the others' size."""
    x = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    D = shape[-1]
    x[..., [(5 + 13 * i) % D for i in range(8)]] *= 8.0
    return x.to(DT[dtype])


def _scale_dtype(case):
    gpt2 = case.get("family", "gpt2" if case["dtype"] == "f16" and case["D"] == 64 else "llama3") == "gpt2"
    return torch.float16 if gpt2 else DT[case["dtype"]]


def _lengths(case, seed):
    """Ragged lengths on the host: spread over the logarithm of [ctx / 64, ctx], the longest ctx."""
    g = torch.Generator().manual_seed(int(seed) & 0x7FFFFFFF)
    lo = max(1, case["ctx"] // 64)
    u = torch.rand(case["B"], generator=g)
    lens = (lo * torch.exp(u * math.log(case["ctx"] / lo))).round().long().clamp(lo, case["ctx"])
    lens[int(torch.randint(case["B"], (1,), generator=g))] = case["ctx"]
    return lens


def _step_inputs(case, g, layer_ctx):
    B, D, dt = case["B"], case["D"], case["dtype"]
    k = _keys(g, B, case["Hkv"], layer_ctx, D, dtype=dt)
    v = _randn(g, B, case["Hkv"], layer_ctx, D, dtype=dt)
    kn = _keys(g, B, case["Hkv"], 1, D, dtype=dt)
    vn = _randn(g, B, case["Hkv"], 1, D, dtype=dt)
    q = _randn(g, B, case["Hq"], 1, D, dtype=dt)
    return q, k, v, kn, vn


def _family(case):
    if case["family"] == "gpt2":
        from kvint4.gpt2 import attention_quant, kv_cache, quantize
        return kv_cache.QuantizedKVCache, quantize, attention_quant.attention_forward_quant
    from kvint4.llama3 import attention_quant, kv_cache, quantize
    return kv_cache.QuantizedKVCache, quantize, attention_quant.attention_forward_quant_gqa


def _rope(x, pos, theta):
    """Rotary embedding of one position, the half-rotation form."""
    D = x.shape[-1]
    inv = theta ** (-torch.arange(0, D, 2, device=x.device, dtype=x.dtype) / D)
    ang = torch.cat((inv, inv)) * pos
    a, b = x[..., : D // 2], x[..., D // 2:]
    return x * ang.cos() + torch.cat((-b, a), -1) * ang.sin()


THETA, EPS = 500000.0, 1e-5


def _model_weights(case, g):
    H, I, V, D = case["hidden"], case["inter"], case["vocab"], case["D"]

    def w(rows, cols):
        return torch.empty(rows, cols, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=g)

    layers = [dict(q=w(case["Hq"] * D, H), k=w(case["Hkv"] * D, H), v=w(case["Hkv"] * D, H), o=w(H, case["Hq"] * D),
                   gate=w(I, H), up=w(I, H), down=w(H, I)) for _ in range(case["layers"])]
    return dict(embed=w(V, H), head=w(V, H), layers=layers)


def _model_inputs(case, g):
    kv = [(_keys(g, 1, case["Hkv"], case["ctx"], case["D"], dtype="bf16"),
           _randn(g, 1, case["Hkv"], case["ctx"], case["D"], dtype="bf16")) for _ in range(case["layers"])]
    tok = torch.randint(0, case["vocab"], (1, 1), generator=g, device="cuda")
    return kv, tok


# ---------------------------------------------------------------------------
# prepare / run


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    from kvint4 import ops

    if kind == "step":
        cache_cls, _, _ = _family(case)
        q, k, v, kn, vn = _step_inputs(case, g, case["ctx"])
        cache = cache_cls(group_size=case["G"], reserve_tokens=case["ctx"] + 64)
        cache.append(k, v, 0)
        cache.append(kn, vn, 0)  # the row that the measured step writes, so that the views below hold no garbage
        views = cache.get_quantized(0)
        cache.crop(-1)
        return dict(kind=kind, cache=cache, q=q, kn=kn, vn=vn, H=case["Hkv"], scale=case["D"] ** -0.5, views=views)
    if kind == "token":
        return _prepare_token(case, g, seed, ops)
    if kind == "paged":
        from kvint4.paged_cache import PagedQuantizedKVCache

        lens = _lengths(case, seed)
        q, k, v, kn, vn = _step_inputs(case, g, case["ctx"])
        # a serving program sizes its pool up front
        cache = PagedQuantizedKVCache(group_size=case["G"], page_size=case["page"],
                                      num_blocks=case["B"] * (case["ctx"] // case["page"] + 1))
        cache.load_ragged(k, v, 0, lens)
        cache.make_static(1)
        pools = cache.pools(0)
        for t in pools:  # rows of the pool that hold no token stay untouched by the step
            used = torch.zeros(t.shape[1], dtype=torch.bool, device=t.device)
            for b, n in enumerate(lens.tolist()):
                pos = torch.arange(n, device=t.device)
                used[cache.block_table()[b, pos // case["page"]].long() * case["page"] + pos % case["page"]] = True
            t[:, ~used] = 0
        table = ops.PageTable(cache.block_table(), case["page"], pools[0].shape[1] // case["page"])
        return dict(kind=kind, q=q, kn=kn, vn=vn, pools=pools, table=table, pos=cache.get_seq_lens(0), H=case["Hkv"],
                    G=case["G"], scale=case["D"] ** -0.5, cache=cache)
    if kind == "append":
        cache_cls, _, _ = _family(case)
        k = _keys(g, case["B"], case["S"], case["Hkv"], case["D"], dtype=case["dtype"]).transpose(1, 2)
        v = _randn(g, case["B"], case["S"], case["Hkv"], case["D"], dtype=case["dtype"]).transpose(1, 2)
        return dict(kind=kind, cls=cache_cls, G=case["G"], k=k, v=v)
    if kind == "codec":
        _, codec, _ = _family(case)
        x = _keys(g, case["B"], case["H"], case["S"], case["D"], dtype=case["dtype"])
        return dict(kind=kind, codec=codec, x=x, G=case["G"], D=case["D"])
    if kind == "attend":
        _, codec, attend = _family(case)
        q, k, v = _attend_inputs(case, g)
        kw = dict(group_size=case["G"], is_causal=case["causal"])
        if case["family"] == "llama3":
            kw.update(n_q_heads=case["Hq"], n_kv_heads=case["Hkv"])
        return dict(kind=kind, attend=attend, q=q, kv=(*codec.quantize_int4(k, case["G"]),
                                                       *codec.quantize_int4(v, case["G"])), kw=kw)
    return _prepare_model(case, g)


def _attend_inputs(case, g):
    q = _randn(g, case["B"], case["Hq"], case["Sq"], case["D"], dtype=case["dtype"])
    k = _keys(g, case["B"], case["Hkv"], case["Sk"], case["D"], dtype=case["dtype"])
    v = _randn(g, case["B"], case["Hkv"], case["Sk"], case["D"], dtype=case["dtype"])
    return q, k, v


def _prepare_token(case, g, seed, ops):
    """One decode token through the layers, captured once: the buffers hold ctx + 1 rows per sequence, and every
    replay writes the new token to the row after each sequence's last and attends over it too."""
    L, B, Hkv, D, G, ctx = case["layers"], case["B"], case["Hkv"], case["D"], case["G"], case["ctx"]
    sd = _scale_dtype(case)
    W, NG = ops.packed_width(D, G), ops.num_groups(D, G)
    kp, vp = (torch.zeros(L, B, Hkv, ctx + 1, W, dtype=torch.uint8, device="cuda") for _ in range(2))
    ks, vs = (torch.zeros(L, B, Hkv, ctx + 1, NG, dtype=sd, device="cuda") for _ in range(2))
    q = torch.empty(L, B, case["Hq"], 1, D, dtype=DT[case["dtype"]], device="cuda")
    kn = torch.empty(L, B, Hkv, 1, D, dtype=DT[case["dtype"]], device="cuda")
    vn, out = torch.empty_like(kn), torch.empty_like(q)
    for i in range(L):
        q[i], k, v, kn[i], vn[i] = _step_inputs(case, g, ctx)
        ops.quantize_into(k, kp[i], ks[i], G, 0)
        ops.quantize_into(v, vp[i], vs[i], G, 0)
    pos = _lengths(case, seed).to("cuda", torch.int32) if case["ragged"] else ctx
    # the graph's own split workspace, as the graph decoder keeps one
    ws = torch.zeros(ops.decode_workspace_bytes(B, case["Hq"], Hkv, D, q.dtype, sd), dtype=torch.uint8, device="cuda")

    def step():
        for i in range(L):
            ops.decode_step(q[i], kn[i], vn[i], kp[i], ks[i], vp[i], vs[i], pos, n_kv_heads=Hkv, group_size=G,
                            sm_scale=D ** -0.5, out=out[i])

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with ops.using_workspace(ws):
        with torch.cuda.stream(side):
            step()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            step()
    return dict(kind="token", graph=graph, ws=ws, q=q, kn=kn, vn=vn, pos=pos, out=dict(out=out, kp=kp, ks=ks, vp=vp, vs=vs))


def _prepare_model(case, g):
    from transformers import LlamaConfig, LlamaForCausalLM

    from kvint4.llama3.kv_cache import QuantizedKVCache
    from kvint4.llama3.llama3_quant import replace_llama_attention_with_quantized

    cfg = LlamaConfig(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["inter"],
                      num_hidden_layers=case["layers"], num_attention_heads=case["Hq"], num_key_value_heads=case["Hkv"],
                      head_dim=case["D"], rope_theta=THETA, max_position_embeddings=131072, rms_norm_eps=EPS,
                      tie_word_embeddings=False)
    with torch.device("meta"):
        model = LlamaForCausalLM(cfg).to(torch.bfloat16).eval()
    w = _model_weights(case, g)

    def put(module, t):
        module.weight = torch.nn.Parameter(t, requires_grad=False)

    put(model.model.embed_tokens, w["embed"])
    put(model.lm_head, w["head"])
    ones = torch.ones(case["hidden"], dtype=torch.bfloat16, device="cuda")
    put(model.model.norm, ones)
    for layer, lw in zip(model.model.layers, w["layers"]):
        for n in "qkvo":
            put(getattr(layer.self_attn, n + "_proj"), lw[n])
        for n in ("gate", "up", "down"):
            put(getattr(layer.mlp, n + "_proj"), lw[n])
        put(layer.input_layernorm, ones)
        put(layer.post_attention_layernorm, ones)
    with torch.device("cuda"):
        model.model.rotary_emb = type(model.model.rotary_emb)(config=cfg)
    model.set_attn_implementation("sdpa")
    replace_llama_attention_with_quantized(model, group_size=case["G"])
    kv, tok = _model_inputs(case, g)
    cache = QuantizedKVCache(group_size=case["G"], reserve_tokens=case["ctx"] + 64)
    for i, (k, v) in enumerate(kv):
        cache.append(k, v, i)
    return dict(kind="model", model=model, cache=cache, tok=tok)


def run(state):
    kind = state["kind"]
    if kind == "step":
        cache = state["cache"]
        out = cache.append_and_attend(state["q"], state["kn"], state["vn"], 0, n_kv_heads=state["H"],
                                      scale=state["scale"])
        cache.crop(-1)
        return [out, *state["views"]]
    if kind == "token":
        state["graph"].replay()
        return state["out"]
    if kind == "paged":
        from kvint4 import ops

        out = ops.decode_step_paged(state["q"], state["kn"], state["vn"], *state["pools"], state["table"], state["pos"],
                                    n_kv_heads=state["H"], group_size=state["G"], sm_scale=state["scale"])
        return [out, *state["pools"]]
    if kind == "append":
        cache = state["cls"](group_size=state["G"])
        cache.append(state["k"], state["v"], 0)
        return list(cache.get_quantized(0))
    if kind == "codec":
        packed, scales = state["codec"].quantize_int4(state["x"], state["G"])
        return [packed, scales, state["codec"].dequantize_int4(packed, scales, state["G"], d_head=state["D"])]
    if kind == "attend":
        return state["attend"](state["q"], *state["kv"], **state["kw"])
    with torch.no_grad():
        out = state["model"](input_ids=state["tok"], past_key_values=state["cache"], use_cache=True, logits_to_keep=1)
    state["cache"].crop(-1)
    return out.logits


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _cache_bytes(case, tokens):
    """Codes and scales of `tokens` tokens, K and V, all KV heads."""
    ng = -(-case["D"] // case["G"])
    sz = 4 if _scale_dtype(case) == torch.float32 else 2
    return 2 * case["Hkv"] * tokens * (ng * ((case["G"] + 1) // 2) + ng * sz)


def work(case):
    kind = case["kind"]
    if kind in ("step", "token", "paged"):
        ragged = kind == "paged" or case.get("ragged", False)
        # a ragged batch's lengths vary with the seed: their mean over the logarithm of [ctx / 64, ctx]
        per = case["ctx"] * (1 - 1 / 64) / math.log(64) if ragged else case["ctx"]
        tokens = int(case["B"] * per)
        io = case["B"] * (2 * case["Hq"] + 2 * case["Hkv"]) * case["D"] * _size(case["dtype"])
        n = case.get("layers", 1)
        return {"bytes": n * (_cache_bytes(case, tokens + case["B"]) + io), "flops": n * 4.0 * case["Hq"] * tokens * case["D"]}
    if kind == "append":
        n = case["B"] * case["S"]
        return {"bytes": 2 * n * case["Hkv"] * case["D"] * _size(case["dtype"]) + _cache_bytes(case, n), "flops": 0}
    if kind == "codec":
        n = case["B"] * case["H"] * case["S"]
        ng = -(-case["D"] // case["G"])
        ssz = 2 if case["family"] == "gpt2" else _size(case["dtype"])
        osz = 2 if case["family"] == "gpt2" else _size(case["dtype"])
        packed = n * ng * ((case["G"] + 1) // 2 + ssz)
        return {"bytes": n * case["D"] * (_size(case["dtype"]) + osz) + 2 * packed, "flops": 0}
    if kind == "attend":
        Sq, Sk = case["Sq"], case["Sk"]
        pairs = Sq * (Sk - Sq) + Sq * (Sq + 1) // 2 if case["causal"] else Sq * Sk
        io = 2 * case["B"] * case["Hq"] * Sq * case["D"] * _size(case["dtype"])
        return {"bytes": _cache_bytes(case, case["B"] * Sk) + io, "flops": 4.0 * case["B"] * case["Hq"] * pairs * case["D"]}
    H, D = case["hidden"], case["D"]
    per = H * D * 2 * (case["Hq"] + case["Hkv"]) + 3 * H * case["inter"]
    weights = 2 * (case["layers"] * per + case["vocab"] * H)
    return {"bytes": weights + case["layers"] * _cache_bytes(case, case["ctx"]), "flops": weights}


def tolerance(case):
    """About four times the distance to the 64-bit result that was measured: 2e-3 for bf16 decoding and 2.3e-4 for fp16
    (the output's rounding and the softmax weights'), 6e-3 and 8.5e-4 for long query blocks (K and V rounded to 16 bits
    after dequantization as well), 1.2e-6 in fp32; a model adds the 16-bit rounding of every activation."""
    if case["kind"] in ("append", "codec"):
        return "exact"
    if case["kind"] == "model":
        return {"rel": 3e-2, "max": 0.3}
    if case["kind"] == "attend":
        return {"bf16": {"rel": 2e-2, "max": 0.2}, "f16": {"rel": 3e-3, "max": 3e-2}, "f32": {"rel": 1e-5, "max": 1e-4}}[case["dtype"]]
    return {"bf16": {"rel": 1e-2, "max": 0.1}, "f16": {"rel": 1e-3, "max": 1e-2}, "f32": {"rel": 1e-5, "max": 1e-4}}[case["dtype"]]


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch


def _codes(x, G, scale_dtype):
    """Codes (-8 .. 7) [.., ng, G] and stored scales [.., ng] of the symmetric INT4 format: scale = max|x| / 7 in
    fp32 (1 for an all-zero group), code = round_half_even(x / scale), the scale then rounded for storage."""
    D = x.shape[-1]
    ng = -(-D // G)
    xf = torch.nn.functional.pad(x.float(), (0, ng * G - D)).unflatten(-1, (ng, G))
    am = xf.abs().amax(-1)
    s = torch.where(am > 0, am / torch.full_like(am, 7.0), torch.ones_like(am))  # a true division, as the format says
    c = torch.round(xf / s.unsqueeze(-1)).clamp(-8, 7)
    return c, s.to(scale_dtype)


def _dequant64(x, G, scale_dtype):
    c, s = _codes(x, G, scale_dtype)
    return (c.double() * s.double().unsqueeze(-1)).flatten(-2)[..., : x.shape[-1]]


def _pack(c):
    n = (c + 8).to(torch.uint8).flatten(-2)
    return n[..., 0::2] | (n[..., 1::2] << 4)


def _attend64(q, k, v, scale, causal, lens=None):
    """q [B, Hq, Sq, D], k and v [B, Hkv, Sk, D] in 64 bits; causal masks aligned to each sequence's end."""
    B, Hq, Sq, D = q.shape
    Hkv, Sk = k.shape[1], k.shape[2]
    out = torch.empty(B, Hq, Sq, D, dtype=torch.float64, device=q.device)
    for b in range(B):
        n = Sk if lens is None else int(lens[b])
        for h in range(Hq):
            kv = h // (Hq // Hkv)
            kk, vv = k[b, kv, :n], v[b, kv, :n]
            for lo in range(0, Sq, 4096):
                qq = q[b, h, lo:lo + 4096].double()
                s = (qq @ kk.T.contiguous()) * scale
                if causal:
                    i = torch.arange(lo, lo + qq.shape[0], device=q.device)[:, None]
                    s = s.masked_fill(torch.arange(n, device=q.device)[None] > n - Sq + i, -math.inf)
                out[b, h, lo:lo + 4096] = torch.softmax(s, -1) @ vv
    return out


def _step64(case, q, k, v, kn, vn, lens):
    """The decode step's output: attention over each sequence's cached rows and its new one."""
    sd, G, B = _scale_dtype(case), case["G"], q.shape[0]
    outs = []
    for b in range(B):
        n = int(lens[b])
        kk = torch.cat((k[b:b + 1, :, :n], kn[b:b + 1]), 2)
        vv = torch.cat((v[b:b + 1, :, :n], vn[b:b + 1]), 2)
        outs.append(_attend64(q[b:b + 1], _dequant64(kk, G, sd), _dequant64(vv, G, sd), case["D"] ** -0.5, False))
    return torch.cat(outs)


def exact(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "step":
        q, k, v, kn, vn = _step_inputs(case, g, case["ctx"])
        sd = _scale_dtype(case)
        rows = []
        for old, new in ((k, kn), (v, vn)):
            c, s = _codes(torch.cat((old, new), 2), case["G"], sd)
            rows += [_pack(c), s]
        return [_step64(case, q, k, v, kn, vn, [case["ctx"]] * case["B"]), *rows]
    if kind == "paged":
        lens = _lengths(case, seed)
        return [_step64(case, *_step_inputs(case, g, case["ctx"]), lens), None, None, None, None]
    if kind == "token":
        lens = _lengths(case, seed) if case["ragged"] else [case["ctx"]] * case["B"]
        out = torch.stack([_step64(case, *_step_inputs(case, g, case["ctx"]), lens) for _ in range(case["layers"])])
        return dict(out=out, kp=None, ks=None, vp=None, vs=None)
    if kind == "append":
        k = _keys(g, case["B"], case["S"], case["Hkv"], case["D"], dtype=case["dtype"]).transpose(1, 2)
        v = _randn(g, case["B"], case["S"], case["Hkv"], case["D"], dtype=case["dtype"]).transpose(1, 2)
        rows = []
        for x in (k, v):
            c, s = _codes(x, case["G"], _scale_dtype(case))
            rows += [_pack(c), s]
        return rows
    if kind == "codec":
        x = _keys(g, case["B"], case["H"], case["S"], case["D"], dtype=case["dtype"])
        sd = torch.float16 if case["family"] == "gpt2" else DT[case["dtype"]]
        c, s = _codes(x, case["G"], sd)
        return [_pack(c), s, _dequant64(x, case["G"], sd)]
    if kind == "attend":
        q, k, v = _attend_inputs(case, g)
        sd = _scale_dtype(case)
        return _attend64(q, _dequant64(k, case["G"], sd), _dequant64(v, case["G"], sd), case["D"] ** -0.5, case["causal"])
    w = _model_weights(case, g)
    kv, tok = _model_inputs(case, g)
    D, sd = case["D"], torch.bfloat16

    def norm(x):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)

    def heads(x, n):
        return x.view(1, 1, n, D).transpose(1, 2)

    x = w["embed"][tok[0]].double()
    for lw, (k, v) in zip(w["layers"], kv):
        h = norm(x)
        q = _rope(heads(h @ lw["q"].double().T, case["Hq"]), case["ctx"], THETA)
        kn = _rope(heads(h @ lw["k"].double().T, case["Hkv"]), case["ctx"], THETA)
        vn = heads(h @ lw["v"].double().T, case["Hkv"])
        kk = torch.cat((_dequant64(k, case["G"], sd), _dequant64(kn.bfloat16(), case["G"], sd)), 2)
        vv = torch.cat((_dequant64(v, case["G"], sd), _dequant64(vn.bfloat16(), case["G"], sd)), 2)
        a = _attend64(q, kk, vv, D ** -0.5, False)
        x = x + a.transpose(1, 2).reshape(1, -1) @ lw["o"].double().T
        h = norm(x)
        u = torch.nn.functional.silu(h @ lw["gate"].double().T) * (h @ lw["up"].double().T)
        x = x + u @ lw["down"].double().T
    return (norm(x) @ w["head"].double().T)[None]
