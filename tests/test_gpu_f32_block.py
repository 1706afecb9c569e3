"""GPU parity: fp32 query blocks on the 16-row fp32 matrix kernel of
kvq_decode_attn (blocks of enough rows; smaller ones stay on the VALU kernel)
against float64 attention over the cache.

Bar: 1e-4 max-abs, the repository's for fp32 inputs, and 2e-6 relative to the
outputs' norm: fp32 products and sums of up to a thousand terms (the VALU
kernel measures 1.2e-6 on a 1000-token prompt). The same call with two splits
asked for runs the VALU kernel, whose output must agree within 2e-5.

Sizes: row counts that are no multiple of 16, chunks that span two heads, key
counts around the 64-key tile, more queries than keys, per-sequence lengths
(zero, shorter than the block), GQA, both head dims, every group size and scale
type, strided and unaligned queries, pages without a block.
"""

from __future__ import annotations

import pytest
import torch

from kvint4 import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
SDT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _dequant64(p, s, G, D):
    n = torch.stack((p & 15, p >> 4), -1).flatten(-2).double() - 8
    return n[..., :D] * s.double().repeat_interleave(G, -1)[..., :D]


def _want(q, k, v, scale, causal, lens=None):
    B, Hq, Sq, D = q.shape
    Sk, ratio = k.shape[2], Hq // k.shape[1]
    out = torch.zeros(B, Hq, Sq, D, dtype=torch.float64, device=q.device)
    i, j = torch.arange(Sq, device=q.device)[:, None], torch.arange(Sk, device=q.device)[None]
    for b in range(B):
        n = Sk if lens is None else int(lens[b])
        ok = j < n if not causal else (j < n) & (j <= n - Sq + i)
        ok = ok.expand(Sq, Sk)
        for h in range(Hq):
            s = (q[b, h].double() @ k[b, h // ratio].T.contiguous() * scale).masked_fill(~ok, float("-inf"))
            out[b, h] = torch.nan_to_num(torch.softmax(s, -1)) @ v[b, h // ratio]
    return out


def _kv(B, Hkv, Sk, D, G, sd, g):
    out = []
    for _ in range(2):
        p, s = ops.quantize(torch.randn(B, Hkv, Sk, D, generator=g, device=DEV), G, SDT[sd])
        out += [p, s]
    return out


def _check(out, want):
    assert torch.isfinite(out).all()
    d = out.double() - want
    assert d.abs().max().item() <= 1e-4
    assert d.norm().item() <= 2e-6 * want.norm().item()


CASES = [
    # B, Hq, Hkv, Sq, Sk, D, G, scales, causal
    (1, 12, 12, 100, 100, 64, 32, "f16", True),     # 6 chunks and 4 rows per head
    (2, 12, 3, 37, 129, 64, 64, "f16", True),       # GQA 4: a chunk spans two query heads; one key past two tiles
    (1, 16, 4, 50, 700, 128, 32, "f32", True),      # below the line for D = 128 (VALU kernel) ...
    (1, 16, 4, 90, 700, 128, 32, "f32", True),      # ... and above it
    (1, 8, 8, 300, 64, 128, 128, "bf16", False),    # one tile exactly
    (1, 12, 12, 90, 63, 64, 32, "f16", True),       # more queries than keys: rows without a key are zeros
    (1, 12, 12, 100, 1030, 64, 32, "f16", True),    # 17 tiles
    (3, 4, 4, 200, 513, 64, 64, "f32", False),
]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,G,sd,causal", CASES)
def test_f32_block_matches_oracle_and_valu(B, Hq, Hkv, Sq, Sk, D, G, sd, causal):
    g = torch.Generator(device=DEV).manual_seed(Sq * Sk)
    q = torch.randn(B, Hq, Sq, D, generator=g, device=DEV)
    kp, ks, vp, vs = _kv(B, Hkv, Sk, D, G, sd, g)
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), D ** -0.5, causal)
    kw = dict(n_kv_heads=Hkv, group_size=G, is_causal=causal, sm_scale=D ** -0.5)
    out = ops.fused_decode_attention(q, kp, ks, vp, vs, **kw)
    _check(out, want)
    if Sk >= 256 and B * Hkv * (Hq // Hkv) * Sq <= 2048:  # split plans hold at most 1024 units
        valu = ops.fused_decode_attention(q, kp, ks, vp, vs, n_split=2, **kw)
        assert (out - valu).abs().max().item() <= 2e-5


@pytest.mark.parametrize("causal", [True, False])
def test_f32_block_per_sequence_lengths(causal):
    B, H, Sq, Sk, D, G = 4, 12, 40, 500, 64, 32
    g = torch.Generator(device=DEV).manual_seed(5)
    q = torch.randn(B, H, Sq, D, generator=g, device=DEV)
    kp, ks, vp, vs = _kv(B, H, Sk, D, G, "f16", g)
    lens = torch.tensor([500, 0, 17, 257], dtype=torch.int32, device=DEV)
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), D ** -0.5, causal, lens.tolist())
    out = ops.fused_decode_attention(q, kp, ks, vp, vs, n_kv_heads=H, group_size=G, is_causal=causal,
                                     sm_scale=D ** -0.5, seq_lens=lens)
    _check(out, want)
    assert torch.all(out[1] == 0)


@pytest.mark.parametrize("form", ["bshd", "odd", "strided_dim"])
def test_f32_block_query_forms(form):
    B, H, Sq, Sk, D, G = 1, 12, 100, 300, 64, 32
    g = torch.Generator(device=DEV).manual_seed(6)
    if form == "bshd":
        q = torch.randn(B, Sq, H, D, generator=g, device=DEV).transpose(1, 2)
    elif form == "odd":
        q = torch.randn(B, H, Sq, D + 1, generator=g, device=DEV)[..., 1:]
    else:
        q = torch.randn(B, H, D, Sq, generator=g, device=DEV).transpose(2, 3)
    kp, ks, vp, vs = _kv(B, H, Sk, D, G, "f16", g)
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), D ** -0.5, True)
    _check(ops.fused_decode_attention(q, kp, ks, vp, vs, n_kv_heads=H, group_size=G, is_causal=True,
                                      sm_scale=D ** -0.5), want)


def test_f32_block_paged_with_missing_page():
    """Keys of a page without a block are not attended (as in the VALU kernel)."""
    B, H, Sq, D, G, P, S = 2, 12, 60, 64, 32, 64, 400
    g = torch.Generator(device=DEV).manual_seed(8)
    q = torch.randn(B, H, Sq, D, generator=g, device=DEV)
    cols = -(-S // P)
    nb = B * cols + 2
    kp, ks, vp, vs = (t[0] for t in _kv(1, H, nb * P, D, G, "f16", g))
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(2))[: B * cols].view(B, cols).to(DEV, torch.int32)
    table[1, 2] = -1
    pt = ops.PageTable(table, P, nb)
    out = ops.fused_decode_attention_paged(q, kp, ks, vp, vs, pt, n_kv_heads=H, group_size=G, is_causal=False,
                                           sm_scale=D ** -0.5, seq_len=S)
    t = torch.arange(S, device=DEV)
    for b in range(B):
        rows = table[b, t // P].long() * P + t % P
        rows = rows[table[b, t // P] >= 0]
        want = _want(q[b:b + 1], _dequant64(kp[:, rows], ks[:, rows], G, D)[None],
                     _dequant64(vp[:, rows], vs[:, rows], G, D)[None], D ** -0.5, False)
        _check(out[b:b + 1], want)


def test_f32_block_nan_key_scale():
    """A key whose score is not a number weighs nothing and the row keeps its other keys, as on the VALU kernel."""
    B, H, Sq, Sk, D, G, bad = 1, 12, 100, 300, 64, 32, 130
    g = torch.Generator(device=DEV).manual_seed(12)
    q = torch.randn(B, H, Sq, D, generator=g, device=DEV)
    kp, ks, vp, vs = _kv(B, H, Sk, D, G, "f16", g)
    ks[:, :, bad, 1] = float("nan")
    kw = dict(n_kv_heads=H, group_size=G, is_causal=True, sm_scale=D ** -0.5)
    out = ops.fused_decode_attention(q, kp, ks, vp, vs, **kw)
    keep = [t for t in range(Sk) if t != bad]  # (a causal row before the key, too, has the same keys without it)
    want = torch.empty(B, H, Sq, D, dtype=torch.float64, device=DEV)
    k, v = _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D)
    for h in range(H):
        s = q[0, h].double() @ k[0, h][keep].T.contiguous() * D ** -0.5
        lim = Sk - Sq + torch.arange(Sq, device=DEV)[:, None]
        s = s.masked_fill(torch.tensor(keep, device=DEV)[None] > lim, float("-inf"))
        want[0, h] = torch.softmax(s, -1) @ v[0, h][keep]
    _check(out, want)
    valu = ops.fused_decode_attention(q, kp, ks, vp, vs, n_split=2, **kw)
    assert (out - valu).abs().max().item() <= 2e-5


def test_f32_block_missing_page_reads_no_pool_row():
    """A tile without a block contributes nothing whatever the pool's unused rows (row 0 among them) hold."""
    B, H, Sq, D, G, P, S = 2, 12, 60, 64, 32, 64, 400
    g = torch.Generator(device=DEV).manual_seed(14)
    q = torch.randn(B, H, Sq, D, generator=g, device=DEV)
    cols = -(-S // P)
    nb = B * cols + 2
    kp, ks, vp, vs = (t[0] for t in _kv(1, H, nb * P, D, G, "f16", g))
    table = 1 + torch.randperm(nb - 1, generator=torch.Generator().manual_seed(2))[: B * cols].view(B, cols)
    table = table.to(DEV, torch.int32)
    table[0, 0], table[1, 2], table[1, 6] = -1, -1, -1
    used = torch.zeros(nb, dtype=torch.bool, device=DEV)
    used[table[table >= 0].long()] = True
    for s in (ks, vs):
        s[:, ~used.repeat_interleave(P)] = float("nan")
    pt = ops.PageTable(table, P, nb)
    out = ops.fused_decode_attention_paged(q, kp, ks, vp, vs, pt, n_kv_heads=H, group_size=G, is_causal=False,
                                           sm_scale=D ** -0.5, seq_len=S)
    t = torch.arange(S, device=DEV)
    for b in range(B):
        rows = table[b, t // P].long() * P + t % P
        rows = rows[table[b, t // P] >= 0]
        want = _want(q[b:b + 1], _dequant64(kp[:, rows], ks[:, rows], G, D)[None],
                     _dequant64(vp[:, rows], vs[:, rows], G, D)[None], D ** -0.5, False)
        _check(out[b:b + 1], want)


@pytest.mark.parametrize("H,Sq,Sk,causal", [
    (12, 1000, 1000, True),    # 756 units: both chunk orders, the change of order inside a head's chunks
    (3, 4105, 300, False),     # a head's last chunk is unit 256: the second head starts just past it
    (3, 4105, 4200, True),
])
def test_f32_block_many_units(H, Sq, Sk, causal):
    """Launches past 256 units, where every other 256 units' heads take their chunks in the other order: each chunk is
    written once, whichever order it is taken in (the output starts as NaN)."""
    D, G = 64, 32
    g = torch.Generator(device=DEV).manual_seed(Sq + Sk)
    q = torch.randn(1, H, Sq, D, generator=g, device=DEV)
    kp, ks, vp, vs = _kv(1, H, Sk, D, G, "f16", g)
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), D ** -0.5, causal)
    out = torch.full_like(q, float("nan"))
    ops.fused_decode_attention(q, kp, ks, vp, vs, n_kv_heads=H, group_size=G, is_causal=causal, sm_scale=D ** -0.5,
                               out=out)
    _check(out, want)


@pytest.mark.parametrize("sd", ["bf16", "f32"])
def test_f32_block_largest_key_scales(sd):
    """Keys near the largest fp32 value (scales above 2^124) under small queries: a dequantized key times 16 would
    overflow, its scores do not."""
    B, H, Sq, Sk, D, G = 1, 12, 100, 300, 64, 32
    g = torch.Generator(device=DEV).manual_seed(15)
    q = torch.randn(B, H, Sq, D, generator=g, device=DEV) * 1e-38
    kp, ks = ops.quantize(torch.randn(B, H, Sk, D, generator=g, device=DEV).clamp(-3, 3) * 1.13e38, G, SDT[sd])
    vp, vs = ops.quantize(torch.randn(B, H, Sk, D, generator=g, device=DEV), G, SDT[sd])
    assert ks.float().max().item() > 2.0 ** 125
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), D ** -0.5, True)
    _check(ops.fused_decode_attention(q, kp, ks, vp, vs, n_kv_heads=H, group_size=G, is_causal=True,
                                      sm_scale=D ** -0.5), want)
