"""GPU parity of the staged prefill route (long query blocks whose K and V are
dequantized once, in matrix-operand order, into the workspace) with the
unstaged kernel, which the same C entry point runs when it gets no workspace.

Both dequantize with the same rounding, so they differ in the order of fp32
sums and in which power of two a softmax weight is rounded under. Bars: the
file's 2e-2 against float64 attention over the cache, and a root mean square
error no more than 1.1 times the unstaged kernel's (its own spread over
inputs is under 2 %).

Sizes: key counts around tile (64) and row counts around wave and workgroup
(32, 128, 256) boundaries, odd and even tile counts (the pipelined loop takes
tiles in pairs), one tile, more queries than keys, GQA 1/4/8, D 64/128, G
32/64/128, both types, negative and zero softmax scales; and the forms of
arguments the route accepts: views of larger caches, [B, S, H, D] queries,
unaligned query and code rows, pools with missing pages.
"""

from __future__ import annotations

import pytest
import torch

from kvint4 import _native as nat
from kvint4 import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TDT = {"bf16": torch.bfloat16, "f16": torch.float16}


def _dequant64(p, s, G, D):
    n = torch.stack((p & 15, p >> 4), -1).flatten(-2).double() - 8
    return n[..., :D] * s.double().repeat_interleave(G, -1)[..., :D]


def _want(q, k, v, scale, causal):
    """float64 attention, k and v [B, Hkv, Sk, D] in float64."""
    B, Hq, Sq, D = q.shape
    Sk, ratio = k.shape[2], Hq // k.shape[1]
    out = torch.zeros(B, Hq, Sq, D, dtype=torch.float64, device=q.device)
    i, j = torch.arange(Sq, device=q.device)[:, None], torch.arange(Sk, device=q.device)[None]
    for b in range(B):
        for h in range(Hq):
            s = q[b, h].double() @ k[b, h // ratio].T.contiguous() * scale
            if causal:
                s = s.masked_fill(j > Sk - Sq + i, float("-inf"))
            out[b, h] = torch.nan_to_num(torch.softmax(s, -1)) @ v[b, h // ratio]
    return out


def _call(q, kp, ks, vp, vs, Hkv, G, causal, scale, staged, pt=None, seq_len=None):
    """kvq_prefill_attn (or _paged) with the staged route's workspace, or with none."""
    B, Hq, Sq, D = q.shape
    Sk = kp.shape[2] if pt is None else seq_len
    out = torch.full_like(q, float("nan"))
    lib = nat.lib()
    n = lib.kvq_prefill_attn_staged_workspace_bytes(B, Hq, Hkv, Sq, D, Sk)
    images = B * Hkv * -(-Sk // 64) * D * 256
    assert n >= min(images, 1 << 20), "this shape is not staged"
    ws = torch.full((n,), 255, dtype=torch.uint8, device=DEV) if staged else None  # NaN bits in every piece
    dt, sd = nat.DTYPE_CODE[q.dtype], nat.DTYPE_CODE[ks.dtype]
    st = torch.cuda.current_stream().cuda_stream
    tail = (1 if causal else 0, float(scale), ws.data_ptr() if staged else None, n if staged else 0, st)
    if pt is None:
        rc = lib.kvq_prefill_attn(
            q.data_ptr(), dt, nat.i64_array(q.stride()), kp.data_ptr(), nat.i64_array(kp.stride()[:3]), ks.data_ptr(),
            nat.i64_array(ks.stride()[:3]), vp.data_ptr(), nat.i64_array(vp.stride()[:3]), vs.data_ptr(),
            nat.i64_array(vs.stride()[:3]), sd, out.data_ptr(), nat.i64_array(out.stride()), B, Hq, Hkv, Sq, D, G, Sk,
            *tail)
    else:
        rc = lib.kvq_prefill_attn_paged(
            q.data_ptr(), dt, nat.i64_array(q.stride()), kp.data_ptr(), nat.i64_array(kp.stride()[:2]), ks.data_ptr(),
            nat.i64_array(ks.stride()[:2]), vp.data_ptr(), nat.i64_array(vp.stride()[:2]), vs.data_ptr(),
            nat.i64_array(vs.stride()[:2]), sd, *pt.args(), out.data_ptr(), nat.i64_array(out.stride()), B, Hq, Hkv, Sq,
            D, G, Sk, *tail)
    nat.check(rc, "kvq_prefill_attn")
    return out


def _compare(q, kp, ks, vp, vs, Hkv, G, causal, scale, want, **kw):
    a = _call(q, kp, ks, vp, vs, Hkv, G, causal, scale, True, **kw)
    b = _call(q, kp, ks, vp, vs, Hkv, G, causal, scale, False, **kw)
    ea, eb = (a.double() - want), (b.double() - want)
    assert torch.isfinite(a).all()
    print(f"staged max-abs {ea.abs().max().item():.2e} rms {ea.square().mean().sqrt().item():.2e}; "
          f"unstaged {eb.abs().max().item():.2e} rms {eb.square().mean().sqrt().item():.2e}", flush=True)
    assert ea.abs().max().item() <= 2e-2
    assert ea.square().mean().sqrt().item() <= 1.1 * eb.square().mean().sqrt().item() + 1e-12


def _quantized(B, Hkv, Sk, D, dtype, G, g, cap=0, pad=0):
    """Codes and scales of random K and V: views of the first Sk rows of `cap` rows, `pad` spare bytes per code row."""
    t, out = TDT[dtype], []
    for _ in range(2):
        p, s = ops.quantize(torch.randn(B, Hkv, max(Sk, cap), D, generator=g, device=DEV).to(t), G, t)
        if pad:
            wide = torch.zeros(*p.shape[:-1], p.shape[-1] + pad, dtype=torch.uint8, device=DEV)
            wide[..., pad:] = p
            p = wide[..., pad:]
        out += [p[:, :, :Sk], s[:, :, :Sk]]
    return out


CASES = [
    # B, Hq, Hkv, Sq, Sk, D, G, dtype, causal, scale
    (1, 32, 8, 512, 1025, 128, 32, "bf16", True, None),    # 17 tiles: an odd count, the last with one key
    (1, 32, 8, 520, 1088, 128, 32, "f16", True, None),     # 17 tiles, the last row block of 32 rows
    (1, 32, 8, 4096, 128, 128, 32, "bf16", False, None),   # two tiles, eight waves per workgroup
    (1, 32, 8, 8200, 64, 128, 64, "bf16", False, None),    # one tile; a last row block of 32 rows
    (1, 32, 8, 8192, 70, 128, 32, "bf16", True, None),     # most rows have no key: zeros
    (2, 64, 8, 250, 1100, 128, 128, "bf16", True, None),   # GQA 8, G 128
    (1, 12, 12, 1500, 1500, 64, 32, "f16", True, None),    # MHA, D 64
    (3, 16, 4, 333, 4100, 64, 64, "bf16", True, None),     # D 64, a split over keys
    (1, 4, 1, 777, 9001, 128, 32, "f16", True, None),      # few units: split over keys
    (1, 32, 8, 600, 1200, 128, 32, "bf16", True, -0.09),   # negative scale
    (1, 32, 8, 600, 1200, 128, 32, "bf16", True, 0.0),     # every key alike
]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,G,dtype,causal,scale", CASES)
def test_staged_matches_unstaged(B, Hq, Hkv, Sq, Sk, D, G, dtype, causal, scale):
    g = torch.Generator(device=DEV).manual_seed(Sq + Sk)
    q = torch.randn(B, Hq, Sq, D, generator=g, device=DEV).to(TDT[dtype])
    kp, ks, vp, vs = _quantized(B, Hkv, Sk, D, dtype, G, g, cap=Sk + 37)
    scale = D ** -0.5 if scale is None else scale
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), scale, causal)
    _compare(q, kp, ks, vp, vs, Hkv, G, causal, scale, want)


@pytest.mark.parametrize("form", ["bshd", "odd_query", "odd_codes"])
def test_staged_argument_forms(form):
    """[B, S, H, D] queries; query rows one element off 16-byte alignment; code rows three bytes off."""
    B, Hq, Hkv, Sq, Sk, D, G = 1, 32, 8, 520, 1100, 128, 32
    g = torch.Generator(device=DEV).manual_seed(7)
    if form == "bshd":
        q = torch.randn(B, Sq, Hq, D, generator=g, device=DEV).to(torch.bfloat16).transpose(1, 2)
    elif form == "odd_query":
        q = torch.randn(B, Hq, Sq, D + 1, generator=g, device=DEV).to(torch.bfloat16)[..., 1:]
    else:
        q = torch.randn(B, Hq, Sq, D, generator=g, device=DEV).to(torch.bfloat16)
    kp, ks, vp, vs = _quantized(B, Hkv, Sk, D, "bf16", G, g, pad=3 if form == "odd_codes" else 0)
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), D ** -0.5, True)
    a = _call(q, kp, ks, vp, vs, Hkv, G, True, D ** -0.5, True)
    assert (a.double() - want).abs().max().item() <= 2e-2


def test_staged_paged_with_missing_pages():
    """A permuted block table, one page of which has no block (its keys read as zeros and are attended as such by both
    kernels), sequence end inside a page."""
    B, Hq, Hkv, Sq, Sk, D, G, P = 2, 32, 8, 300, 1500, 128, 32, 128
    g = torch.Generator(device=DEV).manual_seed(9)
    q = torch.randn(B, Hq, Sq, D, generator=g, device=DEV).to(torch.bfloat16)
    cols = -(-Sk // P)
    nb = B * cols + 3
    pools = _quantized(1, Hkv, nb * P, D, "bf16", G, g)
    kp, ks, vp, vs = (t[0] for t in pools)
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(1))[: B * cols].view(B, cols).to(DEV, torch.int32)
    table[1, 3] = -1
    pt = ops.PageTable(table, P, nb)
    t = torch.arange(Sk, device=DEV)
    rows = table[:, t // P].long() * P + t % P
    hole = rows < 0
    k, v = (_dequant64(p, s, G, D)[:, rows.clamp(min=0)].transpose(0, 1) * ~hole[:, None, :, None] for p, s in ((kp, ks), (vp, vs)))
    want = _want(q, k, v, D ** -0.5, True)
    _compare(q, kp, ks, vp, vs, Hkv, G, True, D ** -0.5, want, pt=pt, seq_len=Sk)


def test_staged_units_in_groups():
    """Images of more than 256 MiB run in groups of units through one workspace: 40 units of 16K keys (8 MiB each) in
    groups of 31 and 9."""
    B, Hq, Hkv, Sq, Sk, D, G = 5, 8, 8, 256, 16448, 128, 32
    g = torch.Generator(device=DEV).manual_seed(11)
    n = nat.lib().kvq_prefill_attn_staged_workspace_bytes(B, Hq, Hkv, Sq, D, Sk)
    assert n < (256 << 20) + (64 << 20)
    q = torch.randn(B, Hq, Sq, D, generator=g, device=DEV).to(torch.bfloat16)
    kp, ks, vp, vs = _quantized(B, Hkv, Sk, D, "bf16", G, g)
    a = _call(q, kp, ks, vp, vs, Hkv, G, True, D ** -0.5, True)
    b = _call(q, kp, ks, vp, vs, Hkv, G, True, D ** -0.5, False)
    # outputs average thousands of values (|out| < 0.2): two bf16 roundings of them and of the weights
    assert (a.float() - b.float()).abs().max().item() <= 2e-3


def _attended(q, Sk, ratio, bad, causal):
    """[Sq]: whether a query position attends key `bad`."""
    i = torch.arange(q.shape[2], device=DEV)
    return (Sk - q.shape[2] + i >= bad) if causal else torch.ones_like(i, dtype=torch.bool)


@pytest.mark.parametrize("what,value", [("key", float("nan")), ("key", float("inf")), ("value", float("nan")),
                                        ("value", float("inf")), ("value", float("-inf"))])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,dtype,bad", [
    (1, 32, 8, 2048, 2048, 128, "bf16", 1000),   # eight waves per workgroup
    (1, 32, 8, 530, 1088, 128, "f16", 700),      # four; the key's tile begins in the second half of their rows
    (4, 16, 16, 1030, 1030, 64, "bf16", 700),    # MHA, D 64, eight waves; the same
    (1, 4, 1, 777, 9001, 128, "f16", 8500),      # a split over keys
])
def test_staged_non_finite_scales(what, value, B, Hq, Hkv, Sq, Sk, D, dtype, bad):
    """One key with a scale that is not finite: its rows' outputs are not finite, as on the unstaged kernel, and every
    row that the unstaged kernel keeps finite (a wave's masked keys share matrix products with the rows before them, in
    both kernels) stays finite and right."""
    G, ratio = 32, Hq // Hkv
    g = torch.Generator(device=DEV).manual_seed(Sk + bad)
    q = torch.randn(B, Hq, Sq, D, generator=g, device=DEV).to(TDT[dtype])
    kp, ks, vp, vs = _quantized(B, Hkv, Sk, D, dtype, G, g)
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), D ** -0.5, True)
    (ks if what == "key" else vs)[:, :, bad] = value
    a = _call(q, kp, ks, vp, vs, Hkv, G, True, D ** -0.5, True)
    b = _call(q, kp, ks, vp, vs, Hkv, G, True, D ** -0.5, False)
    fa, fb = torch.isfinite(a).all(-1), torch.isfinite(b).all(-1)
    attends = _attended(q, Sk, ratio, bad, True)
    print(f"rows that attend the key {attends.sum().item()}, not finite: staged {(~fa[0, 0]).sum().item()}, "
          f"unstaged {(~fb[0, 0]).sum().item()}", flush=True)
    assert not fa[:, :, attends].any() and not fb[:, :, attends].any()
    assert fa[fb].all()
    assert fa[:, :, ~attends].any()
    assert (a.double() - want).abs()[fa].max().item() <= 2e-2


def test_staged_largest_scales():
    """Key scales above 2^125 (-8 times them overflows) under small queries and a small softmax scale."""
    B, Hq, Hkv, Sq, Sk, D, G = 1, 32, 8, 520, 1088, 128, 32
    g = torch.Generator(device=DEV).manual_seed(3)
    q = (torch.randn(B, Hq, Sq, D, generator=g, device=DEV) * 1e-10).bfloat16()
    kp, ks, vp, vs = _quantized(B, Hkv, Sk, D, "bf16", G, g)
    kp, ks = ops.quantize((torch.randn(B, Hkv, Sk, D, generator=g, device=DEV).clamp(-3, 3) * 1.1e38).bfloat16(), G,
                          torch.bfloat16)
    assert ks.float().max().item() > 2.0 ** 125
    want = _want(q, _dequant64(kp, ks, G, D), _dequant64(vp, vs, G, D), 8e-30, True)
    _compare(q, kp, ks, vp, vs, Hkv, G, True, 8e-30, want)


def test_staged_long_blocks_in_groups():
    """Units in groups (31 and 9 of 40) with eight waves per workgroup: 2048 rows over 16448 keys."""
    B, Hq, Hkv, Sq, Sk, D, G = 5, 32, 8, 512, 16448, 128, 32
    g = torch.Generator(device=DEV).manual_seed(13)
    shape = (B, Hq, Hkv, Sq, D, Sk)
    n = nat.lib().kvq_prefill_attn_staged_workspace_bytes(*shape)
    assert (200 << 20) < n < (320 << 20) and n > nat.lib().kvq_prefill_attn_workspace_bytes(*shape)
    q = torch.randn(B, Hq, Sq, D, generator=g, device=DEV).to(torch.bfloat16)
    kp, ks, vp, vs = _quantized(B, Hkv, Sk, D, "bf16", G, g)
    a = _call(q, kp, ks, vp, vs, Hkv, G, True, D ** -0.5, True)
    b = _call(q, kp, ks, vp, vs, Hkv, G, True, D ** -0.5, False)
    # outputs average thousands of values (|out| < 0.2): two bf16 roundings of them and of the weights
    assert (a.float() - b.float()).abs().max().item() <= 2e-3
