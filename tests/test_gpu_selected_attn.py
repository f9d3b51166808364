"""fused_sparse_attention on the matrix cores (gsa_selected_attn) against float64 and
against the gather kernel, whose semantics it keeps.

Bound, bf16: the weights keep 24 bits (three bf16 parts) and the sums are fp32, so an
output is within one rounding to bf16 (half an ulp, 2^-9 relative, and 2^-8 allowed
for a value at a rounding boundary) of the float64 result plus fp32 sum error of
sum_j p_j |v_j| <= max|v|, far below 2^-16 max|v|.  What those bounds leave open,
fewer bits in the weights or longer chains of fp32 sums, test_selected_attention_precision
pins.
"""

import pytest
import torch

from gsa_gdn_benchmarkstudy_amd import _abi
from oracle import gsa_oracle as orc
from gsa_gdn_benchmarkstudy_amd import gsa as G

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


def _log(msg):
    print(msg, flush=True)


def _selection(B, T, Tkv, K, seed, kind):
    """idx int64 [B,T,K] without repeats per row, mask bool."""
    g = torch.Generator().manual_seed(seed)
    r = torch.rand(B, T, Tkv, generator=g)
    if kind == "causal":
        r.masked_fill_(torch.ones(T, Tkv, dtype=torch.bool).triu_(1), -1.0)
    elif kind == "window":          # keys near 2t: the blocks' tiles start past 0 and end before the last
        d = torch.arange(Tkv)[None, :] - 2 * torch.arange(T)[:, None]
        r.masked_fill_(d.abs() > K, -1.0)
    val, idx = r.topk(K, dim=-1)
    return idx, val >= 0


def _attend64(q, k, v, idx, mask, scale):
    """Every list entry weighs once: counts of repeats multiply exp(s)."""
    B, T, H, d = q.shape
    n = torch.zeros(B, T, k.shape[1], dtype=torch.float64, device=q.device)
    n.scatter_add_(2, idx.clamp(0, k.shape[1] - 1), mask.double())
    out = torch.zeros(B, T, H, d, dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(H):
            s = (q[b, :, h].double() @ k[b, :, h].double().t().contiguous()) * scale
            s = s + torch.log(n[b])
            p = torch.softmax(s, dim=-1).nan_to_num(0.0)
            out[b, :, h] = p @ v[b, :, h].double()
    return out


def _close(out, ref, v, dtype):
    err = (out.double() - ref).abs()
    if dtype == torch.bfloat16:
        bound = ref.abs() * 2.0 ** -8 + v.abs().max().double() * 2.0 ** -16
    else:
        # fp32: scores of up to about 8 in log2 units carry 128-term dot products
        # (128 * 2^-24 relative to sum |q_i k_i|), which enter the weights linearly
        bound = ref.abs() * 2e-5 + v.abs().max().double() * 1e-5
    assert torch.all(err <= bound), float((err - bound).max())


DTYPES = [torch.bfloat16, torch.float32]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,T,Tkv,H,K,kind", [
    (1, 64, 64, 4, 64, "causal"), (2, 129, 129, 2, 80, "causal"), (1, 255, 255, 1, 100, "causal"),
    (1, 257, 257, 3, 110, "causal"), (1, 700, 700, 2, 200, "causal"), (2, 300, 1000, 2, 300, "any"),
    (1, 513, 1100, 2, 320, "window"), (1, 1000, 65, 2, 64, "any"), (1, 100, 2100, 40, 600, "any"),
])
def test_selected_attention_vs_float64(dev, dtype, B, T, Tkv, H, K, kind):
    _log(f"selected attention {dtype} B={B} T={T} Tkv={Tkv} H={H} K={K} {kind}")
    g = torch.Generator().manual_seed(T + Tkv)
    q = torch.randn(B, T, H, 128, generator=g).to(dtype).to(dev)
    kv = torch.randn(B, Tkv, 2 * H + 1, 128, generator=g).to(dtype).to(dev)   # k, v: strided views of one buffer
    k, v = kv[:, :, :H], kv[:, :, H:2 * H]
    idx, mask = _selection(B, T, Tkv, K, seed=7, kind=kind)
    idx, mask = idx.to(dev), mask.to(dev)
    assert _abi.load().gsa_selected_attn_workspace_bytes(B, T, Tkv, H, K, SCALE, _abi.dtype_code(dtype)) > 0
    out = G.fused_sparse_attention(q, k, v, idx, mask, SCALE)
    assert out.dtype == dtype and out.shape == q.shape
    ref = _attend64(q, k, v, idx, mask, SCALE)
    _close(out, ref, v, dtype)
    # another order of the same keys, 32-bit indices: the same bits
    perm = torch.randperm(K, generator=g).to(dev)
    again = G.fused_sparse_attention(q, k, v, idx[..., perm].int(), mask[..., perm], SCALE)
    assert torch.equal(again, out)


@pytest.mark.parametrize("B,T,Tkv,K,kind", [(1, 700, 700, 200, "causal"), (1, 300, 3000, 600, "any"), (2, 1100, 1100, 512, "causal")])
def test_selected_attention_precision(dev, B, T, Tkv, K, kind):
    """fp32: 3.2e-7 by 2-norm, what the gather kernel's own sums are from float64 (a score in
    four chains of 32 products comes to 2.4e-7, in one chain of 128 to 4.1e-7).  bf16: the share of outputs that are not the
    float64 result's own rounding.  An error e relative to the value makes 2 e / 2^-8 of them
    differ: fp32 sums, e about 2^-22, 1e-4; weights of two bf16 parts, e about 2^-18, 2e-3."""
    H = 2
    g = torch.Generator().manual_seed(K)
    idx, mask = (t.to(dev) for t in _selection(B, T, Tkv, K, seed=3, kind=kind))
    q, k, v = (torch.randn(B, n, H, 128, generator=g) for n in (T, Tkv, Tkv))
    for dtype in DTYPES:
        qd, kd, vd = (t.to(dtype).to(dev) for t in (q, k, v))
        assert _abi.load().gsa_selected_attn_workspace_bytes(B, T, Tkv, H, K, SCALE, _abi.dtype_code(dtype)) > 0
        out = G.fused_sparse_attention(qd, kd, vd, idx, mask, SCALE)
        ref = _attend64(qd, kd, vd, idx, mask, SCALE)
        if dtype == torch.float32:
            err = float((out.double() - ref).norm() / ref.norm())
            _log(f"precision fp32 T={T} Tkv={Tkv}: {err:.2e}")
            assert err < 3.2e-7
        else:
            share = float((out != ref.to(torch.bfloat16)).double().mean())
            _log(f"precision bf16 T={T} Tkv={Tkv}: {share:.2e} of the outputs rounded elsewhere")
            assert share < 5e-4


@pytest.mark.parametrize("dtype", DTYPES)
def test_selected_attention_rows_for_the_gather(dev, dtype):
    """Rows a bitmask cannot express, and values a masked tile cannot skip: keys listed
    twice, indices outside [0, Tkv), rows without a valid key, infinities and NaN in k
    and v (selected by some rows and not by others), products past the mask's range.
    The marked rows equal the gather kernel's bit for bit, the others the same call
    without them."""
    B, T, H, K = 1, 320, 2, 110
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(B, T, H, 128, generator=g).to(dtype) for _ in range(3))
    idx, mask = _selection(B, T, T, K, seed=5, kind="any")
    idx[0, 10, 3] = idx[0, 10, 4]                 # twice
    mask[0, 11] = False                           # no key
    idx[0, 12, 0], idx[0, 12, 1] = -5, T + 9      # clamped to 0 and T - 1
    idx[0, 13, 0] = 2 ** 32 + 17                  # counts by its low 32 bits
    qd, kd, vd, idx, mask = (t.to(dev) for t in (q, k, v, idx, mask))
    plain = G.fused_sparse_attention(qd, kd, vd, idx, mask, SCALE)
    gather = _abi.sparse_attn(qd, kd, vd, idx.to(torch.int32), SCALE, mask=mask.to(torch.uint8))
    assert torch.equal(plain[0, 10], gather[0, 10]) and torch.all(plain[0, 11] == 0)
    _close(plain, _attend64(qd, kd, vd, idx.to(torch.int32).long(), mask, SCALE), vd, dtype)

    for where, what in (("v", float("inf")), ("v", float("nan")), ("k", float("inf")), ("k", float("nan")),
                        ("k", 3e38), ("q", float("nan")), ("q", 1e30)):
        kk, vv, qq = kd.clone(), vd.clone(), qd.clone()
        {"k": kk, "v": vv, "q": qq}[where][0, 200, 1, 5] = what
        out = G.fused_sparse_attention(qq, kk, vv, idx, mask, SCALE)
        ref = _abi.sparse_attn(qq, kk, vv, idx.to(torch.int32), SCALE, mask=mask.to(torch.uint8))
        _log(f"  {where} {what}")
        assert torch.equal(torch.isfinite(out), torch.isfinite(ref))
        fin = torch.isfinite(ref)
        rtol, atol = (2.0 ** -7, 2.0 ** -14) if dtype == torch.bfloat16 else (4e-5, 2e-5)
        assert torch.allclose(out[fin].double(), ref[fin].double(), rtol=rtol, atol=atol)
        assert torch.equal(out[~fin].isnan(), ref[~fin].isnan())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,Tkv,every", [(600, 600, 1), (600, 2000, 1), (700, 700, 2), (513, 1100, 256)])
def test_selected_attention_lists_with_repeats(dev, dtype, T, Tkv, every):
    """Every list, every second one or one a block names a key twice: those rows equal the
    gather kernel's bit for bit (blocks whose rows all do compute no tile of their own), the
    others the same call without repeats."""
    _log(f"selected attention repeats {dtype} T={T} Tkv={Tkv} every={every}")
    B, H, K = 1, 2, 160
    g = torch.Generator().manual_seed(T)
    q = torch.randn(B, T, H, 128, generator=g).to(dtype).to(dev)
    k, v = (torch.randn(B, Tkv, H, 128, generator=g).to(dtype).to(dev) for _ in range(2))
    idx, mask = (t.to(dev) for t in _selection(B, T, Tkv, K, seed=11, kind="any"))
    assert _abi.load().gsa_selected_attn_workspace_bytes(B, T, Tkv, H, K, SCALE, _abi.dtype_code(dtype)) > 0
    plain = G.fused_sparse_attention(q, k, v, idx, mask, SCALE)
    idx[:, ::every, 7] = idx[:, ::every, 90]
    out = G.fused_sparse_attention(q, k, v, idx, mask, SCALE)
    gather = _abi.sparse_attn(q, k, v, idx.int(), SCALE, mask=mask)
    twice = torch.arange(T, device=dev) % every == 0
    assert torch.equal(out[:, twice], gather[:, twice])
    _close(out, _attend64(q, k, v, idx, mask, SCALE), v, dtype)
    _close(out[:, ~twice], plain[:, ~twice].double(), v, dtype)


@pytest.mark.parametrize("mtype", [torch.bool, torch.uint8, torch.int64])
def test_selected_attention_gather_sizes(dev, monkeypatch, mtype):
    """Sizes that the rule gives to the gather kernel: same bits, and a bool or byte mask goes to
    it as it is (no conversion launch)."""
    B, T, H, K = 1, 300, 2, 12
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(B, T, H, 128, generator=g).bfloat16().to(dev) for _ in range(3))
    idx, mask = (t.to(dev) for t in _selection(B, T, T, K, seed=5, kind="causal"))
    assert _abi.load().gsa_selected_attn_workspace_bytes(B, T, T, H, K, SCALE, _abi.DTYPE_BF16) == 0
    want = _abi.sparse_attn(q, k, v, idx.int(), SCALE, mask=mask.to(torch.uint8))
    seen, real = [], _abi.sparse_attn
    monkeypatch.setattr(_abi, "sparse_attn", lambda *a, mask, **kw: seen.append(mask) or real(*a, mask=mask, **kw))
    m = mask.to(mtype)
    assert torch.equal(G.fused_sparse_attention(q, k, v, idx, m, SCALE), want)
    assert mtype == torch.int64 or seen[0].data_ptr() == m.data_ptr()


@pytest.mark.parametrize("scale", [0.0, -0.5, 1e-20, 1e20])
def test_selected_attention_scales_for_the_gather(dev, scale):
    """Scales for which a masked score would not vanish take the gather kernel: same bits."""
    B, T, H, K = 1, 130, 2, 60
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(B, T, H, 128, generator=g).bfloat16().to(dev) for _ in range(3))
    idx, mask = (t.to(dev) for t in _selection(B, T, T, K, seed=5, kind="any"))
    out = G.fused_sparse_attention(q, k, v, idx, mask, scale)
    assert torch.equal(out, _abi.sparse_attn(q, k, v, idx.int(), scale, mask=mask.to(torch.uint8)))


@pytest.mark.parametrize("B,T,H,K", [(1, 64, 2, 64), (2, 129, 3, 60), (1, 257, 2, 100), (1, 700, 40, 200)])
def test_masked_attention_fp32(dev, B, T, H, K):
    """gsa_masked_attn (the fp32 layer's attention) with RoPE(q) and the output gate on
    strided views of one buffer, against float64, and a NaN and an infinity in v, which
    only the rows that select their keys may see (as the gather kernel has it)."""
    _log(f"masked attention B={B} T={T} H={H} K={K}")
    g = torch.Generator().manual_seed(T)
    buf = torch.randn(B, T, 4 * H, 128, generator=g).to(dev)
    q, k, v, og = (buf[:, :, i * H:(i + 1) * H] for i in range(4))
    cos, sin = (t.to(dev) for t in orc.RopeCache(128, torch.float32).tables(T, torch.float32))
    s = torch.rand(B, T, T, generator=g).masked_fill_(torch.ones(T, T, dtype=torch.bool).triu_(1), float("-inf"))
    idx, cnt = (t.to(dev) for t in orc.select_ascending(s, K))
    bits = _abi.selection_mask(idx, T, count=cnt)
    assert _abi.masked_attn_serves(B, T, H, K, torch.float32)
    flags = _abi.ATTN_ROPE_Q | _abi.ATTN_OUT_GATE
    out = _abi.masked_attn(q, k, v, bits, K, SCALE, og=og, cos=cos, sin=sin, flags=flags)
    qr = orc.apply_rope(q.cpu(), cos.cpu()[None, :, None], sin.cpu()[None, :, None]).to(dev)
    mask = torch.arange(K, device=dev)[None, None] < cnt[..., None]
    ref = _attend64(qr, k, v, idx.long(), mask, SCALE) * torch.sigmoid(og.double())
    _close(out, ref, v, torch.float32)
    vv = v.clone()
    vv[0, T // 2, 0, 3], vv[0, T // 3, 1, 7] = float("nan"), float("inf")
    a = _abi.masked_attn(q, k, vv, bits, K, SCALE, og=og, cos=cos, sin=sin, flags=flags)
    b = _abi.sparse_attn(q, k, vv, idx, SCALE, count=cnt, og=og, cos=cos, sin=sin, flags=flags)
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())
    fin = torch.isfinite(b)
    assert torch.allclose(a[fin], b[fin], rtol=4e-5, atol=2e-5)
