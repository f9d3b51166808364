"""The reference's module-level sub-APIs on the GPU, against the oracle.

Each test calls the drop-in API the way the reference's own code does
(gsa_triton/gsa_opt.py:143-176 ``fused_gated_indexer``, :396-401
``apply_rotary_pos_emb``, :404-429 ``RotaryEmbedding``, :434-507 the
sub-modules) and compares with the oracle on identical inputs.  Bars:
  * indexer scores within rtol 2e-5 / atol 1e-6 of the oracle's fp32 scores,
    -inf exactly above the diagonal (causal);
  * the selector's int64 indices, bool mask and k_eff equal to the oracle's
    tie-aware selector (score descending, index ascending), including the
    k_eff > 4096 path and ties;
  * gates: the sigmoid is the hardware exp2/rcp, so one bf16 ulp on a few
    elements (fp32: rtol 2e-6);
  * RoPE and the RoPE tables: bit-exact (same ops, same rounding points).
"""

import math

import pytest
import torch

from gsa_gdn_benchmarkstudy_amd import gsa as G
from oracle import gsa_oracle as orc

pytestmark = pytest.mark.gpu


def _log(msg):
    print(msg, flush=True)


def _init(mod, seed, std=0.05):
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for _, p in sorted(mod.named_parameters()):
            p.copy_(torch.randn(p.shape, generator=g) * std)
    return mod


def _scores_close(s, ref):
    assert torch.equal(torch.isinf(s), torch.isinf(ref))
    fin = torch.isfinite(ref)
    assert torch.allclose(s[fin], ref[fin], rtol=2e-5, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T", [(1, 64), (2, 301)])
def test_gated_lightning_indexer_forward(dev, dtype, B, T):
    """GatedLightningIndexer.forward(x) -> fp32 [B,T,T], -inf above the diagonal."""
    _log(f"GatedLightningIndexer.forward dtype={dtype} B={B} T={T}")
    D = 256
    m = _init(G.GatedLightningIndexer(D), seed=T).to(dev).to(dtype)
    x = torch.randn(B, T, D, generator=torch.Generator().manual_seed(1)).to(dtype).to(dev)
    with torch.no_grad():
        s = m(x).cpu()
        q = m.idx_q_proj(x).view(B, T, 4, 64).cpu()
        k = m.idx_k_proj(x).cpu()
        w = m.idx_w_proj(x).cpu()
    assert s.dtype == torch.float32 and s.shape == (B, T, T)
    ref = orc.indexer_scores(q, k, w, m.idx_bias.detach().float().cpu(), m.scale)
    _scores_close(s, ref)
    assert torch.all(torch.isinf(s) == torch.ones(T, T, dtype=torch.bool).triu(1))


@pytest.mark.parametrize("causal", [True, False])
def test_fused_gated_indexer_launcher(dev, causal):
    """fused_gated_indexer(q_idx, k_idx, w, bias, scale, causal) on strided views."""
    _log(f"fused_gated_indexer causal={causal}")
    B, T = 2, 200
    g = torch.Generator().manual_seed(4)
    buf = torch.randn(B, T, 400, generator=g).to(torch.bfloat16)
    q, k, w = buf[..., :256].view(B, T, 4, 64), buf[..., 256:320], buf[..., 320:324]
    bias = torch.randn(4, generator=g).to(torch.bfloat16)
    bd = buf.to(dev)
    s = G.fused_gated_indexer(bd[..., :256].view(B, T, 4, 64), bd[..., 256:320], bd[..., 320:324],
                              bias.to(dev), 0.125, causal=causal).cpu()
    ref = orc.indexer_scores(q, k, w, bias.float(), 0.125, causal=causal)
    _scores_close(s, ref)


def _tie_scores(B, T, levels, seed):
    g = torch.Generator().manual_seed(seed)
    s = torch.randint(0, levels, (B, T, T), generator=g).float() / levels
    return s.masked_fill(torch.triu(torch.ones(T, T, dtype=torch.bool), 1), float("-inf"))


@pytest.mark.parametrize("B,T,k_base,k_max,levels", [
    (2, 300, 64, 4096, 40),        # ties at the boundary, k_eff = 64
    (1, 100, 2048, 4096, 10**6),   # k_eff clipped to T: every causal key
    (1, 5000, 4500, 4500, 300),    # k_eff = 4500 > 4096: selection then a stable sort by score
])
def test_adaptive_topk_selector_forward(dev, B, T, k_base, k_max, levels):
    """AdaptiveTopKSelector.forward(scores) -> (int64 idx by (score desc, index asc),
    bool mask, k_eff), equal to the oracle's tie-aware selector."""
    _log(f"AdaptiveTopKSelector.forward B={B} T={T} k_base={k_base} k_max={k_max}")
    S = _tie_scores(B, T, levels, seed=T)
    sel = G.AdaptiveTopKSelector(k_base=k_base, k_min=16, k_max=k_max)
    idx, mask, k_eff = sel(S.to(dev))
    assert k_eff == orc.k_effective(k_base, k_max, T)
    assert idx.dtype == torch.int64 and mask.dtype == torch.bool
    ref_idx, ref_mask = orc.select_topk(S, k_eff)
    assert torch.equal(idx.cpu(), ref_idx)
    assert torch.equal(mask.cpu(), ref_mask)


def test_adaptive_topk_selector_forward_variance_mode(dev):
    """mode = "variance": k_t by the oracle's rule; outputs min(k_max, T) wide, the k_t
    best by (score desc, index asc) first, entries past k_t masked out."""
    B, T = 2, 400
    g = torch.Generator().manual_seed(5)
    sig = 0.2 + 1.8 * torch.rand(B, T, 1, generator=g)
    S = (torch.sigmoid(torch.randn(B, T, T, generator=g) * sig) * 4.0).masked_fill(
        torch.ones(T, T, dtype=torch.bool).triu(1), float("-inf"))
    sel = G.AdaptiveTopKSelector(k_base=64, k_min=16, k_max=160)
    sel.mode = "variance"
    idx, mask, k_eff = sel(S.to(dev))
    assert k_eff == 160
    k_rows = sel.last_k.cpu().long()
    k_orc = orc.adaptive_k(S, 64, 16, 160)
    assert torch.all((k_rows - k_orc).abs() <= 1) and (k_rows != k_orc).float().mean() <= 0.02
    ref_idx, ref_mask = orc.select_topk(S, 160)
    keep = torch.arange(160)[None, None, :] < k_rows[..., None]
    mask, idx = mask.cpu(), idx.cpu()
    assert torch.equal(mask, ref_mask & keep)
    assert torch.equal(torch.where(keep, idx, 0), torch.where(keep, ref_idx, 0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_value_and_output_gates(dev, dtype):
    """ValueGate.forward(v, x) and OutputGate.forward(o, x): t * sigmoid(W x + b)."""
    B, T, H, d = 2, 33, 4, 128
    D = H * d
    g = torch.Generator().manual_seed(6)
    x = torch.randn(B, T, D, generator=g).to(dtype).to(dev)
    v = torch.randn(B, T, H, d, generator=g).to(dtype).to(dev)
    for cls, seed in ((G.ValueGate, 7), (G.OutputGate, 8)):
        m = _init(cls(D), seed=seed, std=0.1).to(dev).to(dtype)
        with torch.no_grad():
            out = m(v, x).cpu()
            logits = m.gate_proj(x).cpu()
        ref = v.cpu() * torch.sigmoid(logits).view(B, T, H, d)
        if dtype == torch.bfloat16:
            diff = (out.float() - ref.float()).abs()
            assert (diff <= ref.float().abs() * 2 ** -7 + 1e-30).all(), cls.__name__
            assert (diff > 0).float().mean() < 2e-3, cls.__name__
        else:
            assert torch.allclose(out, ref, rtol=2e-6, atol=1e-7), cls.__name__


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_apply_rotary_pos_emb(dev, dtype):
    """apply_rotary_pos_emb(q, k, cos, sin) with the reference's broadcast tables
    [1,T,1,d] and with plain [T,d] tables: bit-exact with the oracle's ops."""
    B, T, H, d = 2, 50, 3, 128
    g = torch.Generator().manual_seed(9)
    q = torch.randn(B, T, H, d, generator=g).to(dtype)
    k = torch.randn(B, T, H, d, generator=g).to(dtype)
    cos, sin = orc.RopeCache(d, dtype).tables(T, dtype)
    rq = orc.apply_rope(q, cos[None, :, None], sin[None, :, None])
    rk = orc.apply_rope(k, cos[None, :, None], sin[None, :, None])
    for c, s in ((cos[None, :, None], sin[None, :, None]), (cos, sin)):
        oq, ok = G.apply_rotary_pos_emb(q.to(dev), k.to(dev), c.to(dev), s.to(dev))
        assert torch.equal(oq.cpu(), rq) and torch.equal(ok.cpu(), rk)


@pytest.mark.parametrize("B,T,H,dtype", [(1, 1, 1, torch.bfloat16), (1, 5, 3, torch.float32), (3, 1, 16, torch.bfloat16),
                                         (2, 67, 64, torch.float32), (1, 258, 16, torch.bfloat16)])
def test_apply_rotary_pos_emb_rows(dev, B, T, H, dtype):
    """Row counts around the rows a block takes (4), one to 64 heads, q and k views
    with strides of their own, in one launch (one shape) and in two (k with a head
    more): bit-exact with the oracle."""
    g = torch.Generator().manual_seed(T)
    qkv = torch.randn(B, T + 1, 3, H, 128, generator=g).to(dtype)
    q, k, k2 = qkv[:, :T, 0], qkv[:, 1:, 2], torch.randn(B, T, H % 64 + 1, 128, generator=g).to(dtype)
    cos, sin = orc.RopeCache(128, dtype).tables(T, dtype)
    ref = [orc.apply_rope(t, cos[None, :, None], sin[None, :, None]) for t in (q, k, k2)]
    c, s, qd = cos.to(dev), sin.to(dev), qkv.to(dev)
    oq, ok = G.apply_rotary_pos_emb(qd[:, :T, 0], qd[:, 1:, 2], c, s)
    assert oq.is_contiguous() and ok.is_contiguous()
    assert torch.equal(oq.cpu(), ref[0]) and torch.equal(ok.cpu(), ref[1])
    oq, ok = G.apply_rotary_pos_emb(qd[:, :T, 0], k2.to(dev), c, s)
    assert torch.equal(oq.cpu(), ref[0]) and torch.equal(ok.cpu(), ref[2])


@pytest.mark.parametrize("B,T,H,dtype", [(1, 1279, 64, torch.float32), (1, 1280, 64, torch.float32), (2, 1700, 33, torch.float32),
                                         (1, 2600, 32, torch.float32),
                                         (1, 3400, 31, torch.float32), (1, 2560, 64, torch.bfloat16)])
def test_apply_rotary_pos_emb_large(dev, B, T, H, dtype):
    """Around the heads and sizes from which q and k are taken one after the other (40 MiB a
    tensor), q and k as views of one buffer: the oracle's rounding, on the device."""
    g = torch.Generator(device=dev).manual_seed(T)
    qk = torch.randn(B, T, 2, H, 128, generator=g, device=dev).to(dtype)
    cos, sin = (t.to(dev) for t in orc.RopeCache(128, dtype).tables(T, dtype))
    out = G.apply_rotary_pos_emb(qk[:, :, 0], qk[:, :, 1], cos, sin)
    for i in (0, 1):
        assert out[i].is_contiguous()
        assert torch.equal(out[i], orc.apply_rope(qk[:, :, i], cos[None, :, None], sin[None, :, None]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rotary_embedding_tables_on_device(dev, dtype):
    """RotaryEmbedding.forward(seq_len, device, dtype) after a module cast: the cached
    tables, the rebuild past 8192 positions from the cast inv_freq, and a shorter
    request after it, each equal to the oracle's RopeCache."""
    m = G.RotaryEmbedding(128).to(dev).to(dtype)
    rc = orc.RopeCache(128, dtype)
    for n in (100, 8192, 8200, 300):
        c, s = m(n, dev, dtype)
        rcos, rsin = rc.tables(n, dtype)
        assert c.shape == (n, 128) and c.device.type == "cuda"
        assert torch.equal(c.cpu(), rcos) and torch.equal(s.cpu(), rsin), n
    assert math.isclose(float(m.inv_freq[1].float()), float(rc.inv_freq[1].float()))
