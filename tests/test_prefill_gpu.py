"""Prompt attention (kitty_prefill_attention, KittyPagedAttention.forward with
T > 1) against float64 causal attention."""
import math

import pytest
import torch

import kitty  # noqa: F401


def _ref(q, k, v):
    """Causal attention in float64 on the CPU, (B, Hq, T, D)."""
    B, Hq, T, D = q.shape
    gq = Hq // k.shape[1]
    q, k, v = (t.cpu().double() for t in (q, k, v))
    out = torch.empty(B, Hq, T, D, dtype=torch.float64)
    mask = torch.ones(T, T, dtype=torch.bool).triu_(1)
    for b in range(B):
        for h in range(Hq):
            s = (q[b, h] @ k[b, h // gq].t()) / math.sqrt(D)
            out[b, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[b, h // gq]
    return out


# query blocks are 32 rows, tiles 64 tokens, a workgroup four (block, head) waves:
# lengths around both, groups that do not divide four, batches past eight pairs
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,T", [(1, 1, 1, 1), (1, 4, 1, 2), (2, 8, 8, 31), (1, 8, 2, 32), (1, 7, 1, 33),
                                        (3, 6, 2, 63), (1, 8, 2, 64), (2, 3, 3, 65), (1, 20, 1, 129), (1, 8, 1, 300),
                                        (9, 2, 1, 96), (1, 2, 2, 1025)])
def test_prefill_matches_float64(dev, dtype, B, Hq, Hkv, T):
    from kitty.kernels.ops import prefill_attention, prefill_supported
    gen = torch.Generator().manual_seed(B * 1000 + Hq * 100 + T)
    q, k, v = (torch.randn(B, h, T, 128, generator=gen) for h in (Hq, Hkv, Hkv))
    k[..., :16] *= 8.0                      # outlier channels: sharp softmax rows
    q, k, v = (t.to(dtype).to(dev) for t in (q, k, v))
    assert prefill_supported(q, k, v)
    out = prefill_attention(q, k, v, 1.0 / math.sqrt(128))
    assert out.dtype == dtype and out.shape == q.shape
    ref = _ref(q, k, v)
    # fp32 scores and sums, two-term probabilities (2^-16 or better): what is
    # left is the rounding of the output, half an ulp, 2^-11 or 2^-8 relative;
    # scores reach ~100, so fp32 moves a weight by up to 100 * 2^-22
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    err = (out.cpu().double() - ref).abs()
    assert (err <= eps * ref.abs() + 1e-4).all(), float(err.max())


@pytest.mark.gpu
def test_prefill_strided_inputs(dev):
    """Projections handed over as (B, T, H, D) views and slices of a fused
    qkv: read in place, the same result as contiguous copies; layouts the
    kernel does not take go to torch and agree."""
    from kitty.kernels.ops import prefill_attention, prefill_supported
    gen = torch.Generator().manual_seed(3)
    B, T, Hq, Hkv, D = 2, 130, 8, 2, 128
    qkv = torch.randn(B, T, (Hq + 2 * Hkv) * D, generator=gen).half().to(dev)
    x = qkv.view(B, T, Hq + 2 * Hkv, D).permute(0, 2, 1, 3)
    q, k, v = x[:, :Hq], x[:, Hq:Hq + Hkv], x[:, Hq + Hkv:]
    assert prefill_supported(q, k, v)
    out = prefill_attention(q, k, v, 0.1)
    same = prefill_attention(q.contiguous(), k.contiguous(), v.contiguous(), 0.1)
    assert torch.equal(out, same)
    assert not prefill_supported(q[..., ::2], k[..., ::2], v[..., ::2])             # channel stride 2
    odd = torch.empty(q.numel() + 1, dtype=q.dtype, device=dev)[1:].view(q.shape)   # 2-byte aligned
    assert not prefill_supported(odd, k, v)
    assert not prefill_supported(q.float(), k.float(), v.float())
    assert not prefill_supported(q.detach().requires_grad_(), k, v)
    assert not prefill_supported(q[:, :, :5], k, v)


@pytest.mark.gpu
def test_prefill_nonfinite_rows(dev):
    """A NaN or infinite query or key reaches the rows that see it and no others."""
    from kitty.kernels.ops import prefill_attention
    gen = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(1, 1, 200, 128, generator=gen).half() for _ in range(3))
    clean = _ref(q, k, v)
    q[0, 0, 50] = float("nan")
    k[0, 0, 150, 3] = float("inf")
    out = prefill_attention(q.to(dev), k.to(dev), v.to(dev), 1.0 / math.sqrt(128)).cpu().double()[0, 0]
    assert out[50].isnan().all()
    keep = [i for i in range(150) if i != 50]
    assert (out[keep] - clean[0, 0, keep]).abs().max() < 2e-3
    # rows from 150 on: the score is +-inf by the sign of q's channel 3; -inf takes weight 0
    for i in range(150, 200):
        if q[0, 0, i, 3] > 0:
            assert out[i].isnan().all(), i
        else:
            assert out[i].isfinite().all(), i


# one head and groups; an infinite value at the first token (weight 1 in its own
# row), inside tiles, of both signs in one channel, in the last ragged tile
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,T,rows", [(1, 1, 1, [(0, 5, 1)]), (4, 1, 40, [(0, 3, 1), (7, 3, -1), (9, 4, -1)]),
                                           (6, 2, 201, [(0, 0, -1), (70, 5, 1), (75, 6, -1), (150, 5, -1), (200, 7, 1)])])
def test_prefill_nonfinite_values(dev, dtype, Hq, Hkv, T, rows):
    """Infinite and NaN values reach the rows that see them as the product of the
    weights with them does; other channels and tiles before keep their numbers."""
    from kitty.kernels.ops import prefill_attention
    gen = torch.Generator().manual_seed(T)
    q, k, v = (torch.randn(1, h, T, 128, generator=gen).to(dtype) for h in (Hq, Hkv, Hkv))
    clean = _ref(q, k, v)
    for t, c, sign in rows:
        v[0, :, t, c] = sign * float("inf")
    v[0, :, T // 2, 100] = float("nan")
    out = prefill_attention(q.to(dev), k.to(dev), v.to(dev), 1.0 / math.sqrt(128)).cpu().double()
    bad = {c for _, c, _ in rows} | {100}
    keep = [c for c in range(128) if c not in bad]
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert ((out - clean).abs() <= eps * clean.abs() + 1e-4)[..., keep].all()
    for h in range(Hq):
        s = (q[0, h].double() @ k[0, h * Hkv // Hq].double().t()) / math.sqrt(128)
        for i in range(T):
            want = torch.softmax(s[i, :i + 1], 0) @ v[0, h * Hkv // Hq, :i + 1].double()
            for c in bad:
                first = min([t for t, cc, _ in rows if cc == c] + [T // 2] * (c == 100))
                if i >= first:
                    got = out[0, h, i, c]
                    assert got == want[c] or (got.isnan() and want[c].isnan()), (h, i, c)
                elif i // 64 < first // 64:
                    assert (out[0, h, i, c] - clean[0, h, i, c]).abs() <= eps * clean[0, h, i, c].abs() + 1e-4


@pytest.mark.gpu
def test_module_prefill_keeps_gradients(dev):
    """Inputs that need gradients keep torch's differentiable path."""
    from kitty import KittyAttentionFactory, KittyConfig
    cfg = KittyConfig(num_layers=1, num_kv_heads=1, head_dim=128, max_seq_len=512, device="cuda:0")
    bi = torch.full((1, 1, 128), cfg.sentinel, dtype=torch.uint8)
    _, _, layers = KittyAttentionFactory.from_config(cfg, bi, 2)
    gen = torch.Generator().manual_seed(5)
    q = torch.randn(1, 2, 40, 128, generator=gen).half().to(dev).requires_grad_()
    k, v = (torch.randn(1, 1, 40, 128, generator=gen).half().to(dev) for _ in range(2))
    out = layers[0](q, k, v, seq_id=0)
    out.float().sum().backward()
    assert q.grad is not None and torch.isfinite(q.grad).all()
    plain = layers[0](q.detach(), k, v, seq_id=0)
    assert (plain.float() - out.float()).abs().max() < 2e-3


@pytest.mark.gpu
def test_prefill_long_prompt_is_repeatable(dev):
    """A prompt of many tiles, with every workgroup slot in use: repeated
    calls give the same bits, and sampled rows match float64."""
    from kitty.kernels.ops import prefill_attention
    gen = torch.Generator(device=dev).manual_seed(6)
    T = 6001
    q, k, v = (torch.randn(1, h, T, 128, device=dev, generator=gen).half() for h in (32, 8, 8))
    k[..., :16] *= 8.0
    first = prefill_attention(q, k, v, 1.0 / math.sqrt(128))
    for _ in range(12):
        assert torch.equal(prefill_attention(q, k, v, 1.0 / math.sqrt(128)), first)
    for h, i in [(0, 6000), (13, 5593), (31, 3171), (8, 64), (20, 4480)]:
        s = (k[0, h // 4, :i + 1].double() @ q[0, h, i].double()) / math.sqrt(128)
        ref = torch.softmax(s, 0) @ v[0, h // 4, :i + 1].double()
        assert ((first[0, h, i].double() - ref).abs() <= 2.0 ** -11 * ref.abs() + 1e-4).all()


@pytest.mark.gpu
def test_prefill_large_bf16_values(dev):
    """bf16 values near the end of the range, as a float32 product takes them."""
    from kitty.kernels.ops import prefill_attention
    gen = torch.Generator().manual_seed(12)
    q, k, v = (torch.randn(1, 1, 96, 128, generator=gen) * s for s in (0.1, 1.0, 2.0 ** 118))
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    out = prefill_attention(q.to(dev), k.to(dev), v.to(dev), 1.0 / math.sqrt(128)).cpu().double()
    ref = _ref(q, k, v)
    assert ((out - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4 * 2.0 ** 118).all()


@pytest.mark.gpu
def test_module_prompt_of_other_heads_is_refused(dev):
    from kitty import KittyAttentionFactory, KittyConfig
    cfg = KittyConfig(num_layers=1, num_kv_heads=2, head_dim=128, max_seq_len=512, device="cuda:0")
    bi = torch.full((1, 2, 128), cfg.sentinel, dtype=torch.uint8)
    _, _, layers = KittyAttentionFactory.from_config(cfg, bi, 8)
    x = lambda h: torch.randn(1, h, 20, 128, device=dev).half()
    with pytest.raises(RuntimeError, match="must match"):
        layers[0](x(8), x(1), x(1))
