"""bf16 blocks on the 128 x 128 quantise kernel, byte for byte against the
shape-generic kernel (which blocks off 16-byte alignment run) and the oracle."""
import numpy as np
import pytest
import torch

import kitty  # noqa: F401
import oracle as O

D = G = 128


def _bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _blocks(kind, n, H, gen):
    x = torch.randn(n, H, G, D, generator=gen)
    if kind == "outliers":
        x[..., ::9] *= 16.0
    elif kind == "ties":            # quotients on half-integers, ranges that are exact
        x = torch.randint(-6, 7, x.shape, generator=gen).float() * 0.5
        x[..., 0, :], x[..., 1, :] = -1.5, 1.5
    elif kind == "wide":            # exponents over bf16's range, fp16 scales overflow
        x = x * torch.exp2(torch.randint(-100, 120, x.shape, generator=gen).float())
    elif kind == "huge":            # scales whose reciprocal leaves the normal numbers, and infinite ranges
        x = x.clamp(-3, 3) * 1.0e38
    elif kind == "tiny":
        x = x * 1e-30
    elif kind == "constant":
        x[:, :, :, ::2] = 0.75
        x[:, :, ::3] = -2.0
        x[:, 0] = 0.0
    elif kind == "nonfinite":
        x[:, :, 5, 7] = float("inf")
        x[:, :, 9, 11] = -float("inf")
        x[:, :, 30, 40:60] = float("nan")
        x[:, :, :, 77] = float("nan")      # a whole channel
        x[:, :, 100] = float("nan")        # a whole token
    return x.to(torch.bfloat16)


def _pools(P, H, Dk, meta, dev):
    u8 = lambda *s: torch.full(s, 0xA5, dtype=torch.uint8, device=dev)
    m = lambda *s: torch.full(s, 7.0, dtype=meta, device=dev)
    return u8(P, H, D, G // 4), u8(P, H, Dk, G // 4), m(P, H, 2, D), u8(P, H, G, D // 4), m(P, H, G, 2)


def _misaligned(x):
    """The same block values, 2 bytes off a 16-byte boundary."""
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:]
    return flat.copy_(x.reshape(-1)).view(x.shape)


KINDS = ["normal", "outliers", "ties", "wide", "huge", "tiny", "constant", "nonfinite"]


@pytest.mark.gpu
@pytest.mark.parametrize("meta", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", KINDS)
def test_bf16_blocks_match_the_generic_kernel(dev, kind, meta):
    from kitty.kernels.ops import pool_store, quantize_into_pools
    gen = torch.Generator().manual_seed(KINDS.index(kind))
    n, H, Dk = 3, 2, 16
    k, v = _blocks(kind, n, H, gen).to(dev), _blocks(kind, n, H, gen).to(dev)
    bi = torch.full((H, D), Dk + 1, dtype=torch.uint8)
    for h in range(H):
        bi[h, torch.randperm(D, generator=gen)[:Dk]] = torch.arange(Dk, dtype=torch.uint8)
    bi, ids = bi.to(dev), torch.tensor([4, 0, 2], dtype=torch.int32, device=dev)
    got, ref = _pools(5, H, Dk, meta, dev), _pools(5, H, Dk, meta, dev)
    quantize_into_pools(pool_store(*got), k, v, bi, ids, Dk + 1, value_rows=120)
    quantize_into_pools(pool_store(*ref), _misaligned(k), _misaligned(v), bi, ids, Dk + 1, value_rows=120)
    for name, a, b in zip(("key_low", "key_high", "key_meta", "value", "value_meta"), got, ref):
        a, b = (t.view(torch.int16) if t.element_size() == 2 else t for t in (a, b))
        assert torch.equal(a, b), (name, int((a != b).sum()))
    # channel-major keys (the one-page signature's (D, G) block)
    kt = k.transpose(2, 3).contiguous().transpose(2, 3)
    again = _pools(5, H, Dk, meta, dev)
    quantize_into_pools(pool_store(*again), kt, None, bi, ids, Dk + 1)
    for a, b in zip(again[:3], got[:3]):
        a, b = (t.view(torch.int16) if t.element_size() == 2 else t for t in (a, b))
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_bf16_blocks_match_the_oracle(dev):
    from kitty.kernels.ops import pool_store, quantize_into_pools
    gen = torch.Generator().manual_seed(50)
    n, H, Dk = 2, 2, 32
    k, v = _blocks("outliers", n, H, gen), _blocks("normal", n, H, gen)
    bi = torch.full((H, D), Dk + 1, dtype=torch.uint8)
    for h in range(H):
        bi[h, torch.randperm(D, generator=gen)[:Dk]] = torch.arange(Dk, dtype=torch.uint8)
    pools = _pools(n, H, Dk, torch.bfloat16, dev)
    quantize_into_pools(pool_store(*pools), k.to(dev), v.to(dev), bi.to(dev),
                        torch.arange(n, dtype=torch.int32, device=dev), Dk + 1)
    kb, kh, km, vp, vm = pools
    for p in range(n):
        for h in range(H):
            a, b, s, z = O.quantize_key_bf16(_bits(k[p, h].t()), bi[h].numpy(), Dk, Dk + 1)
            assert np.array_equal(kb[p, h].cpu().numpy(), a) and np.array_equal(kh[p, h].cpu().numpy(), b)
            assert np.array_equal(_bits(km[p, h, 0]), s)
            assert np.array_equal(O.bf16_to_f32(_bits(km[p, h, 1])), O.bf16_to_f32(z))
            c, vs, vz = O.quantize_value_bf16(_bits(v[p, h]))
            assert np.array_equal(vp[p, h].cpu().numpy(), c) and np.array_equal(_bits(vm[p, h, :, 0]), vs)
            assert np.array_equal(O.bf16_to_f32(_bits(vm[p, h, :, 1])), O.bf16_to_f32(vz))


@pytest.mark.gpu
def test_bf16_value_shift(dev):
    """The value window's shift moves 16-bit rows whatever their type."""
    from kitty.kernels.ops import QuantizePlan, pool_store
    gen = torch.Generator().manual_seed(51)
    H, R = 2, 100
    buf = torch.randn(1, H, G + R, D, generator=gen).to(torch.bfloat16).to(dev)
    before = buf.clone()
    pools = _pools(1, H, 16, torch.bfloat16, dev)
    plan = QuantizePlan(pool_store(*pools), None, buf[:, :, :G], None, torch.zeros(1, dtype=torch.int32, device=dev), 17,
                        value_shift=R)
    plan.run()
    assert torch.equal(buf[:, :, :R], before[:, :, G:]) and torch.equal(buf[:, :, R:], before[:, :, R:])


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["normal", "ties", "constant", "nonfinite"])
def test_fp16_blocks_into_bf16_pools(dev, kind):
    """fp16 blocks into bf16 pools quantise as on the shape-generic kernel
    whatever their alignment, all-NaN channels and tokens included."""
    from kitty.kernels.ops import pool_store, quantize_into_pools
    gen = torch.Generator().manual_seed(60 + KINDS.index(kind))
    n, H, Dk = 2, 2, 16
    k, v = (_blocks(kind, n, H, gen).to(torch.float16).to(dev) for _ in range(2))
    bi = torch.full((H, D), Dk + 1, dtype=torch.uint8, device=dev)
    bi[:, :Dk] = torch.arange(Dk, dtype=torch.uint8, device=dev)
    ids = torch.tensor([1, 0], dtype=torch.int32, device=dev)
    got, ref = _pools(n, H, Dk, torch.bfloat16, dev), _pools(n, H, Dk, torch.bfloat16, dev)
    quantize_into_pools(pool_store(*got), k, v, bi, ids, Dk + 1)
    quantize_into_pools(pool_store(*ref), _misaligned(k), _misaligned(v), bi, ids, Dk + 1)
    for a, b in zip(got, ref):
        a, b = (t.view(torch.int16) if t.element_size() == 2 else t for t in (a, b))
        assert torch.equal(a, b)
