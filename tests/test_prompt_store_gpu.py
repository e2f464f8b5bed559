"""New prompts through the device path of push_chunk (kitty_store_prompt) and
reset_sequence (kitty_zero_regions), bit for bit against the torch copies that
prompts off 16-byte alignment take."""
import ctypes

import numpy as np
import pytest
import torch

from kitty import KittyAttentionFactory, KittyConfig


def _state(layout, pipe):
    bits = lambda t: t.view(torch.int16) if t.element_size() == 2 else t
    return {k: bits(v).cpu() for k, v in dict(
        kb=layout.key_baseline, kh=layout.key_boost, km=layout.key_metadata, vp=layout.value_pool,
        vm=layout.value_metadata, sk=pipe._sink_k, sv=pipe._sink_v, qk=pipe._qbuf_k, vb=pipe._vbuf, lens=pipe.lens,
        bt=pipe._block_table).items()} | dict(
            counts=torch.from_numpy(pipe._counts.copy()), pages=torch.from_numpy(pipe._pages.copy()))


def _assert_same(a, b):
    for k in a:
        assert torch.equal(a[k], b[k]), k


def _pipe(S, G, R, H, D, L, B, T, dtype):
    cfg = KittyConfig(num_layers=L, num_kv_heads=H, head_dim=D, sink_size=S, q_buffer_size=G, local_value_window=R,
                      max_seq_len=max(T, S + G) + G, max_batch_size=B + 1, dtype=dtype, device="cuda:0",
                      pool_pages_override=((T // G) + 2) * (B + 1) * L)
    gen = torch.Generator().manual_seed(1)
    bi = torch.full((L, H, D), cfg.sentinel, dtype=torch.uint8)
    for l in range(L):
        for h in range(H):
            bi[l, h, torch.randperm(D, generator=gen)[:cfg.d_boost]] = torch.arange(cfg.d_boost, dtype=torch.uint8)
    layout, pipe, _ = KittyAttentionFactory.from_config(cfg, bi, H)
    return layout, pipe


def _off(x):
    """The same values 2 bytes off a 16-byte boundary."""
    return torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].copy_(x.reshape(-1)).view(x.shape)


# prompts shorter than the sinks, without pages, without value pages, many
# pages; no sinks; one stream (R = 0); windows that are no multiple of a page;
# small heads and pages; more layers than the one written; a view per head
@pytest.mark.gpu
@pytest.mark.parametrize("S,G,R,H,D,L,B,T,dtype,form", [
    (32, 128, 128, 2, 128, 1, 1, 5, "float16", "plain"),
    (32, 128, 128, 2, 128, 2, 3, 32, "float16", "plain"),
    (32, 128, 128, 8, 128, 1, 2, 159, "float16", "tokens_first"),
    (32, 128, 128, 2, 128, 1, 2, 160, "bfloat16", "plain"),
    (32, 128, 128, 2, 128, 2, 2, 416, "float16", "tokens_first"),
    (32, 128, 128, 4, 128, 1, 3, 1111, "bfloat16", "plain"),
    (0, 128, 128, 2, 128, 1, 2, 700, "float16", "plain"),
    (32, 128, 0, 2, 128, 1, 2, 300, "float16", "plain"),
    (4, 16, 5, 2, 64, 1, 2, 101, "float16", "tokens_first"),
    (3, 8, 21, 1, 16, 3, 2, 40, "bfloat16", "plain"),
    (32, 128, 600, 8, 128, 1, 40, 800, "float16", "plain"),     # separate key and value launches
    (32, 128, 128, 2, 128, 1, 4, 300, "float16", "expanded"),
])
def test_prompt_store_matches_torch_copies(dev, S, G, R, H, D, L, B, T, dtype, form):
    gen = torch.Generator().manual_seed(T + B)
    dt = torch.float16 if dtype == "float16" else torch.bfloat16
    k, v = (torch.randn(B, H, T, D, generator=gen).to(dt).to(dev) for _ in range(2))
    if form == "tokens_first":       # (B, T, H, D) projections
        k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (k, v))
    elif form == "expanded":         # one prompt for all sequences
        k, v = (t[:1].expand(B, H, T, D) for t in (k, v))
    states = []
    for kk, vv in ((k, v), (_off(k), _off(v))):
        layout, pipe = _pipe(S, G, R, H, D, L, B, T, dtype)
        pipe.slot(99)                                 # the run does not start at slot 0
        pipe.push_chunk(L - 1, kk, vv, list(range(B)))
        states.append(_state(layout, pipe))
        # a decode token works on what the prompt left
        pipe.push_tokens(L - 1, kk[:, :, 0].clone(), vv[:, :, 0].clone(), list(range(B)))
        states.append(_state(layout, pipe))
        pipe.reset_sequence(1 if B > 1 else 0)
        states.append(_state(layout, pipe))
    for a, b in zip(states[:3], states[3:]):
        _assert_same(a, b)
    s = 2 if B > 1 else 1                              # the reset sequence's slot holds nothing
    for name in ("sk", "sv", "qk", "vb"):
        assert int(states[2][name][s].ne(0).sum()) == 0
    assert int(states[2]["bt"][:, s].ne(0).sum()) == 0 and int(states[2]["lens"][:, :, s].ne(0).sum()) == 0
    assert int(states[2]["lens"].ne(0).sum()) == (0 if B == 1 else int(states[1]["lens"][:, :, [0] + list(range(1, s)) +
                                                  list(range(s + 1, B + 1))].ne(0).sum()))


@pytest.mark.gpu
def test_prompt_shape_errors_stay_errors(dev):
    layout, pipe = _pipe(32, 128, 128, 2, 128, 1, 2, 300, "float16")
    k = torch.randn(2, 2, 300, 128).half().to(dev)
    with pytest.raises((RuntimeError, ValueError, IndexError)):
        pipe.push_chunk(0, k[:, :, :, :64].contiguous(), k[:, :, :, :64].contiguous(), [0, 1])
    with pytest.raises((RuntimeError, ValueError, IndexError)):
        pipe.push_chunk(0, k.repeat(1, 2, 1, 1), k.repeat(1, 2, 1, 1), [0, 1])


@pytest.mark.gpu
def test_zero_regions(dev):
    """Aligned and 4-byte regions, rows with a stride, empty ones, more than one launch's worth."""
    from kitty import _hip
    L = _hip.load()
    x = torch.ones(40, 1000, dtype=torch.int32, device=dev)
    keep = x.clone()
    regions = []
    for i in range(20):
        c, w = (4 * i, 8) if i % 2 else (4 * i + 1, 7)      # 16-byte vectors or single words
        regions.append(_hip.ZeroRegion(x.data_ptr() + 4 * (1000 * i + c), 2, 4 * w, 4 * 20 * 1000))
        keep[[i, i + 20], c:c + w] = 0
    regions.append(_hip.ZeroRegion(0, 0, 0, 0))
    arr = (_hip.ZeroRegion * len(regions))(*regions)
    _hip.check(L.kitty_zero_regions(arr, len(regions), _hip.stream_ptr(dev)))
    assert torch.equal(x, keep)
    bad = (_hip.ZeroRegion * 1)(_hip.ZeroRegion(x.data_ptr() + 2, 1, 4, 0))
    with pytest.raises(ValueError):
        _hip.check(L.kitty_zero_regions(bad, 1, _hip.stream_ptr(dev)))
