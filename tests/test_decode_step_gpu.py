"""Module decode steps whose append and decode go out in one call
(kitty_decode_step), bit for bit against steps taken apart."""
import ctypes
import gc
import warnings
import weakref

import numpy as np
import pytest
import torch

from kitty import KittyAttentionFactory, KittyConfig


def _module(dtype, Hq, H, B, T, R=128):
    cfg = KittyConfig(num_layers=1, num_kv_heads=H, head_dim=128, max_seq_len=T, max_batch_size=B, dtype=dtype,
                      local_value_window=R, device="cuda:0")
    gen = torch.Generator().manual_seed(2)
    bi = torch.full((1, H, 128), cfg.sentinel, dtype=torch.uint8)
    for h in range(H):
        bi[0, h, torch.randperm(128, generator=gen)[:cfg.d_boost]] = torch.arange(cfg.d_boost, dtype=torch.uint8)
    return KittyAttentionFactory.from_config(cfg, bi, Hq)


# from empty sequences through the sinks (32), into pages and across key and
# value spills; one sequence and batches, groups the kernels pad, both streams
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,Hq,H,B,prompt,steps,R", [
    ("float16", 8, 8, 1, 0, 40, 128), ("float16", 8, 2, 1, 270, 30, 128), ("bfloat16", 8, 2, 1, 400, 30, 128),
    ("float16", 6, 2, 3, 150, 20, 128), ("bfloat16", 8, 1, 4, 410, 20, 128), ("float16", 20, 1, 2, 280, 12, 0),
    ("bfloat16", 4, 4, 2, 20, 30, 5),
])
def test_fused_steps_match_separate_ones(dev, dtype, Hq, H, B, prompt, steps, R):
    dt = torch.float16 if dtype == "float16" else torch.bfloat16
    gen = torch.Generator().manual_seed(prompt + steps)
    rnd = lambda *s: torch.randn(*s, generator=gen).to(dt).to(dev)
    prompts = [rnd(B, h, max(prompt, 1), 128) for h in (Hq, H, H)]
    toks = [[rnd(B, h, 1, 128) for h in (Hq, H, H)] for _ in range(steps)]
    runs = []
    for fused in (True, False):
        layout, pipe, layers = _module(dtype, Hq, H, B, 1024, R)
        calls = []
        if fused:
            push = pipe._push
            pipe._push = lambda *a: calls.append(push(*a)) or calls[-1]
        outs = []
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", RuntimeWarning)
            if prompt:
                layers[0](*prompts)
            for q, k, v in toks:
                if not fused:       # a query that is not contiguous goes the separate way
                    q = torch.cat([q, q], 3)[..., :128]
                outs.append(layers[0](q, k, v).clone())
        assert all(o.dtype == dt and o.shape == (B, Hq, 1, 128) for o in outs)
        assert not fused or sum(bool(c) for c in calls) >= steps - 3 - (B > 1 and prompt < 32) * 32
        runs.append((outs, pipe.lens.clone(), layout.value_pool.clone(), layout.key_baseline.clone(),
                     torch.from_numpy(pipe._counts.copy())))
    for i, (a, b) in enumerate(zip(runs[0][0], runs[1][0])):
        assert torch.equal(a, b), i
    for a, b in zip(runs[0][1:], runs[1][1:]):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_steps_after_resets_use_the_new_slots(dev):
    """The same ids on other slots after a reset: cached steps do not survive it."""
    layout, pipe, layers = _module("float16", 8, 2, 3, 512)
    attn = layers[0]
    gen = torch.Generator().manual_seed(9)
    rnd = lambda h, t: torch.randn(1, h, t, 128, generator=gen).half().to(dev)
    tok = {s: (rnd(8, 60), rnd(2, 60), rnd(2, 60)) for s in (1, 2, 3)}

    def run(seq, n):
        q, k, v = tok[seq]
        return [attn(*(t[:, :, i:i + 1].contiguous() for t in (q, k, v)), seq_id=seq).clone() for i in range(n)]
    a1, a2 = run(1, 50), run(2, 50)            # slots 0 and 1
    pipe.reset_sequence(1)
    a3 = run(3, 50)                            # sequence 3 on slot 0
    pipe.reset_sequence(2)
    b1 = run(1, 50)                            # sequence 1 on slot 1
    b3 = attn(*(t[:, :, 50:51].contiguous() for t in tok[3]), seq_id=3)
    for x, y in zip(a1, b1):
        assert torch.equal(x, y)
    pipe.reset_sequence(3)
    c3 = run(3, 51)
    for x, y in zip(a3 + [b3], c3):
        assert torch.equal(x, y)


@pytest.mark.gpu
def test_full_pool_raises_before_the_step(dev):
    layout, pipe, layers = _module("float16", 4, 1, 1, 160)
    attn = layers[0]
    x = lambda h: torch.ones(1, h, 1, 128, dtype=torch.float16, device=dev)
    for _ in range(159):
        attn(x(4), x(1), x(1))
    layout._num_free = 0
    before = pipe.lens.clone()
    with pytest.raises(RuntimeError, match="exhausted"):
        attn(x(4), x(1), x(1))
    assert torch.equal(pipe.lens, before)


@pytest.mark.gpu
def test_steps_keep_no_plan_alive(dev):
    """The module keeps at most the 16 plans of _plans (each with a workspace of
    its own), whatever batches have stepped and whichever were reset since."""
    layout, pipe, layers = _module("float16", 4, 1, 24, 256)
    attn = layers[0]
    x = lambda h: torch.ones(1, h, 1, 128, dtype=torch.float16, device=dev)
    plans = []
    for s in range(24):
        attn(x(4), x(1), x(1), seq_id=s)
        plans += [weakref.ref(p) for p in attn._plans.values() if p not in [r() for r in plans]]
        attn(x(4), x(1), x(1), seq_id=s)
    gc.collect()
    assert len(plans) == 24 and sum(r() is not None for r in plans) == len(attn._plans) <= 16


def _raw_step(dev, B, slots):
    """A pipeline of four 100-token sequences and the arguments of a step of the
    decode's rows 1 .. B with the append's slots."""
    from kitty import _hip
    layout, pipe, layers = _module("float16", 8, 2, 4, 512)
    gen = torch.Generator().manual_seed(8)
    k = torch.randn(4, 2, 100, 128, generator=gen).half().to(dev)
    pipe.push_chunk(0, k, -k, [0, 1, 2, 3])
    tok = torch.randn(B, 2, 128, generator=gen).half().to(dev)
    q = torch.randn(B, 8, 1, 128, generator=gen).half().to(dev)
    plan = layers[0]._plan(q[:, :, 0].contiguous(), list(range(1, 1 + B)))
    a, keep = pipe._append_setup(0, np.array(slots), 2, 128)
    a.key = a.value = tok.data_ptr()
    a.key_s_seq = a.value_s_seq = 256
    a.key_s_head = a.value_s_head = 128
    out = torch.empty_like(q)
    d = plan.step_args(q, out)
    d.plan_pages = 1

    def step():
        _hip.check(pipe._lib.kitty_decode_step(ctypes.byref(a), ctypes.byref(d), pipe._tickets.data_ptr(),
                                               _hip.stream_ptr(dev)))
        torch.cuda.synchronize()
    return pipe, d, tok, out, step, (layers, plan, q, keep)


@pytest.mark.gpu
def test_step_whose_lengths_are_not_the_appends(dev):
    """A decode over a copy of the counters: the token goes where the append's
    own counters say, the decode sees the lengths it was given."""
    pipe, d, tok, out, step, _keep = _raw_step(dev, 2, [1, 2])
    lens = pipe.lens[:, 0, 1:3].clone()
    lens[1] -= 5
    lens[4] -= 5                                   # five tokens fewer: rows 63 .. 67 are not theirs
    d.sink_len, d.tail_len, d.num_pages, d.num_pages_v, d.tail_len_v = (lens[i].data_ptr() for i in (0, 1, 2, 3, 4))
    qbuf, vbuf, n = pipe._qbuf_k.clone(), pipe._vbuf.clone(), pipe.lens.clone()
    step()
    for s in (1, 2):
        qbuf[s, 0, :, 68] = tok[s - 1]
        vbuf[s, 0, :, 68] = tok[s - 1]
        n[1, 0, s] += 1
        n[4, 0, s] += 1
    assert torch.equal(pipe._qbuf_k, qbuf) and torch.equal(pipe._vbuf, vbuf) and torch.equal(pipe.lens, n)
    assert out.isfinite().all() and not pipe._tickets.any()


@pytest.mark.gpu
def test_step_with_slots_of_other_rows(dev):
    """Slots that are not the decode's rows are refused, one by one."""
    pipe, d, tok, out, step, _keep = _raw_step(dev, 3, [1, 3, 2])
    qbuf, vbuf, n = pipe._qbuf_k.clone(), pipe._vbuf.clone(), pipe.lens.clone()
    step()
    qbuf[1, 0, :, 68] = tok[0]
    vbuf[1, 0, :, 68] = tok[0]
    n[1, 0, 1] += 1
    n[4, 0, 1] += 1
    assert torch.equal(pipe._qbuf_k, qbuf) and torch.equal(pipe._vbuf, vbuf) and torch.equal(pipe.lens, n)
    assert pipe._overflow.tolist()[:3] == [0, 1, 1] and not pipe._tickets.any()


@pytest.mark.gpu
def test_reset_clears_the_tickets(dev):
    layout, pipe, layers = _module("float16", 8, 2, 2, 512)
    x = lambda h: torch.ones(2, h, 1, 128, dtype=torch.float16, device=dev)
    layers[0](x(8), x(2), x(2))
    pipe._tickets += 1                              # as a lost launch leaves them
    pipe.reset_sequence(1)
    assert pipe._tickets.tolist() == [[1, 0]]
