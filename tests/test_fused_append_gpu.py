"""kitty_decode_step in one launch (tickets given): the append's corner cases
against kitty_append_tokens and kitty_paged_decode, bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

from kitty import KittyAttentionFactory, KittyConfig, _hip


# a token into the sinks, an empty sequence's first, into a key tail, a full key
# buffer (flagged, decoded as it stands) and a slot out of range (nothing written);
# groups of 1, 4 and 8, one with members the kernel pads, and a long-context hint
# that takes the separate launches
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,Hq,H,hint", [("float16", 2, 2, 4), ("bfloat16", 8, 2, 4), ("float16", 16, 2, 4),
                                             ("bfloat16", 6, 2, 4), ("float16", 16, 1, 4), ("float16", 8, 2, 4000)])
def test_one_launch_step_matches_append_then_decode(dev, dtype, Hq, H, hint):
    dt = torch.float16 if dtype == "float16" else torch.bfloat16
    B, D, maxlen = 5, 128, 65536 if hint > 100 else 1024
    cfg = KittyConfig(num_layers=1, num_kv_heads=H, head_dim=D, max_seq_len=maxlen, max_batch_size=B, dtype=dtype,
                      device="cuda:0")
    gen = torch.Generator().manual_seed(Hq + H)
    bi = torch.full((1, H, D), cfg.sentinel, dtype=torch.uint8)
    bi[0, :, :cfg.d_boost] = torch.arange(cfg.d_boost, dtype=torch.uint8)
    rnd = lambda *s: torch.randn(*s, generator=gen).to(dt).to(dev)
    prompts = [[rnd(1, h, t, D) for h in (Hq, H, H)] for t in (300, 7, 32, 280, 700)]
    q, k, v = rnd(B, Hq, 1, D), rnd(B, H, D), rnd(B, H, D)
    runs = []
    for fused in (True, False):
        layout, pipe, (attn,) = KittyAttentionFactory.from_config(cfg, bi, Hq)
        for s, x in enumerate(prompts):
            attn(*x, seq_id=s)
        ids = list(range(B))
        slots = np.arange(B)
        assert [pipe.slot(s) for s in ids] == ids
        plan = attn._plan(q[:, :, 0].contiguous(), ids)
        G = cfg.q_buffer_size
        fill, qlen, npk, npv, vlen = (pipe.lens[i, 0] for i in range(5))
        qlen[3] = G                       # its key buffer is full, its value tail as long as that asks
        vlen[3] = (npk[3] - npv[3]) * G + G
        a, keep = pipe._append_setup(0, slots, H, D)
        keep[4] = B                       # no such slot
        a.key, a.value = k.data_ptr(), v.data_ptr()
        a.key_s_seq = a.value_s_seq = H * D
        a.key_s_head = a.value_s_head = D
        out = torch.empty_like(q)
        args = plan.step_args(q, out)
        args.plan_pages = hint
        tickets = torch.zeros(B, dtype=torch.int32, device=dev)
        stream = _hip.stream_ptr(q.device)
        lib = _hip.load()
        state = []
        for step in range(3):
            if fused:
                _hip.check(lib.kitty_decode_step(ctypes.byref(a), ctypes.byref(args), tickets.data_ptr(), stream))
            else:
                _hip.check(lib.kitty_append_tokens(ctypes.byref(a), stream))
                _hip.check(lib.kitty_paged_decode(ctypes.byref(args), stream))
            state += [out.clone(), pipe.lens.clone(), pipe._overflow.clone()]
        assert not tickets.any()
        assert pipe._overflow.tolist() == [0, 0, 0, 1, 0]
        assert fill.tolist()[1] == 10 and qlen.tolist()[0] == 300 - 32 - 256 + 3 and qlen.tolist()[2] == 3
        assert torch.isfinite(out).all()
        runs.append(state + [pipe._sink_k, pipe._sink_v, pipe._qbuf_k, pipe._vbuf])
    for i, (x, y) in enumerate(zip(*runs)):
        assert torch.equal(x, y), i
