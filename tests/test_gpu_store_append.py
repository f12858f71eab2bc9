"""Storing a prefill chunk (nkv_store_append and its parts) and the recent ring.

The history, codes, scales and sink are compared with torch's fp32 arithmetic
on the CPU bit for bit, the representatives with the oracle's picks in 64
bits; the ring, through chunks, verify commits, decode steps and replays, with
a plain list of tokens or the path without a device ring.  The one-pass entry
point and the three that store its parts are instantiations of one kernel:
that they agree says that the parts do not disturb each other, no more.
"""

import numpy as np
import pytest
import torch

from oracle import nkv_oracle as O

pytestmark = pytest.mark.gpu


def _kv(layers, T, hkv, seed):
    g = torch.Generator().manual_seed(seed)
    k = (torch.randn(layers, T, hkv, 128, generator=g) * 0.1).to(torch.bfloat16)
    v = (torch.randn(layers, T, hkv, 128, generator=g) * 3.0).to(torch.bfloat16)
    k[0, 0, 0, :5] = 0.0
    k[0, T // 2] = 0.0          # a zero key
    v[0, T - 1] *= 1e-9         # a tiny row
    return k, v


def _store(layers, hkv, r, fmt, cap, sink=64, recent=128):
    from nanokv_amd.store import SparseKVStore
    return SparseKVStore(layers, num_heads=2 * hkv, num_kv_heads=hkv, head_dim=128, block_size=64, r=r,
                         cap_blocks=cap, sink_tokens=sink, recent_tokens=recent, kv_format=fmt)


def _blocks(x, nb):
    L, T, hkv, D = x.shape
    pad = torch.zeros(L, nb * 64 - T, hkv, D)
    return torch.cat((x.float(), pad), 1).view(L, nb, 64, hkv, D).permute(0, 3, 1, 2, 4).contiguous()


CASES = [(1, 2, 1, 1), (2, 63, 8, 4), (1, 64, 8, 8), (3, 65, 2, 2), (1, 130, 4, 4), (2, 700, 8, 4), (1, 1025, 3, 4)]


@pytest.mark.parametrize("fmt", ["bf16", "int8", "int8_token"])
@pytest.mark.parametrize("layers,T,hkv,r", CASES)
def test_append_stores_what_torch_computes(layers, T, hkv, r, fmt):
    nb, start = -(-T // 64), 2
    a, b = (_store(layers, hkv, r, fmt, nb + start + 1) for _ in range(2))
    k, v = _kv(layers, T, hkv, T)
    kd, vd = k.cuda(), v.cuda()
    n = min(T, 128)
    slot = 100
    a.append(0, kd, vd, start, True, True, T - n, n, slot)
    b.store_chunk(0, kd, vd, start, True, True)
    b.build_reps(0, kd, start)
    b.recent_update(0, layers, kd, vd, T - n, n, slot, 0, 0)
    for name in ("hist_k", "hist_v", "reps", "sink_k", "sink_v", "recent_k", "recent_v", "k_scale", "v_scale",
                 "k_tscale", "v_tscale"):
        x, y = getattr(a, name), getattr(b, name)
        assert (x is None) == (y is None)
        if x is not None:
            assert torch.equal(x, y), name

    kb, vb = _blocks(k, nb), _blocks(v, nb)
    hk, hv = a.hist_k[:, :, start:start + nb].cpu(), a.hist_v[:, :, start:start + nb].cpu()
    if fmt == "bf16":
        assert torch.equal(hk.float(), kb) and torch.equal(hv.float(), vb)
    else:
        if fmt == "int8":
            ks = (k.float().abs().amax(dim=1).clamp_min(1e-8) / 127.0)
            vs = vb.abs().amax(dim=(3, 4)).clamp_min(1e-8) / 127.0
            assert torch.equal(a.k_scale.cpu(), ks)
            assert torch.equal(a.v_scale[:, :, start:start + nb].cpu(), vs)
            ks, vs = ks[:, :, None, None], vs[..., None, None]
        else:
            ks, vs = ((x.abs().amax(dim=4) / 127.0).clamp_min(2.0 ** -24).half() for x in (kb, vb))
            lo, hi = start * 64, (start + nb) * 64
            assert torch.equal(a.k_tscale[:, :, lo:hi].cpu().view(ks.shape), ks)
            assert torch.equal(a.v_tscale[:, :, lo:hi].cpu().view(vs.shape), vs)
            ks, vs = ks.float()[..., None], vs.float()[..., None]
        for got, x, s in ((hk, kb, ks), (hv, vb, vs)):
            assert torch.equal(got.float(), torch.round(x / s).clamp(-127, 127))
    s = min(64, T)
    assert torch.equal(a.sink_k[:, :, :s].cpu(), k[:, :s].transpose(1, 2))
    assert torch.equal(a.sink_v[:, :, :s].cpu(), v[:, :s].transpose(1, 2))
    at = (slot + torch.arange(n)) % 128
    assert torch.equal(a.recent_k[:, :, at].cpu(), k[:, T - n:].transpose(1, 2))
    # the representatives are the oracle's, except where its winner and its
    # runner-up are nearer than fp32 sums can tell (equal ones, as padding and
    # zero keys are, fall to the first on both sides)
    reps = a.reps[:, :, start:start + nb].cpu().float()
    for layer in range(layers):
        sel, want, margins = O.build_reps(kb[layer].permute(1, 2, 0, 3).numpy(), r)
        assert all(len(set(row)) == r for row in sel.reshape(-1, r).tolist())    # no key twice
        clear = ~((margins > 0) & (margins <= 1e-5)).any(axis=2)                 # [nb, hkv]
        same = (reps[layer].numpy() == want).all(axis=(2, 3)).T
        # (the 2 keys of a last block lie at the same angle to their mean: not clear)
        assert same[clear].all(), np.argwhere(~same & clear)
        assert clear[:T // 64].sum() >= 0.8 * clear[:T // 64].size
    assert not a.hist_k[:, :, :start].any() and not a.hist_k[:, :, start + nb:].any()


@pytest.mark.parametrize("layers,T,hkv", [(1, 8191, 1), (1, 8192, 1), (2, 8193, 3), (1, 20000, 8), (1, 9001, 128)])
def test_key_scales_of_long_chunks(layers, T, hkv):
    """Few and many workgroups on both sides of the length from which a
    chunk's tokens are split over workgroups; stale scales do not count."""
    g = torch.Generator(device="cuda").manual_seed(T)
    k = torch.randn(layers, T, hkv, 128, generator=g, device="cuda").bfloat16()
    k[0, T - 1, 0, 3], k[0, 0, hkv - 1, 127], k[layers - 1, T // 2, 0, 64] = 50.0, -60.0, 70.0
    k[:, :, :, 9] = 0.0
    st = _store(layers, hkv, 1, "int8", -(-T // 64), sink=0, recent=64)
    st.k_scale.fill_(1e3)
    st.store_chunk(0, k, k, 0, True, False)
    assert torch.equal(st.k_scale.cpu(), k.float().abs().amax(dim=1).cpu().clamp_min(1e-8) / 127.0)   # (the CPU divides)


def test_recent_update_entry_moves_carried_slots():
    """nkv_recent_update with slots to move (old_len > carry > 0), around the ring's end."""
    st = _store(2, 3, 4, "bf16", 4)
    k, v = _kv(2, 200, 3, 9)
    R = 128
    for start, old, carry, n in [(0, 128, 120, 8), (77, 128, 63, 65), (127, 100, 28, 100), (5, 128, 128, 0)]:
        before = torch.randn(2, 3, R, 128).to(torch.bfloat16)
        st.recent_k.copy_(before)
        st.recent_v.copy_(-before)
        st.recent_update(0, 2, k.cuda(), v.cuda(), 3, n, start, old, carry)
        want = before.clone()
        i = torch.arange(carry)
        want[:, :, (start + i) % R] = before[:, :, (start + old - carry + i) % R]
        want_v = -want
        j = torch.arange(n)
        want[:, :, (start + carry + j) % R] = k[:, 3:3 + n].transpose(1, 2)
        want_v[:, :, (start + carry + j) % R] = v[:, 3:3 + n].transpose(1, 2)
        assert torch.equal(st.recent_k.cpu(), want) and torch.equal(st.recent_v.cpu(), want_v), (start, old, carry, n)


def test_ring_holds_the_last_tokens_through_chunks_commits_and_decodes():
    from nanokv_amd.sparse import M12Config, M12ModelRuntime
    cfg = M12Config(num_heads=4, num_kv_heads=2, max_model_len=8192, recent_tokens=128, top_k_blocks=4)
    rt = M12ModelRuntime(2, cfg)
    seen = []

    def tokens(n, seed):
        k, v = _kv(2, n, 2, seed)
        seen.extend(k.unbind(1))
        return k.cuda(), v.cuda()

    def check():
        core = rt.core
        n = min(128, core.valid_len)
        at = (core.ring_start + torch.arange(n)) % 128
        got = rt.store.recent_k[:, :, at].cpu()
        assert torch.equal(got, torch.stack(seen[-n:], 2))

    q = torch.randn(2, 8, 4, 128).to(torch.bfloat16).cuda()
    for i, n in enumerate([50, 40, 100, 3, 300, 64, 127, 129]):   # short, filling and overflowing chunks
        rt.prefill(*tokens(n, i))
        check()
    for i, (n, take) in enumerate([(6, 6), (6, 2), (8, 0), (5, 1)]):
        k, v = tokens(n, 100 + i)
        rt.verify(q[:, :n].contiguous(), k, v)
        rt.commit_verified(take)
        del seen[len(seen) - n + take:]
        check()
        k, v = tokens(1, 200 + i)
        rt.decode(q[:, :1].contiguous(), k, v)
        check()


def test_commit_keeps_a_device_ring_in_step():
    """A commit moves the ring start in device memory too, where a device-ring
    step reads it."""
    from nanokv_amd.sparse import M12Config, M12LayerRuntime
    cfg = M12Config(num_heads=4, num_kv_heads=2, max_model_len=8192, recent_tokens=128, top_k_blocks=4)
    k, v = _kv(1, 700, 2, 1)
    q = torch.randn(8, 4, 128).to(torch.bfloat16).cuda()
    outs = []
    for ring in (False, True):
        rt = M12LayerRuntime(0, cfg)
        rt.prefill_first(None, k[0].cuda(), v[0].cuda())
        rt.device_ring = ring
        o = []
        for i in range(3):
            o.append(rt.decode(q[:1], k[0, i:i + 1].cuda(), v[0, i:i + 1].cuda()))
            rt.verify_tokens(q[:5], k[0, 10:15].cuda(), v[0, 10:15].cuda())
            rt.commit_verified(3)
            c = rt._core
            assert not ring or c._ring_dev.tolist() == [c.ring_start]
        outs.append(o)
    for a, b in zip(*outs):
        assert torch.equal(a, b)


def test_commits_between_the_replays_of_a_captured_step():
    """A captured decode step reads the ring start from device memory: replays
    with verify commits between them, several full turns of the ring, against
    a runtime without device ring or graph."""
    from nanokv_amd.sparse import M12Config, M12LayerRuntime
    cfg = M12Config(num_heads=4, num_kv_heads=2, max_model_len=8192, recent_tokens=128, top_k_blocks=4)
    k, v = (x[0].cuda() for x in _kv(1, 700, 2, 1))
    g = torch.Generator().manual_seed(4)
    q = torch.randn(60, 4, 128, generator=g).to(torch.bfloat16).cuda()
    a, b = (M12LayerRuntime(0, cfg) for _ in range(2))
    for rt in (a, b):
        rt.prefill_first(None, k, v)
    b.device_ring = True
    ins = [x[:1].clone() for x in (q, k, v)]
    assert torch.equal(a.decode(*ins), b.decode(*ins))      # makes the ring and the workspaces
    state = b.decode_state()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = b.decode(*ins)
    b.restore_decode_state(state)
    for i in range(60):
        for x, src in zip(ins, (q, k, v)):
            x.copy_(src[i:i + 1])
        graph.replay()
        b.ring_replayed()
        want = a.decode(q[i:i + 1], k[i:i + 1], v[i:i + 1])
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(a.last_block_ids, b.last_block_ids), f"replay {i}"
        n = i % 7
        if n:
            lo = 70 + 8 * i
            outs = [rt.verify_tokens(q[:8], k[lo:lo + 8], v[lo:lo + 8]) for rt in (a, b)]
            for rt in (a, b):
                rt.commit_verified(n)
            assert torch.equal(*outs), f"round {i}"
    assert b._core._ring_dev.tolist() == [b._core.ring_start] == [a._core.ring_start]
    assert a.valid_len > 700 + 128


@pytest.mark.parametrize("layers,T,hq,nseg", [(1, 511, 32, 1), (1, 512, 32, 1), (1, 513, 3, 1), (3, 1100, 16, 2),
                                              (1, 4097, 32, 1), (5, 1030, 5, 2), (8, 700, 32, 1)])
def test_query_means_on_both_sides_of_the_launch_rule(layers, T, hq, nseg):
    """Few and many workgroups, short and long segments: the bf16 rounding of
    the exact mean (summed in fp64, where sums of these values are exact)."""
    from nanokv_amd.store import query_summaries
    q = torch.randn(layers, T, hq, 128, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16)
    out = query_summaries(q.cuda(), nseg).cpu()
    mean = torch.stack([p.double().mean(1) for p in q.tensor_split(nseg, dim=1)], 1)
    up, down = (torch.nextafter(mean.float(), torch.tensor(x)).to(torch.bfloat16) for x in (float("inf"), -float("inf")))
    near = mean.to(torch.bfloat16)
    # where fp32's own rounding cannot change the bf16 result the two agree
    sure = (up == near) & (down == near)
    assert torch.equal(out[sure], near[sure]) and float(sure.float().mean()) > 0.99
    assert bool(((out == up) | (out == down)).all())
