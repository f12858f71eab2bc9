"""The per-layer runtime's one-call decode and its ids kept on the device."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _kv(n, hkv, seed):
    g = torch.Generator().manual_seed(seed)
    return tuple((torch.randn(n, hkv, 128, generator=g) * 128 ** -0.5).to(torch.bfloat16).cuda() for _ in range(2))


@pytest.mark.parametrize("hq,hkv,T,fmt", [(32, 8, 700, "bf16"), (64, 8, 3000, "int8"), (16, 1, 1300, "token"),
                                          (4, 4, 100, "bf16"), (8, 4, 64 * 2100, "bf16")])
def test_one_call_decode_equals_select_then_attend(hq, hkv, T, fmt):
    """Bit for bit, over heads per KV head 1 to 16, short windows, rows past the
    step form (more than 2048 blocks) and with the profiling switch that takes
    the two-call path."""
    from nanokv_amd.sparse import M12Config, M12LayerRuntime
    cfg = M12Config(num_heads=hq, num_kv_heads=hkv, max_model_len=T + 64, quant_history=fmt != "bf16",
                    quant_scale_layout="token" if fmt == "token" else "channel_block")
    k, v = _kv(T, hkv, T)
    nk, nv = _kv(6, hkv, 1)
    q = torch.randn(6, hq, 128, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    rts = [M12LayerRuntime(0, cfg) for _ in range(2)]
    rts[1].profile_torch_stages = True
    for rt in rts:
        rt.prefill_first(None, k, v)
    for i in range(6):
        a, b = (rt.decode(q[i:i + 1], nk[i:i + 1], nv[i:i + 1]) for rt in rts)
        assert torch.equal(a, b)
        assert torch.equal(rts[0].last_block_ids, rts[1].last_block_ids)
        assert set(rts[0].timings) == set(rts[1].timings)
        if i == 2:   # a chunk between: the kept launch arguments change
            for rt in rts:
                rt.prefill_chunk(q[:5], nk[:5], nv[:5])
    assert torch.equal(rts[0].store.recent_k, rts[1].store.recent_k)
    assert not rts[0]._core._ws["keys"].any()


@pytest.mark.parametrize("T", [700, 64 * 600])   # the top-k inside the attention launch, and a launch of its own
def test_timings_tell_the_selection_from_the_attention(T):
    from time import perf_counter

    from nanokv_amd.sparse import M12Config, M12LayerRuntime
    rt = M12LayerRuntime(0, M12Config(num_heads=8, num_kv_heads=2, max_model_len=T + 64))
    rt.prefill_first(None, *_kv(T, 2, T))
    q = torch.randn(1, 8, 128, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).cuda()
    nk, nv = _kv(1, 2, 1)
    for _ in range(3):
        t0 = perf_counter()
        rt.decode(q, nk, nv)
        wall = (perf_counter() - t0) * 1000.0
        t = rt.timings
        assert t["selector_ms"] == t["selector_enqueue_ms"] > 0.0 and t["packed_attn_ms"] > 0.0
        assert t["selector_ms"] + t["packed_attn_ms"] <= wall


def test_prefill_ids_survive_later_selections_and_streams():
    from nanokv_amd.sparse import M12Config, M12LayerRuntime
    cfg = M12Config(num_heads=8, num_kv_heads=2, max_model_len=8192, top_k_blocks=8)
    rt = M12LayerRuntime(0, cfg)
    k, v = _kv(2048, 2, 5)
    g = torch.Generator().manual_seed(3)
    q = torch.randn(256, 8, 128, generator=g).to(torch.bfloat16).cuda()
    rt.prefill_first(None, k, v)
    want = rt._gpu_select(torch.stack([q.double().mean(0)]).to(torch.bfloat16))[0]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        rt.prefill_chunk(q, k[:256], v[:256])
    held = rt._last_prefill_ids
    torch.cuda.current_stream().wait_stream(side)
    rt.decode(q[:1], k[:1], v[:1])              # overwrites the selection workspace
    assert rt.last_prefill_block_ids.dtype == torch.int64 and not rt.last_prefill_block_ids.is_cuda
    assert torch.equal(rt.last_prefill_block_ids, want)
    rt.last_prefill_block_ids.zero_()           # a reader's edit reaches nobody else
    assert torch.equal(held.cpu(), want)
    rt.verify_tokens(q[:4], k[:4], v[:4])
    ids = rt.last_verify_block_ids
    assert torch.equal(rt.last_block_ids, ids) and ids.numel() == 8
    rt.reset()
    assert rt.last_prefill_block_ids is None and rt.last_block_ids is None


@pytest.mark.parametrize("nb,top_k,fmt", [(1, 4, "bf16"), (3, 32, "int8"), (10, 1, "bf16"), (33, 64, "token"),
                                          (511, 64, "bf16"), (512, 32, "int8"), (513, 32, "bf16"), (90, 65, "bf16")])
@pytest.mark.parametrize("layers", [1, 3])
def test_step_with_its_selection_inside_equals_the_separate_launches(layers, nb, top_k, fmt):
    """nkv_decode_step (its top-k inside the attention launch at these sizes,
    up to 512 blocks and 64 ids) against nkv_select + nkv_attend: ids, outputs
    and the ring bit for bit, the keys cleared, ids past the selectable blocks
    untouched; equal scores break to the lower block."""
    from nanokv_amd.sparse import M12Config, M12ModelRuntime
    cfg = M12Config(num_heads=8, num_kv_heads=2, max_model_len=nb * 64, top_k_blocks=top_k, quant_history=fmt != "bf16",
                    quant_scale_layout="token" if fmt == "token" else "channel_block", attend_splits=5)
    rts = [M12ModelRuntime(layers, cfg) for _ in range(2)]
    k, v = _kv(layers * (nb * 64 - 5), 2, nb)
    for rt in rts:
        rt.prefill(k.view(layers, -1, 2, 128), v.view(layers, -1, 2, 128))
        rt.store.reps[:, :, nb // 2:] = rt.store.reps[:, :, nb // 2:nb // 2 + 1]     # ties
    g = torch.Generator().manual_seed(nb)
    for i in range(3):
        q = torch.randn(layers, 1, 8, 128, generator=g).to(torch.bfloat16).cuda()
        nk, nv = (x.view(layers, 1, 2, 128) for x in _kv(layers, 2, 100 + i))
        a = rts[0].decode(q, nk, nv)
        core = rts[1].core
        ids, _, n = core.select(q, top_k)
        b, _, _ = core.decode_attend(q, nk, nv, ids, ids.shape[-1], n)
        assert torch.equal(a, b)
        assert rts[0].last_n_selected == n
        assert torch.equal(rts[0].last_ids_dev[:, 0, :n], ids[:, 0, :n])
        assert torch.equal(rts[0].store.recent_k, rts[1].store.recent_k)
        assert not rts[0].core._ws["keys/step"].any()


@pytest.mark.parametrize("recent", [64, 512, 8192])
def test_protected_lists_of_the_store_table_and_of_a_store_without_one(recent, monkeypatch):
    """The table's rows, histories shorter than the window among them, and the
    lists copied from the host where the table would be too large."""
    from nanokv_amd.sparse import M12Config, M12LayerRuntime
    from nanokv_amd.store import SparseKVStore
    cfg = M12Config(num_heads=8, num_kv_heads=2, max_model_len=8192, recent_tokens=recent, top_k_blocks=4)
    with_table = M12LayerRuntime(0, cfg)
    n = min(recent // 64, 128)
    rows = with_table.store.protected_rows(n).cpu()
    for nb in range(1, 129):
        want = [0, *range(max(1, nb - n), nb)]
        assert rows[nb].tolist() == want + [0] * (1 + n - len(want))
    monkeypatch.setattr(SparseKVStore, "PROTECTED_ROWS_BYTES", 4 * 129 * (1 + n) - 1)
    without = M12LayerRuntime(0, cfg)
    assert without.store.protected_rows(n) is None
    for i, T in enumerate((70, 130, 1000, 500)):
        k, v = _kv(T, 2, T)
        q = torch.randn(1, 8, 128, generator=torch.Generator().manual_seed(i)).to(torch.bfloat16).cuda()
        outs = []
        for rt in (with_table, without):
            (rt.prefill_first if i == 0 else rt.prefill_chunk)(q.expand(T, 8, 128), k, v)
            outs.append((rt.decode(q, k[:1], v[:1]), rt.last_block_ids))
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
