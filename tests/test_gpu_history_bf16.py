"""int8 prefill over the selected blocks' bf16 values, formed once per chunk
(nkv_history_bf16) instead of in every query tile."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _filled(layers, hq, hkv, fmt, nb, recent=128):
    from nanokv_amd.store import SparseKVStore
    st = SparseKVStore(layers, num_heads=hq, num_kv_heads=hkv, head_dim=128, block_size=64, r=4, cap_blocks=nb + 1,
                       sink_tokens=64, recent_tokens=recent, kv_format=fmt)
    g = torch.Generator(device="cuda").manual_seed(nb)
    k = torch.randn(layers, nb * 64 - 7, hkv, 128, generator=g, device="cuda").bfloat16()
    v = (torch.randn(layers, nb * 64 - 7, hkv, 128, generator=g, device="cuda") * 3).bfloat16()
    st.append(0, k, v, 0, True, True, 0, recent, 0)
    return st


@pytest.mark.parametrize("fmt", ["int8", "int8_token"])
def test_values_and_ids(fmt):
    st = _filled(3, 6, 3, fmt, 6)
    ids = torch.tensor([[5, 0, -1, 3, 99], [1, 1, 7, 4, -5]], dtype=torch.int32, device="cuda")
    desc, out_ids, (k, v) = st.history_bf16(1, 2, ids, 5, 4)   # layers 1 and 2, the first 4 ids of each
    assert out_ids.tolist() == [[0, 1, -1, 3], [0, 1, -1, 3]]
    assert (desc.cap_blocks, desc.num_layers, desc.kv_format) == (4, 2, 0)
    for layer in (0, 1):
        for i in range(4):
            b = int(ids[layer, i])
            if not 0 <= b < st.cap_blocks:
                continue
            for got, codes, name in ((k, st.hist_k, "k"), (v, st.hist_v, "v")):
                c = codes[layer + 1, :, b].float()
                if fmt == "int8_token":
                    s = getattr(st, name + "_tscale")[layer + 1, :, 64 * b:64 * b + 64].float().unsqueeze(-1)
                else:
                    s = st.k_scale[layer + 1].unsqueeze(1) if name == "k" else st.v_scale[layer + 1, :, b].view(-1, 1, 1)
                assert torch.equal(got[layer, :, i], (c * s).to(torch.bfloat16))


@pytest.mark.parametrize("layers,layer0,T,hq,hkv,fmt", [(1, 0, 300, 8, 2, "int8"), (3, 1, 97, 16, 1, "int8_token"),
                                                        (20, 0, 200, 32, 8, "int8")])
def test_attention_through_either_is_the_same(layers, layer0, T, hq, hkv, fmt):
    """Bit for bit, with ids outside the history among the selected ones."""
    nl = layers - layer0
    st = _filled(layers, hq, hkv, fmt, 9)
    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn(nl, T, h, 128, generator=g, device="cuda").bfloat16() for h in (hq, hkv, hkv))
    ids = torch.tensor([8, 2, -1, 5, 10, 0, 44], dtype=torch.int32, device="cuda").repeat(nl, 1).contiguous()
    n = 6
    part = torch.empty(st.prefill_workspace_floats(nl, T, 3), device="cuda")
    outs = [torch.full_like(q, float("nan")) for _ in range(2)]
    st.prefill_attend(layer0, q, k, v, ids, 7, n, None, 64, 17, 3, 100, 128 ** -0.5, outs[0], 0, 3, part)
    desc, ids2, keep = st.history_bf16(layer0, nl, ids, 7, n)
    st.prefill_attend(0, q, k, v, ids2, n, n, None, 64, 17, 3, 100, 128 ** -0.5, outs[1], 0, 3, part, desc)
    assert torch.equal(*outs) and bool(outs[0].isfinite().all())


def test_runtime_takes_the_form_its_rule_says():
    from nanokv_amd.sparse import M12Config, M12LayerRuntime
    cfg = M12Config(num_heads=16, num_kv_heads=2, max_model_len=4096, quant_history=True, top_k_blocks=6)
    rts = [M12LayerRuntime(0, cfg) for _ in range(2)]
    rts[0]._core.HISTORY_BF16_ROWS = 1 << 30
    assert rts[1]._core.HISTORY_BF16_ROWS == 2048
    g = torch.Generator(device="cuda").manual_seed(1)
    for T in (1500, 255, 256, 511):        # 2040 and 2048 rows on either side
        q, k, v = (torch.randn(T, h, 128, generator=g, device="cuda").bfloat16() for h in (16, 2, 2))
        if rts[0].prefill_len == 0:
            for rt in rts:
                rt.prefill_first(q, k, v)
        else:
            assert torch.equal(*[rt.prefill_chunk(q, k, v) for rt in rts])


def test_the_copy_is_bounded_and_never_needed():
    """A copy of more bytes than the limit, or more than the device has left,
    is not made: the attention forms the values in its tiles, with the same
    bits and without the memory."""
    from nanokv_amd.sparse import M12Config, M12ModelRuntime
    cfg = M12Config(num_heads=16, num_kv_heads=2, max_model_len=4096, quant_history=True, top_k_blocks=24)
    g = torch.Generator(device="cuda").manual_seed(2)
    k, v = (torch.randn(3, 2500, 2, 128, generator=g, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(3, 300, 16, 128, generator=g, device="cuda").bfloat16()
    size = 2 * 3 * 2 * 24 * 64 * 128 * 2   # K and V x layers x KV heads x blocks x tokens x dims x bytes
    assert 36 / 3 * 8 / 2 * 32 / 24 * size <= 512 << 20   # 36 layers, 8 KV heads, the default 32 blocks are within
    outs, made, peaks = [], [], []
    for limit in (size, size - 1, None):
        rt = M12ModelRuntime(3, cfg)
        rt.prefill(k, v)
        core, inner = rt.core, rt.store.history_bf16
        if limit is not None:
            core.HISTORY_BF16_BYTES = limit
        made.append(0)

        def counted(*args):
            made[-1] += 1
            if limit is None:
                raise torch.OutOfMemoryError("the device is full")
            return inner(*args)

        rt.store.history_bf16 = counted
        rt.prefill_chunk(q, k[:, :300].contiguous(), v[:, :300].contiguous())   # every workspace is there now
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        outs.append(rt.prefill_chunk(q, k[:, 300:600].contiguous(), v[:, 300:600].contiguous()))
        peaks.append(torch.cuda.max_memory_allocated() - before)
    assert made == [2, 0, 2]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    # (the allocator hands out whole cached blocks, up to 1 MiB larger than asked for)
    assert peaks[0] - max(peaks[1:]) > size - (2 << 20) > 0
