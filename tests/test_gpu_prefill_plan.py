"""The matrix-core prefill kernel's split plan (nkv_prefill_attend, splits > 1).

Tiles longer than the plan's piece size are cut into pieces whose partial
softmax states a merge kernel combines; the others write their output
directly.  Every split limit must give the plain causal attention in 64 bits:
|o - exact| <= u (|exact| + sum p |v| / l), u = 2^-8 (P and the output are
each rounded to bf16 once), +1 % and 1e-5 for the fp32 sums.  The records are
poisoned with NaN first, so a piece that is merged but was never written, or
written past its record, shows.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, keys_before):
    """q [T, hq, D]; k / v [hkv, keys_before + T, D] -> (exact, sum p |v| / l)."""
    T, hq, D = q.shape
    g = hq // k.shape[0]
    kk, vv = k.double().repeat_interleave(g, 0), v.double().repeat_interleave(g, 0)
    s = torch.matmul(q.double().transpose(0, 1), kk.transpose(1, 2)) * D ** -0.5
    hide = torch.triu(torch.ones(T, T, dtype=torch.bool, device=q.device), 1)
    s[:, :, keys_before:].masked_fill_(hide, float("-inf"))
    p = torch.softmax(s, dim=-1)
    return torch.matmul(p, vv).transpose(0, 1), torch.matmul(p, vv.abs()).transpose(0, 1)


# one tile and less, one more than a tile, ragged tiles of each width, several
# layers (layer index inside the plan), no history (tiles of 1 .. n segments)
# and a history (tiles of nearly equal length); one and two tiles of a long
# history (more pieces than runs in the plan's table); the last three have
# enough tiles for the 192-column kernel, in every history format
CASES = [(2, 40, 32, 8, 0, "bf16"), (1, 97, 32, 8, 0, "bf16"), (1, 700, 32, 8, 3, "bf16"),
         (3, 385, 16, 8, 0, "bf16"), (1, 1501, 32, 8, 0, "bf16"), (2, 509, 32, 2, 5, "int8"),
         (1, 130, 8, 8, 9, "int8_token"), (1, 260, 4, 4, 1, "bf16"), (1, 8, 16, 1, 300, "bf16"),
         (2, 13, 32, 2, 77, "int8"), (28, 200, 32, 8, 2, "bf16"), (28, 193, 32, 8, 2, "int8"),
         (16, 200, 64, 8, 1, "int8_token")]


@pytest.mark.parametrize("layers,T,hq,hkv,nhist,fmt", CASES)
def test_every_split_limit_gives_the_exact_attention(layers, T, hq, hkv, nhist, fmt):
    from nanokv_amd.store import SparseKVStore
    print(f"layers={layers} T={T} hq={hq} hkv={hkv} nhist={nhist} {fmt}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(layers * 1000 + T)

    def rand(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)

    st = SparseKVStore(layers, num_heads=hq, num_kv_heads=hkv, head_dim=128, block_size=64, r=4,
                       cap_blocks=max(nhist, 1), sink_tokens=64, recent_tokens=64, kv_format=fmt)
    hist = []   # the history as bf16 values
    for name in ("k", "v"):
        h = getattr(st, f"hist_{name}")
        if fmt == "bf16":
            h.copy_(rand(*h.shape))
            hist.append(h)
            continue
        h.copy_(torch.randint(-127, 128, h.shape, generator=g, device="cuda", dtype=torch.int32))
        if fmt == "int8_token":
            s = getattr(st, f"{name}_tscale")
            s.copy_(torch.rand(s.shape, generator=g, device="cuda") * 0.02 + 0.001)
            s = s.float().view(*h.shape[:4], 1)
        else:
            s = getattr(st, f"{name}_scale")
            s.copy_(torch.rand(s.shape, generator=g, device="cuda") * 0.02 + 0.001)
            s = s[:, :, None, None] if name == "k" else s[..., None, None]
        hist.append((h.float() * s).to(torch.bfloat16))
    q, k, v = rand(layers, T, hq, 128), rand(layers, T, hkv, 128), rand(layers, T, hkv, 128)
    ids = torch.arange(max(nhist, 1), dtype=torch.int32, device="cuda").repeat(layers, 1).contiguous()
    refs = []
    for layer in range(layers):
        kk = torch.cat((hist[0][layer, :, :nhist].reshape(hkv, -1, 128), k[layer].transpose(0, 1)), 1)
        vv = torch.cat((hist[1][layer, :, :nhist].reshape(hkv, -1, 128), v[layer].transpose(0, 1)), 1)
        refs.append(_reference(q[layer], kk, vv, 64 * nhist))
    for splits in (1, 2, 3, 7, 16, 64):
        n = st.prefill_workspace_floats(layers, T, splits)
        part = torch.full((max(n, 1),), float("nan"), device="cuda")
        out = torch.full_like(q, float("nan"))
        st.prefill_attend(0, q, k, v, ids, ids.shape[1], nhist, None, 0, 0, 0, 0, 128 ** -0.5, out, 0, splits, part)
        for layer, (o, pv) in enumerate(refs):
            err = (out[layer].double() - o).abs()
            bound = 2.0 ** -8 * (o.abs() + pv) * 1.01 + 1e-5
            assert bool((err <= bound).all()), (splits, layer, float((err / bound).max()))


@pytest.mark.parametrize("splits,least", [(64, 50), (16, 15), (5, 5)])
def test_one_tile_is_cut_as_finely_as_its_caller_allows(splits, least):
    """One query tile of 301 segments on an idle device: up to `splits` pieces
    (a record is written by its piece alone), not a fixed few long ones."""
    from nanokv_amd.store import SparseKVStore
    st = SparseKVStore(1, num_heads=16, num_kv_heads=1, head_dim=128, block_size=64, r=4, cap_blocks=300,
                       sink_tokens=64, recent_tokens=64)
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn(1, 8, h, 128, generator=g, device="cuda").to(torch.bfloat16) for h in (16, 1, 1))
    ids = torch.arange(300, dtype=torch.int32, device="cuda").view(1, 300)
    part = torch.full((st.prefill_workspace_floats(1, 8, splits),), float("nan"), device="cuda")
    st.prefill_attend(0, q, k, v, ids, 300, 300, None, 0, 0, 0, 0, 128 ** -0.5, torch.empty_like(q), 0, splits, part)
    assert least <= _written(part) <= splits


def _written(part):
    """Records that were written of a workspace filled with NaN."""
    size = 128 * 132   # a record: 128 (token, head) columns of m, l, two of padding, 128 sums
    records = part[:part.numel() // size * size].view(-1, 128, 132)
    return int((~records[:, 0, 0].isnan()).sum())


def test_union_selections_are_cut_as_finely_as_their_caller_allows():
    """A union's list ends in ids that attend nothing: pieces sized by the
    list's length alone would leave most of them idle."""
    from nanokv_amd.store import SparseKVStore
    layers, hkv, nhist, splits = 17, 4, 392, 23
    st = SparseKVStore(layers, num_heads=32, num_kv_heads=hkv, head_dim=128, block_size=64, r=4, cap_blocks=64,
                       sink_tokens=64, recent_tokens=64)
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn(layers, 8, h, 128, generator=g, device="cuda").to(torch.bfloat16) for h in (32, hkv, hkv))
    st.hist_k.normal_(generator=g)
    st.hist_v.normal_(generator=g)
    ids = torch.full((layers, nhist), -1, dtype=torch.int32, device="cuda")
    ids[:, :60] = torch.arange(60, device="cuda")
    allowed = torch.zeros(layers, 8, nhist, dtype=torch.uint8, device="cuda")
    allowed[:, :, :60] = torch.rand(layers, 8, 60, generator=g, device="cuda") < 0.5
    part = torch.full((st.prefill_workspace_floats(layers, 8, splits),), float("nan"), device="cuda")
    out = torch.empty_like(q)
    st.prefill_attend(0, q, k, v, ids, nhist, nhist, allowed, 0, 0, 0, 0, 128 ** -0.5, out, 8 * nhist, splits, part)
    # (pieces of ids that attend nothing write a record of weight 0, not NaN)
    assert _written(part) >= 20 * layers * hkv
    for layer in (0, layers - 1):
        kk = torch.cat((st.hist_k[layer, :, :60].reshape(hkv, -1, 128), k[layer].transpose(0, 1)), 1).double()
        vv = torch.cat((st.hist_v[layer, :, :60].reshape(hkv, -1, 128), v[layer].transpose(0, 1)), 1).double()
        s = torch.matmul(q[layer].double().transpose(0, 1), kk.repeat_interleave(8, 0).transpose(1, 2)) * 128 ** -0.5
        hide = torch.zeros(8, 60 * 64 + 8, dtype=torch.bool, device="cuda")
        hide[:, :60 * 64] = (allowed[layer, :, :60] == 0).repeat_interleave(64, 1)
        hide[:, 60 * 64:] = torch.triu(torch.ones(8, 8, dtype=torch.bool, device="cuda"), 1)
        p = torch.softmax(s.masked_fill(hide, float("-inf")), -1)
        o, pv = (torch.matmul(p, x.repeat_interleave(8, 0)).transpose(0, 1) for x in (vv, vv.abs()))
        err = (out[layer].double() - o).abs()
        assert bool((err <= 2.0 ** -8 * (o.abs() + pv) * 1.01 + 1e-5).all())


@pytest.mark.parametrize("splits", [2, 3, 5, 6, 7, 10])
def test_an_infinite_value_stays_one_through_the_merge(splits):
    """An infinite value in a tile's last piece is attended by the queries from
    it on: their outputs are infinite there, with any number of pieces."""
    from nanokv_amd.store import SparseKVStore
    st = SparseKVStore(1, num_heads=4, num_kv_heads=1, head_dim=128, block_size=64, r=4, cap_blocks=40,
                       sink_tokens=64, recent_tokens=64)
    g = torch.Generator(device="cuda").manual_seed(1)

    def rand(*shape):
        return (0.1 * torch.randn(*shape, generator=g, device="cuda")).to(torch.bfloat16)

    st.hist_k.copy_(rand(*st.hist_k.shape))
    st.hist_v.copy_(rand(*st.hist_v.shape))
    q, k, v = rand(1, 20, 4, 128), rand(1, 20, 1, 128), rand(1, 20, 1, 128)
    v[0, 0, 0, 5], v[0, 0, 0, 77] = float("inf"), -float("inf")    # every query sees chunk token 0
    ids = torch.arange(40, dtype=torch.int32, device="cuda").view(1, 40)
    part = torch.empty(st.prefill_workspace_floats(1, 20, splits), device="cuda")
    out = torch.empty_like(q)
    st.prefill_attend(0, q, k, v, ids, 40, 40, None, 0, 0, 0, 0, 128 ** -0.5, out, 0, splits, part)
    assert bool((out[..., 5] == float("inf")).all()) and bool((out[..., 77] == -float("inf")).all())
    rest = [d for d in range(128) if d not in (5, 77)]
    assert bool(out[..., rest].isfinite().all())
