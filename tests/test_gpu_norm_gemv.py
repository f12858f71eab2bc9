"""RMSNorm + GEMV in one launch (nkv_norm_gemv, nkv_norm_gemv_silu_mul).

The normalised row and the residual are those of nkv_rmsnorm bit for bit; the
product is bounded as the plain GEMV's is: |y - x.W^T| <= 2^-8 |x.W^T| (bf16
output) + 2^-22 sum |x||W| (fp32 accumulation, generous).
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

# k at the edges of a lane's chunks (512 dims each); n odd, one row pair, more
# pairs than one round of wavefronts
SHAPES = [(1, 8), (2, 504), (7, 512), (513, 520), (64, 1024), (33, 1032), (6144, 2560), (9, 2568), (20001, 1536),
          (1003, 4096)]


def _operands(n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(1, k, generator=g, device="cuda").bfloat16()
    res = (torch.randn(1, k, generator=g, device="cuda") * 2).bfloat16()
    nw = (1 + 0.1 * torch.randn(k, generator=g, device="cuda")).bfloat16()
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.05).bfloat16()
    return x, res, nw, w


@pytest.mark.parametrize("with_residual", [False, True])
@pytest.mark.parametrize("n,k", SHAPES)
def test_norm_gemv_is_the_norm_then_the_product(n, k, with_residual):
    from nanokv_amd.qwen3 import norm_gemv_dev, rmsnorm_dev
    x, res, nw, w = _operands(n, k, n + k)
    if with_residual:
        xn, want = rmsnorm_dev(x, nw, 1e-6, res)
    else:
        xn, want, res = rmsnorm_dev(x, nw, 1e-6), x, None
    y, got = norm_gemv_dev(x, res, nw, 1e-6, w)
    assert torch.equal(got, want)
    ref = xn.double() @ w.double().T
    mag = xn.double().abs() @ w.double().abs().T
    err = (y.double() - ref).abs()
    assert bool((err <= 2.0 ** -8 * ref.abs() + 2.0 ** -22 * mag + 1e-30).all())


@pytest.mark.parametrize("inter,k", [(1, 8), (3, 520), (1001, 1024), (9728, 2560), (515, 4096)])
def test_norm_gemv_silu_mul_rounds_where_the_launches_do(inter, k):
    """gate and up are rounded to bf16, silu(gate) to bf16, then the product:
    recomputed from the 64-bit products, an output may differ only where one
    of them lies within the fp32 accumulation error of a rounding boundary."""
    from nanokv_amd.qwen3 import norm_gemv_dev, rmsnorm_dev
    x, res, nw, w = _operands(2 * inter, k, inter + k)
    xn, want = rmsnorm_dev(x, nw, 1e-6, res)
    y, got = norm_gemv_dev(x, res, nw, 1e-6, w, silu_mul=True)
    assert torch.equal(got, want)
    gate, up = (xn.double() @ w.double().T).to(torch.bfloat16).chunk(2, dim=-1)
    ref = torch.nn.functional.silu(gate) * up
    same = (y == ref).float().mean()
    assert float(same) > 0.98 or inter < 50
    # one bf16 step of gate, of silu and of the product
    assert bool(((y.double() - ref.double()).abs() <= 2.0 ** -6 * ref.double().abs() + 1e-6).all())


def test_decoder_layer_takes_the_fused_norms_only_without_hooks():
    from nanokv_amd import qwen3
    from nanokv_amd.attention import attach_m12_runtimes, set_context
    from nanokv_amd.sparse import M12Config
    cfg = qwen3.Qwen3Config(hidden_size=1024, intermediate_size=3072, num_hidden_layers=1, num_attention_heads=16)
    torch.manual_seed(0)
    with torch.device("cuda"):
        layer = qwen3.Qwen3DecoderLayer(cfg, 2048).to(torch.bfloat16).requires_grad_(False)
    qwen3.init_random_(layer, 3)
    h = torch.randn(701, 1024, device="cuda").bfloat16()
    res = torch.randn(701, 1024, device="cuda").bfloat16()
    pos = torch.arange(701, device="cuda")
    rt = attach_m12_runtimes(layer, M12Config(num_heads=16, max_model_len=1024), "cuda")[0]
    outs = []
    for hook in (False, True):
        rt.reset()
        set_context(True, max_seqlen_q=700)
        layer(pos[:700], h[:700], res[:700])
        seen = []
        handles = [m.register_forward_hook(lambda *a: seen.append(1)) for m in
                   (layer.input_layernorm, layer.mlp)] if hook else []
        set_context(False, max_seqlen_q=1)
        outs.append(layer(pos[700:], h[700:].clone(), res[700:].clone()))
        assert len(seen) == (2 if hook else 0)
        for x in handles:
            x.remove()
    for a, b in zip(*outs):   # roundings of one layer in bf16
        assert float((a.double() - b.double()).norm()) <= 1e-2 * float(b.double().norm())


@pytest.mark.parametrize("rows,hq,hkv", [(1, 32, 8), (63, 16, 8), (64, 1, 1), (65, 5, 2), (257, 4, 4)])
def test_qk_norm_rope_is_the_same_for_aligned_and_unaligned_operands(rows, hq, hkv):
    """The 16-byte form and the one for unaligned operands give the same bits."""
    from nanokv_amd.qwen3 import _rope_table, qk_norm_rope_dev
    g = torch.Generator(device="cuda").manual_seed(rows)
    n = rows * (hq + 2 * hkv) * 128
    store = torch.empty(n + 8, dtype=torch.bfloat16, device="cuda")
    qkv = torch.randn(n, generator=g, device="cuda").bfloat16()
    qw, kw = ((1 + 0.1 * torch.randn(128, generator=g, device="cuda")).bfloat16() for _ in range(2))
    cos, sin = _rope_table(128, 1e6, 512, "cuda")
    pos = torch.randint(-3, 600, (rows,), generator=g, device="cuda")   # clamped to the table
    outs = []
    for off in (0, 1, 8):
        x = store[off:off + n]
        x.copy_(qkv)
        assert x.data_ptr() % 16 == (2 * off) % 16
        outs.append(qk_norm_rope_dev(x.view(rows, -1), pos, hq, hkv, qw, kw, 1e-6, cos, sin))
    for other in outs[1:]:
        for a, b in zip(outs[0], other):
            assert torch.equal(a, b)


def test_a_wrapped_projection_adds_its_term_at_decode():
    """A low-rank adapter around qkv_proj counts for the prompt and for the token."""
    from nanokv_amd import qwen3
    from nanokv_amd.attention import attach_m12_runtimes, set_context
    from nanokv_amd.sparse import M12Config

    class Adapter(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner, self.weight, self.bias = inner, inner.weight, None
            self.down = torch.randn(4, inner.in_features, device="cuda").bfloat16() * 0.05
            self.up = torch.randn(inner.out_features, 4, device="cuda").bfloat16()

        def forward(self, x):
            return self.inner(x) + x @ self.down.T @ self.up.T

    cfg = qwen3.Qwen3Config(hidden_size=1024, intermediate_size=3072, num_hidden_layers=1, num_attention_heads=16)
    torch.manual_seed(0)
    with torch.device("cuda"):
        layer = qwen3.Qwen3DecoderLayer(cfg, 2048).to(torch.bfloat16).requires_grad_(False)
    qwen3.init_random_(layer, 3)
    qkv = layer.self_attn.qkv_proj
    layer.self_attn.qkv_proj = adapter = Adapter(qkv)
    merged = qwen3.Linear(qkv.in_features, qkv.out_features, bias=False, device="cuda", dtype=torch.bfloat16)
    merged.weight = torch.nn.Parameter((qkv.weight.double() + adapter.up.double() @ adapter.down.double()).bfloat16(),
                                       requires_grad=False)
    h, res = (torch.randn(701, 1024, device="cuda").bfloat16() for _ in range(2))
    pos = torch.arange(701, device="cuda")
    rt = attach_m12_runtimes(layer, M12Config(num_heads=16, max_model_len=1024), "cuda")[0]
    outs = []
    for proj in (adapter, merged, qkv):
        layer.self_attn.qkv_proj = proj
        rt.reset()
        set_context(True, max_seqlen_q=700)
        layer(pos[:700], h[:700], res[:700])
        set_context(False, max_seqlen_q=1)
        outs.append(layer(pos[700:], h[700:].clone(), res[700:].clone())[0].double())
    far = float((outs[2] - outs[1]).norm())
    assert float((outs[0] - outs[1]).norm()) <= 0.1 * far   # the term is far above the roundings of a layer
    assert far > 0.05 * float(outs[1].norm())


@pytest.mark.parametrize("k", [8, 504, 520, 1016, 1032, 1800, 2048, 2568, 3080, 4088])
def test_an_infinite_weight_gives_an_infinity(k):
    """A row's chunks are padded up to a whole number a lane: the padding must
    add nothing, also where the row's last columns are infinite."""
    from nanokv_amd.qwen3 import gemv_dev, norm_gemv_dev, rmsnorm_dev
    x, res, nw, w = _operands(40, k, k)
    w[3, k - 8:] = float("inf")
    w[4, k - 1] = -float("inf")
    w[25, 0] = float("inf")
    w[37, k - 3] = float("nan")
    x = x.abs() + 0.5     # no zero meets an infinity
    res = res.abs()
    xn, _ = rmsnorm_dev(x, nw, 1e-6, res)
    want = gemv_dev(xn, w)
    y, _ = norm_gemv_dev(x, res, nw, 1e-6, w)
    assert bool(want[0, 3].isinf()) and bool(want[0, 4].isinf()) and bool(want[0, 37].isnan())
    odd = ~want.isfinite()
    assert torch.equal(odd, ~y.isfinite()) and torch.equal(torch.nan_to_num(y[odd]), torch.nan_to_num(want[odd]))
    z, _ = norm_gemv_dev(x, res, nw, 1e-6, w, silu_mul=True)      # gate rows 0 .. 19, up rows 20 .. 39
    gate, up = want.chunk(2, dim=-1)
    ref = torch.nn.functional.silu(gate) * up
    odd = ~ref.isfinite()
    assert torch.equal(odd, ~z.isfinite()) and torch.equal(torch.nan_to_num(z[odd]), torch.nan_to_num(ref[odd]))
