"""A decode token of a decoder layer whose modules were replaced or overridden.

The fused norm + projection stands for calls of this package's own modules
only: with any of them replaced (a subclass, an adapter wrapper, another
module, a forward assigned on the instance), the layer must call what is
there.  The device functions are stood in for by their tensor formulas, so
the routing is checked without a GPU.
"""

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from nanokv_amd import qwen3

CFG = qwen3.Qwen3Config(vocab_size=64, hidden_size=256, intermediate_size=384, num_hidden_layers=1,
                        num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=64)


class _Mean(nn.Module):
    """Stands for the sparse attention: each query head gets its KV head's value."""

    def forward(self, q, k, v):
        return v.repeat_interleave(q.shape[1] // v.shape[1], dim=1)


class _Adapter(nn.Module):
    """A wrapper that shows the wrapped module's parameters and adds a term."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner
        self.weight, self.bias = inner.weight, getattr(inner, "bias", None)
        self.eps = getattr(inner, "eps", None)

    def forward(self, *args):
        y = self.inner(*args)
        return (y[0] + 1, *y[1:]) if isinstance(y, tuple) else y + 1


class _Bare(nn.Module):
    """A replacement with neither weight, bias nor eps."""

    def __init__(self, inner):
        super().__init__()
        self.inner = nn.ModuleList([inner])

    def forward(self, *args):
        return self.inner[0](*args)


class _OtherMLP(nn.Module):
    """An MLP of another structure."""

    def __init__(self, n):
        super().__init__()
        self.proj = nn.Linear(n, n)

    def forward(self, x):
        return self.proj(x)


def _subclass(m):
    base = type(m)

    class Sub(base):
        def forward(self, *args):
            y = super().forward(*args)
            return (y[0] * 2, *y[1:]) if isinstance(y, tuple) else y * 2

    m.__class__ = Sub
    return m


def _on_instance(m):
    inner = m.forward
    m.forward = lambda *args: inner(*args)
    return m


@pytest.fixture
def fused(monkeypatch):
    """The fused calls as tensor formulas, accepted for any one-row CPU tensor; counts them."""
    calls = []

    def norm_gemv(x, residual, w, eps, weight, silu_mul=False):
        calls.append(silu_mul)
        s = x.float() if residual is None else x.float() + residual.float()
        h = (s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + eps)).to(x.dtype) * w
        y = F.linear(h, weight)
        if silu_mul:
            gate, up = y.chunk(2, dim=-1)
            y = F.silu(gate) * up
        return y, x if residual is None else s.to(x.dtype)

    def gemv_silu(x, weight):
        gate, up = F.linear(x, weight).chunk(2, dim=-1)
        return F.silu(gate) * up

    monkeypatch.setattr(qwen3, "_gemv_ok", lambda x, weight: x.dim() == 2 and x.shape[0] == 1)
    monkeypatch.setattr(qwen3, "gemv_dev", F.linear)
    monkeypatch.setattr(qwen3, "gemv_silu_mul_dev", gemv_silu)
    monkeypatch.setattr(qwen3, "norm_gemv_dev", norm_gemv)
    return calls


def _layer():
    torch.manual_seed(1)
    layer = qwen3.Qwen3DecoderLayer(CFG, 64).to(torch.bfloat16).requires_grad_(False)
    qwen3.init_random_(layer, 2)
    layer.self_attn.attn = _Mean()
    return layer


def _replaced():
    """(name, layer, fused calls that remain)"""
    for path, other in (("input_layernorm", 1), ("self_attn.qkv_proj", 1), ("post_attention_layernorm", 1),
                        ("mlp.gate_up_proj", 1), ("self_attn", 1), ("mlp", 1)):
        for name, change in (("adapter", _Adapter), ("bare", _Bare), ("subclass", _subclass),
                             ("instance", _on_instance)):
            if name in ("adapter", "bare") and path in ("self_attn", "mlp", "mlp.gate_up_proj"):
                continue
            layer = _layer()
            parent, _, leaf = path.rpartition(".")
            owner = layer.get_submodule(parent)
            setattr(owner, leaf, change(getattr(owner, leaf)))
            yield f"{path}/{name}", layer, other
    layer = _layer()
    layer.mlp = _OtherMLP(CFG.hidden_size).to(torch.bfloat16)
    yield "mlp/other", layer, 1


def _token(layer):
    g = torch.Generator().manual_seed(5)
    h, res = (torch.randn(1, CFG.hidden_size, generator=g).to(torch.bfloat16) for _ in range(2))
    return layer(torch.tensor([7]), h, res)


def _modulewise(layer):
    """The layer's own definition: every module called."""
    g = torch.Generator().manual_seed(5)
    h, res = (torch.randn(1, CFG.hidden_size, generator=g).to(torch.bfloat16) for _ in range(2))
    h, res = layer.input_layernorm(h, res)
    h = layer.self_attn(torch.tensor([7]), h)
    h, res = layer.post_attention_layernorm(h, res)
    return layer.mlp(h), res


def test_own_modules_take_both_fused_calls(fused):
    layer = _layer()
    got = _token(layer)
    assert fused == [False, True]
    for a, b in zip(got, _modulewise(layer)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name,layer,left", _replaced(), ids=lambda x: x if isinstance(x, str) else "")
def test_a_replaced_module_is_called(fused, name, layer, left):
    got = _token(layer)
    assert len(fused) == left
    for a, b in zip(got, _modulewise(layer)):
        assert torch.equal(a, b)


def test_a_forward_patched_on_the_class_is_called(fused, monkeypatch):
    layer = _layer()
    inner = qwen3.RMSNorm.forward
    monkeypatch.setattr(qwen3.RMSNorm, "forward", lambda self, *a: inner(self, *a))
    got = _token(layer)
    assert fused == []
    for a, b in zip(got, _modulewise(layer)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("change", [_Adapter, _Bare, _subclass, _on_instance])
def test_the_mlp_calls_a_replaced_gate_up_projection(fused, change):
    mlp = _layer().mlp
    mlp.gate_up_proj = change(mlp.gate_up_proj)
    x = torch.randn(1, CFG.hidden_size, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    gate, up = mlp.gate_up_proj(x).chunk(2, dim=-1)
    assert torch.equal(mlp(x), mlp.down_proj(F.silu(gate) * up))


@pytest.mark.parametrize("leaf", ["q_norm", "k_norm"])
@pytest.mark.parametrize("change", [_Adapter, _Bare, _subclass, _on_instance])
def test_attention_calls_a_replaced_head_norm(fused, monkeypatch, leaf, change):
    attn = _layer().self_attn
    setattr(attn, leaf, change(getattr(attn, leaf)))
    qkv = torch.randn(3, attn.qkv_proj.out_features, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    want = attn.attend(torch.arange(3), qkv)            # CPU tensors: module by module
    monkeypatch.setattr(qwen3, "_fused", lambda t: t.dtype == torch.bfloat16 and t.shape[-1] > CFG.head_dim)
    monkeypatch.setattr(qwen3, "qk_norm_rope_dev", lambda *a: pytest.fail("the replaced norm was skipped"))
    monkeypatch.setattr(qwen3, "rmsnorm_dev", lambda *a: pytest.fail("a head norm of the CPU path"))
    assert torch.equal(attn.attend(torch.arange(3), qkv), want)
