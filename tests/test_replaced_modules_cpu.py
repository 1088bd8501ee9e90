"""Blocks whose modules were replaced, subclassed or hooked call them: the
fused forms (SiLU in the projection's kernel, embedding and RoPE rows in one
launch) answer only for the modules that the framework builds. On the CPU,
with the kernels' wrappers standing in as plain torch."""
import pytest
import torch
import torch.nn.functional as F
from torch import nn

from tinyvllm import layers
from tinyvllm.models import qwen3

CONFIG = qwen3.Qwen3Config(
    vocab_size=64, hidden_size=64, intermediate_size=96, num_hidden_layers=1,
    max_position_embeddings=32, num_attention_heads=2, num_key_value_heads=1, head_dim=32,
    rms_norm_eps=1e-6, rope_theta=1e4, tie_word_embeddings=True)


def _silu_and_mul(x):
    gate, up = x.chunk(2, -1)
    return F.silu(gate) * up


@pytest.fixture
def fused_calls(monkeypatch):
    """Lets CPU calls take the fused forms, and counts them."""
    calls = []

    def linear(x, weight, *, slices=0, silu=False):
        calls.append("silu" if silu else "plain")
        y = F.linear(x, weight)
        return _silu_and_mul(y) if silu else y[None] if slices else y

    monkeypatch.setattr(layers.few_rows, "fits", lambda x, w: not torch.is_grad_enabled())
    monkeypatch.setattr(layers.few_rows, "few_rows_linear", linear)
    monkeypatch.setattr(layers, "silu_and_mul", _silu_and_mul)
    return calls


def _value(y):
    return y.materialize() if isinstance(y, layers.SplitKPartials) else y


class _Wrapper(nn.Module):
    """Any module around a projection, with none of its other methods."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        return self.inner(x) + 1.0


class _Doubled(layers.PackedLinear):
    def forward(self, x):
        return 2.0 * super().forward(x)


def _gelu_and_mul(x):
    gate, up = x.chunk(2, -1)
    return F.gelu(gate) * up


def _replace(mlp, what, seen):
    if what == "act_fn":
        mlp.act_fn = nn.Module()
        mlp.act_fn.forward = _gelu_and_mul
    elif what == "act_fn.forward":
        mlp.act_fn.forward = _gelu_and_mul
    elif what == "wrapped":
        mlp.gate_up_proj = _Wrapper(mlp.gate_up_proj)
    elif what == "subclass":
        new = _Doubled(64, (96, 96))
        new.weight = mlp.gate_up_proj.weight
        mlp.gate_up_proj = new
    elif what == "hook":
        mlp.act_fn.register_forward_hook(lambda m, a, y: seen.append(m) or y + 1.0)
    elif what == "pre_hook":
        mlp.gate_up_proj.register_forward_pre_hook(lambda m, a: seen.append(m) or (a[0] * 2,))
    elif what == "global_hook":
        return nn.modules.module.register_module_forward_hook(
            lambda m, a, y: seen.append(m) if m is mlp.act_fn else None)
    return None


@pytest.mark.parametrize("what", ["act_fn", "act_fn.forward", "wrapped", "subclass", "hook",
                                  "pre_hook", "global_hook"])
def test_mlp_calls_what_was_put_in(fused_calls, what):
    torch.manual_seed(0)
    mlp = qwen3.Qwen3MLP(CONFIG)
    x = torch.randn(3, 64)
    with torch.no_grad():
        mlp(x)
        assert "silu" in fused_calls  # as built: the fused form
        seen = []
        handle = _replace(mlp, what, seen)
        try:
            got = _value(mlp(x))
            expect = _value(mlp.down_proj(mlp.act_fn(mlp.gate_up_proj(x))))
            torch.testing.assert_close(got, expect)
            assert "hook" not in what or len(seen) == 2
        finally:
            if handle is not None:
                handle.remove()


@pytest.mark.parametrize("what", ["embed", "rope", "max_norm", "global_hook"])
def test_embedding_calls_what_was_put_in(monkeypatch, what):
    def fused(*args):
        raise AssertionError("the fused gather answered for a replaced module")

    monkeypatch.setattr(qwen3, "embed_rope", fused)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    model = qwen3.Qwen3Model(CONFIG, dtype=torch.bfloat16)
    ids, positions = torch.tensor([3, 5]), torch.tensor([0, 1])
    handle = None
    with torch.no_grad():
        with pytest.raises(AssertionError, match="fused gather"):
            model._embed(ids, positions)
        if what == "embed":
            model.embed_tokens = _Wrapper(model.embed_tokens)
        elif what == "rope":
            old = model.rotary_emb
            model.rotary_emb = nn.Module()
            model.rotary_emb.forward = lambda p, dtype: old.forward(p, dtype)
        elif what == "max_norm":
            model.embed_tokens.max_norm = 1.0
        else:
            handle = nn.modules.module.register_module_forward_pre_hook(lambda m, a: None)
        try:
            hidden, rope = model._embed(ids, positions)
        finally:
            if handle is not None:
                handle.remove()
        assert hidden.shape == (2, 64) and rope[0].shape == (2, 1, 16)
