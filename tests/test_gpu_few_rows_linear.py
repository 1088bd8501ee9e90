"""The few-rows linear kernel at the edges of its row tiles (16, 32, 64), with
reductions that leave a wave one, a few or no steps, strided input rows and
both half types: against the fp32 product, rounded once (half an ulp plus the
fp32 sums' own rounding), its fp32 slices, and the SiLU epilogue against
silu_and_mul over the rounded projection."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(rows, columns, width, dtype, device, pad):
    g = torch.Generator().manual_seed(rows * 7 + columns + width)
    x = torch.randn(rows, width + pad, generator=g).to(dtype).to(device)[:, pad:]
    w = (torch.randn(columns, width, generator=g) * width ** -0.5).to(dtype).to(device)
    return x, w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("columns,width", [(32, 32), (64, 96), (4096, 1024), (96, 2080)])
@pytest.mark.parametrize("rows,pad", [(1, 0), (15, 8), (16, 0), (17, 0), (32, 24), (33, 0),
                                      (64, 8)])
def test_few_rows_linear(device, rows, pad, columns, width, dtype):
    from tinyvllm.kernels.linear import few_rows_linear
    from tinyvllm.kernels.pointwise import silu_and_mul

    x, w = _inputs(rows, columns, width, dtype, device, pad)
    exact = x.double() @ w.double().T
    # fp32 sums of `width` products: relative 2^-23 per addition of magnitudes
    # up to sum |x w|.
    slack = (x.double().abs() @ w.double().abs().T) * width * 2.0 ** -23
    ulp = torch.finfo(dtype).eps
    y = few_rows_linear(x, w)
    assert y.dtype == dtype and y.shape == (rows, columns)
    # Rounding to nearest: half an ulp, itself at most eps times the value.
    tiny = 2.0 ** -24  # fp16 results below its normal range round to this grid
    assert bool(((y.double() - exact).abs() <= slack + ulp / 2 * (exact.abs() + slack) + tiny).all())
    for slices in (1, 3, 4, 8):
        parts = few_rows_linear(x, w, slices=slices)
        assert parts.shape == (slices, rows, columns) and parts.dtype == torch.float32
        assert bool(((parts.double().sum(0) - exact).abs() <= slack).all())
    if columns % 64 == 0:
        # The two sum over other slices, so a gate and an up value may round
        # apart by one ulp each: silu turns that into (1 + |gate|) ulp of its
        # value, |gate| < 5 here; two more roundings follow.
        torch.testing.assert_close(few_rows_linear(x, w, silu=True), silu_and_mul(y),
                                   rtol=9 * ulp, atol=4 * tiny)


def test_layers_take_the_kernel_only_outside_autograd(device):
    """With gradients enabled the projections stay torch ops, with the same
    values up to the order of the fp32 sums."""
    from tinyvllm.layers import PackedLinear, SplitKLinear

    x = torch.randn(5, 1024, device=device, dtype=torch.bfloat16)
    packed = PackedLinear(1024, (1024, 1024), device=device, dtype=torch.bfloat16)
    split = SplitKLinear(1024, 1024, device=device, dtype=torch.bfloat16)
    y = packed(x)
    assert y.requires_grad and not packed.takes_few_rows(x) and packed.gated(x) is None
    assert split(x).partials.requires_grad
    with torch.no_grad():
        assert packed.takes_few_rows(x) and packed.gated(x).shape == (5, 1024)
        assert not packed(x).requires_grad
        torch.testing.assert_close(packed(x), y.detach(), rtol=2 ** -7, atol=2 ** -9)
        assert not packed.takes_few_rows(x[:, ::2][:, :1024].expand(5, 512))
        assert split(x).partials.shape == (8, 5, 1024)


def test_tangents_and_transforms_pass_the_projections(device):
    """no_grad leaves forward-mode AD on, and vmap has no data pointers: both
    go through torch's ops, as the embedding's rows do."""
    import torch.autograd.forward_ad as fwad
    from tinyvllm.layers import PackedLinear, SplitKLinear
    from tinyvllm.models.qwen3 import Qwen3Config, Qwen3Model

    torch.manual_seed(0)
    x, t = (torch.randn(4, 1024, device=device, dtype=torch.bfloat16) for _ in range(2))
    packed = PackedLinear(1024, (512, 512), device=device, dtype=torch.bfloat16)
    split = SplitKLinear(1024, 1024, device=device, dtype=torch.bfloat16)
    with torch.no_grad():
        with fwad.dual_level():
            y = packed(fwad.make_dual(x, t))
            tangent = fwad.unpack_dual(y).tangent
        torch.testing.assert_close(tangent, torch.nn.functional.linear(t, packed.weight))
        stacked = torch.stack([x, t])
        y = torch.func.vmap(packed)(stacked)
        torch.testing.assert_close(y, torch.nn.functional.linear(stacked, packed.weight))
        assert isinstance(split(x).partials, torch.Tensor)
        config = Qwen3Config(
            vocab_size=64, hidden_size=64, intermediate_size=96, num_hidden_layers=1,
            max_position_embeddings=32, num_attention_heads=2, num_key_value_heads=1, head_dim=32,
            rms_norm_eps=1e-6, rope_theta=1e4, tie_word_embeddings=True)
        model = Qwen3Model(config, device=device, dtype=torch.bfloat16)
        ids, positions = torch.tensor([3, 5], device=device), torch.tensor([0, 1], device=device)
        weight = model.embed_tokens.weight
        del model.embed_tokens.weight
        with fwad.dual_level():
            model.embed_tokens.weight = fwad.make_dual(weight.detach(), torch.ones_like(weight))
            hidden, _ = model._embed(ids, positions)
            assert bool((fwad.unpack_dual(hidden).tangent == 1).all())
