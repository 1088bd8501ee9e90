"""SplitKLinear host logic on the CPU: the slice choice and the F.linear
fallback for inputs split-K cannot view (CPU tensors, strided rows), and the row limits of the few-rows kernel."""
import pytest
import torch

from tinyvllm import layers
from tinyvllm.layers import PackedLinear, SplitKLinear


def test_splits_for_table():
    cases = {  # (in, out): slices at rows 1, 128, 129, 512, 513
        (3072, 1024): (8, 8, 2, 2, 1),
        (4096, 4096): (4, 4, 4, 4, 1),
        (12288, 4096): (4, 4, 8, 8, 1),
        (25600, 5120): (4, 4, 8, 8, 1),
        (100, 4096): (1, 1, 1, 1, 1),  # reduction not divisible into slices
    }
    for (k, n), expect in cases.items():
        lin = SplitKLinear(k, n, device="meta")
        assert tuple(lin.splits_for(r) for r in (1, 128, 129, 512, 513)) == expect, (k, n)


def test_cpu_and_strided_inputs_take_linear():
    torch.manual_seed(0)
    lin = SplitKLinear(256, 64)
    x = torch.randn(8, 512)[:, ::2]
    y = lin(x)
    assert isinstance(y, torch.Tensor)
    torch.testing.assert_close(y, torch.nn.functional.linear(x, lin.weight))
    y2 = lin(x.contiguous())
    torch.testing.assert_close(y2, torch.nn.functional.linear(x.contiguous(), lin.weight))


# (columns, width): most rows of the few-rows kernel, at model widths and at the
# edges of the measured rules.
ROUNDED = {(4096, 1024): 64, (8192, 1024): 32, (4096, 2048): 32, (2048, 2048): 64,
           (1024, 2048): 32, (6144, 1280): 16, (2048, 4096): 24, (256, 4096): 16,
           (1536, 5120): 8, (1024, 6144): 0, (64, 65536): 0, (512, 8192): 0, (6144, 4096): 0,
           (16384, 256): 32, (32768, 256): 16, (131072, 32): 0, (96, 4096): 0}
GATED = {(6144, 1024): 64, (12288, 2048): 16, (19456, 2560): 16, (16384, 2560): 0,
         (24576, 4096): 16, (24576, 3584): 0, (51200, 5120): 0, (256, 4096): 0, (512, 16384): 0,
         (4096, 2048): 64, (1024, 2048): 32, (512, 2048): 16, (16384, 1280): 8, (65536, 64): 0}
PARTIALS = {(1024, 2048): 64, (1024, 3072): 64, (2048, 6144): 0, (2048, 4096): 32,
            (2048, 1024): 32, (1024, 4096): 64, (512, 8192): 24, (256, 53248): 16,
            (128, 32768): 0, (2560, 4096): 32, (2560, 9728): 32, (5120, 8192): 32,
            (5120, 25600): 24, (4096, 4096): 0, (7168, 9728): 0, (7168, 4096): 32,
            (3584, 17408): 0, (2048, 256): 16, (2560, 32768): 0}


@pytest.mark.parametrize("limit,table", [(layers._rounded_limit, ROUNDED),
                                         (layers._gated_limit, GATED),
                                         (layers._partials_limit, PARTIALS)])
def test_few_rows_limits(limit, table):
    assert {shape: limit(*shape) for shape in table} == table


def test_few_rows_rule_follows_the_limits(monkeypatch):
    """The modules ask their own limit, at it and one row past it."""
    asked = []
    monkeypatch.setattr(layers.few_rows, "fits", lambda x, w: True)
    monkeypatch.setattr(layers.few_rows, "few_rows_linear",
                        lambda x, w, **kw: asked.append((x.shape[0], kw)) or kw)
    for rows, takes in ((24, True), (25, False)):
        packed = PackedLinear(4096, (1024, 1024), device="meta")
        assert packed.takes_few_rows(torch.empty(rows, 4096, device="meta")) is takes
    for rows, takes in ((16, True), (17, False)):
        packed = PackedLinear(2560, (9728, 9728), device="meta")
        got = packed.gated(torch.empty(rows, 2560, device="meta"))
        assert got == ({"silu": True} if takes else None)
    for rows, takes in ((24, True), (25, False)):
        split = SplitKLinear(25600, 5120, device="meta")
        assert split.takes_few_rows(torch.empty(rows, 25600, device="meta")) is takes
    assert asked == [(16, {"silu": True})]
    assert PackedLinear(64, (48, 24, 24), device="meta").gated(
        torch.empty(1, 64, device="meta")) is None  # no gate and up
