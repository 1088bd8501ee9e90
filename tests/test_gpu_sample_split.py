"""The sampler's split path (rows spread over spans) draws the same tokens as
the one-workgroup path, which the oracle tests pin: every filter at the edges
of the spans (8192 tokens), of the bins (scores 32 below the maximum) and of
the gathered list (4096 tokens of one bin), and rows without a finite maximum."""
import pytest
import torch

pytestmark = pytest.mark.gpu

PARAMS = [(t, k, p) for t in (0.0, 0.05, 0.7, 1.0, 30.0, float("inf"))
          for k in (0, 1, 3, 40, 4096, 4097, 5000)
          for p in (1.0, 0.9, 0.5, 1e-6)]


def _draw(logits, temp, k, p, seeds, counters, *, split):
    from tinyvllm.kernels._extension import check, dtype_code, load_kernels, stream_of

    lib = load_kernels()
    rows, vocab = logits.shape
    size = lib.tvllm_sample_split_workspace_size(rows, vocab) if split else 0
    work = torch.empty(max(size, 1), dtype=torch.uint8, device=logits.device)
    work.fill_(255)  # nothing may rely on a cleared workspace
    out = torch.full((rows,), -7, dtype=torch.long, device=logits.device)
    check(lib.tvllm_sample(
        logits.data_ptr(), rows, vocab, logits.stride(0), temp.data_ptr(), k.data_ptr(),
        p.data_ptr(), seeds.data_ptr(), counters.data_ptr(), out.data_ptr(),
        work.data_ptr() if size else None, size, dtype_code(logits.dtype),
        stream_of(logits.device)))
    return out.cpu()


def _logits(kind, rows, vocab, g):
    x = torch.randn(rows, vocab, generator=g) * 2
    if kind == "flat":  # thousands of tokens in one bin
        x = x * 0.02
    elif kind == "tied":
        x = torch.full((rows, vocab), 1.5)
    elif kind == "masked":  # mostly excluded tokens, scores far below the bins
        x = torch.where(torch.rand(rows, vocab, generator=g) < 0.99, -float("inf"), x)
        x[:, vocab // 2] = 100.0
    elif kind == "special":
        for r in range(rows):
            x[r, r * 31 % vocab] = (float("nan"), float("inf"), -float("inf"))[r % 3]
    return x


@pytest.mark.parametrize("kind", ["normal", "flat", "tied", "masked", "special"])
@pytest.mark.parametrize("vocab,dtype", [
    (1, torch.bfloat16), (9, torch.float32), (8191, torch.bfloat16), (8192, torch.float16),
    (8195, torch.bfloat16), (20000, torch.float32), (40003, torch.bfloat16)])
def test_split_draws_equal_one_workgroup_draws(device, vocab, dtype, kind):
    g = torch.Generator().manual_seed(vocab + len(kind))
    rows = len(PARAMS)
    x = _logits(kind, rows, vocab, g).to(dtype)
    strides = (vocab, -(-vocab // 8) * 8)  # unaligned and vector-aligned rows
    temp, k, p = (torch.tensor(c, dtype=d).to(device) for c, d in
                  zip(zip(*PARAMS), (torch.float32, torch.long, torch.float32)))
    seeds = torch.arange(rows).to(device) * 104729 + vocab
    for stride in strides:
        wide = torch.zeros(rows, stride, dtype=dtype)
        wide[:, :vocab] = x
        logits = wide.to(device)[:, :vocab]
        for step in (0, 1):
            counters = torch.full((rows,), step, dtype=torch.long, device=device)
            whole = _draw(logits, temp, k, p, seeds, counters, split=False)
            split = _draw(logits, temp, k, p, seeds, counters, split=True)
            bad = [(PARAMS[i], int(whole[i]), int(split[i])) for i in range(rows)
                   if whole[i] != split[i]]
            assert not bad, (stride, step, bad[:5])
