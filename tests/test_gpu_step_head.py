"""The one-launch heads of a step against the ops they replace, bit for bit:
embedding and RoPE row gathers, and table updates with token resolution."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,width,half,dtype", [
    (1, 8, 8, torch.bfloat16), (3, 1024, 64, torch.bfloat16), (65, 4096, 64, torch.float16),
    (700, 1032, 128, torch.bfloat16)])
def test_embed_rope_copies_rows(device, tokens, width, half, dtype):
    from tinyvllm.kernels.pointwise import embed_rope

    g = torch.Generator().manual_seed(tokens)
    embed = torch.randn(517, width, generator=g).to(dtype).to(device)
    cos, sin = (torch.randn(300, half, generator=g).to(dtype).to(device) for _ in range(2))
    ids = torch.randint(0, 517, (tokens,), generator=g)
    positions = torch.randint(0, 300, (tokens,), generator=g)
    ids[-1], positions[-1] = 516, 299
    ids, positions = ids.to(device), positions.to(device)
    out, c, s = embed_rope(ids, positions, embed, cos, sin)
    assert torch.equal(out, embed[ids])
    assert torch.equal(c, cos[positions][:, None]) and torch.equal(s, sin[positions][:, None])


def test_embed_rope_outside_the_tables_is_nan(device):
    from tinyvllm.kernels.pointwise import embed_rope

    table = torch.ones(4, 16, dtype=torch.bfloat16, device=device)
    ids = torch.tensor([-1, 4, 0], device=device)
    positions = torch.tensor([0, 3, 1 << 40], device=device)
    out, c, s = embed_rope(ids, positions, table, table, table)
    assert out.isnan().all(1).tolist() == [True, True, False]
    assert c.isnan().all(-1).flatten().tolist() == [False, False, True]
    assert torch.equal(c.isnan(), s.isnan())


@pytest.mark.parametrize("rows,count", [(1, 0), (16, 16), (300, 70000)])
def test_begin_decode_equals_its_two_ops(device, rows, count):
    from tinyvllm.kernels.kv_store import apply_table_updates, begin_decode
    from tinyvllm.kernels.sampling import resolve_tokens

    g = torch.Generator().manual_seed(rows)
    size = max(1, count) + 5
    updates = torch.empty(1 + 2 * size, dtype=torch.long)
    updates[0] = count
    updates[1::2] = torch.randperm(size, generator=g) - 2  # two indices outside
    updates[2::2] = torch.randint(0, 1000, (size,), generator=g)
    src = torch.randint(-1, rows + 2, (rows,), generator=g)
    prev = torch.randint(0, 1000, (rows,), generator=g)
    updates, src, prev = updates.to(device), src.to(device), prev.to(device)
    results = []
    for fused in (False, True):
        table = torch.arange(size, device=device) + 5000
        tokens = torch.arange(rows, device=device) + 9000
        if fused:
            begin_decode(table, updates, tokens, src, prev)
        else:
            apply_table_updates(table, updates)
            resolve_tokens(tokens, src, prev)
        results.append((table.clone(), tokens.clone()))
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_unaligned_embedding_takes_the_modules(device):
    """A table that starts off a 16-byte boundary (a view into a larger
    buffer) gives its rows all the same."""
    from tinyvllm.models.qwen3 import Qwen3Config, Qwen3Model

    config = Qwen3Config(
        vocab_size=64, hidden_size=64, intermediate_size=96, num_hidden_layers=1,
        max_position_embeddings=32, num_attention_heads=2, num_key_value_heads=1, head_dim=32,
        rms_norm_eps=1e-6, rope_theta=1e4, tie_word_embeddings=True)
    model = Qwen3Model(config, device=device, dtype=torch.bfloat16)
    flat = torch.randn(1 + 64 * 64, device=device).to(torch.bfloat16)
    model.embed_tokens.weight = torch.nn.Parameter(flat[1:].view(64, 64))
    ids, positions = torch.tensor([3, 63], device=device), torch.tensor([0, 31], device=device)
    with torch.no_grad():
        hidden, (cos, _) = model._embed(ids, positions)
    assert torch.equal(hidden, flat[1:].view(64, 64)[ids])
    assert torch.equal(cos, model.rotary_emb.tables(torch.bfloat16)[0][positions][:, None])
