"""The matrix-core kernels of head dims 32, 64 and 256 (and 128 for groups
above 16): decode and prefill at the edges of their row tiles (16 rows, 64 and
128 rows), key chunks (32 and 64 keys) and key splits, against the oracle; an
infinity in V; and queries and outputs without vector alignment."""
import math

import pytest
import torch

from helpers import assert_bf16_close
from oracle import attention as OA
from test_gpu_fp8 import _fp8_cache
from test_gpu_kernels import _Cache

pytestmark = pytest.mark.gpu


def _pool(g, contexts, bs=16):
    pages = [math.ceil(n / bs) for n in contexts]
    perm = torch.randperm(sum(pages) + 3, generator=g)
    offsets = torch.tensor([0] + pages).cumsum(0)
    return sum(pages) + 3, perm[:sum(pages)], offsets


def _setup(g, contexts, kv_heads, dim, dtype, fp8, device, layout):
    pool, blocks, offsets = _pool(g, contexts)
    k = torch.randn(pool * 16, kv_heads, dim, generator=g)
    v = torch.randn(pool * 16, kv_heads, dim, generator=g)
    if fp8:
        return (*_fp8_cache(k * 0.5, v * 2, 16, device, 0.5, 2.0, layout), blocks, offsets)
    k, v = k.to(dtype), v.to(dtype)
    return _Cache(k.to(device), v.to(device), 16, layout=layout), k, v, blocks, offsets


def _prefill(device, q, cache, k, v, blocks, offsets, queries, contexts, dim, pad=0):
    from tinyvllm.kernels.paged_prefill import paged_prefill_attention
    from tinyvllm.runtime.contracts import MultiQueryMetadata

    starts = torch.tensor([0] + queries).cumsum(0)
    lengths = torch.tensor(contexts)
    meta = MultiQueryMetadata(starts.to(device), blocks.to(device), offsets.to(device),
                              lengths.to(device), max(queries))
    wide = torch.zeros(*q.shape[:2], dim + pad, dtype=q.dtype, device=device)
    qd = wide[..., pad:]
    qd.copy_(q)
    out = torch.zeros_like(wide)[..., pad:]
    paged_prefill_attention(qd, cache, 0, meta, out, scale=dim ** -0.5)
    expect = torch.zeros(q.shape, dtype=q.dtype)
    OA.prefill_attention(q, k, v, starts, blocks, offsets, lengths, 16, dim ** -0.5, expect)
    return out.cpu(), expect


@pytest.mark.parametrize("dim,dtype,fp8", [(32, torch.bfloat16, False), (64, torch.float16, False),
                                           (64, torch.bfloat16, True), (256, torch.bfloat16, False),
                                           (256, torch.float16, True)])
@pytest.mark.parametrize("kv_heads,group,items", [
    (2, 4, [(5, 5), (8, 40), (9, 9), (1, 64)]),               # up to 36 rows: both kernels' side
    (1, 2, [(8, 31), (16, 33)]),                              # 32 rows at most: 16-row groups
    (1, 1, [(64, 64), (65, 97), (63, 127), (129, 400)]),      # 64-row tiles
    (8, 8, [(77, 200)] * 5 + [(2, 65), (40, 40)]),            # 128-row tiles (256+ workgroups)
])
def test_prefill_tiles_match_oracle(device, dim, dtype, fp8, kv_heads, group, items):
    g = torch.Generator().manual_seed(dim + group)
    if kv_heads == 8:
        items = items * 2
    queries, contexts = [list(x) for x in zip(*items)]
    cache, k, v, blocks, offsets = _setup(g, contexts, kv_heads, dim, dtype, fp8, device,
                                          "head_major" if group == 4 else "token_major")
    q = torch.randn(sum(queries), kv_heads * group, dim, generator=g).to(dtype)
    out, expect = _prefill(device, q, cache, k, v, blocks, offsets, queries, contexts, dim)
    assert_bf16_close(out, expect)


@pytest.mark.parametrize("dim,pad", [(64, 1), (256, 4), (32, 2)])
def test_unaligned_query_and_output_rows(device, dim, pad):
    g = torch.Generator().manual_seed(dim)
    queries, contexts = [50, 3], [90, 3]
    cache, k, v, blocks, offsets = _setup(g, contexts, 2, dim, torch.bfloat16, False, device,
                                          "token_major")
    q = torch.randn(53, 4, dim, generator=g).to(torch.bfloat16)
    out, expect = _prefill(device, q, cache, k, v, blocks, offsets, queries, contexts, dim, pad)
    assert_bf16_close(out, expect)


def test_longest_chunks_of_wide_groups(device):
    """65535 queries of 128 heads on one KV head: more row tiles than a grid
    dimension holds (the bound alone; the items themselves are short)."""
    from tinyvllm.kernels.paged_prefill import paged_prefill_attention
    from tinyvllm.runtime.contracts import MultiQueryMetadata

    g = torch.Generator().manual_seed(1)
    cache, k, v, blocks, offsets = _setup(g, [40, 3], 1, 256, torch.bfloat16, False, device,
                                          "token_major")
    q = torch.randn(7, 128, 256, generator=g).to(torch.bfloat16)
    starts, lengths = torch.tensor([0, 5, 7]), torch.tensor([40, 3])
    meta = MultiQueryMetadata(starts.to(device), blocks.to(device), offsets.to(device),
                              lengths.to(device), 65535)
    out = torch.zeros_like(q, device=device)
    paged_prefill_attention(q.to(device), cache, 0, meta, out, scale=256 ** -0.5)
    expect = torch.zeros_like(q)
    OA.prefill_attention(q, k, v, starts, blocks, offsets, lengths, 16, 256 ** -0.5, expect)
    assert_bf16_close(out, expect)


@pytest.mark.parametrize("dim", [32, 64, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fp8_rows_at_8_byte_boundaries(device, dim, dtype):
    """FP8 cache rows 8 bytes off every 16-byte boundary, decode and prefill."""
    from tinyvllm.kernels.paged_decode import paged_decode_attention
    from tinyvllm.runtime.contracts import SingleQueryMetadata

    g = torch.Generator().manual_seed(dim)
    contexts, kv_heads = [300, 17, 64], 2
    aligned, k, v, blocks, offsets = _setup(g, contexts, kv_heads, dim, dtype, True, device,
                                            "token_major")
    slots, row = aligned.num_slots, kv_heads * dim + 24

    def shifted(t):
        bytes_ = torch.zeros(slots * row + 8, dtype=torch.uint8, device=device)
        view = bytes_[8:].view(slots, row)[:, :kv_heads * dim].unflatten(1, (kv_heads, dim))
        view.copy_(t.view(torch.uint8))
        return view.view(torch.float8_e4m3fn)

    cache = _Cache(shifted(aligned.key[0]), shifted(aligned.value[0]), 16, 0.5, 2.0,
                   layout="token_major")
    assert cache.key[0].data_ptr() % 16 == 8 and cache.key[0].stride(0) % 16 == 8
    q = torch.randn(3, 4 * kv_heads, dim, generator=g).to(dtype)
    rows, lengths = torch.arange(3), torch.tensor(contexts)
    meta = SingleQueryMetadata(rows.to(device), blocks.to(device), offsets.to(device),
                               lengths.to(device), max(contexts))
    out = torch.zeros(q.shape, dtype=dtype, device=device)
    paged_decode_attention(q.to(device), cache, 0, meta, out, scale=dim ** -0.5)
    expect = torch.zeros(q.shape, dtype=dtype)
    OA.decode_attention(q, k, v, rows, blocks, offsets, lengths, 16, dim ** -0.5, expect)
    assert_bf16_close(out, expect)
    queries = [30, 17, 1]
    q = torch.randn(sum(queries), 4 * kv_heads, dim, generator=g).to(dtype)
    out, expect = _prefill(device, q, cache, k, v, blocks, offsets, queries, contexts, dim)
    assert_bf16_close(out, expect)


@pytest.mark.parametrize("dim,group,dtype", [
    (32, 2, torch.bfloat16), (64, 4, torch.bfloat16), (256, 3, torch.bfloat16),
    (128, 20, torch.bfloat16), (64, 4, torch.float16), (256, 3, torch.float16)])
@pytest.mark.parametrize("longest", [30, 5000])
def test_decode_with_an_infinite_value(device, dim, group, dtype, longest):
    """Rows whose V holds an infinity give that infinity (their weights there
    are positive); the other rows and dims are untouched by it."""
    from tinyvllm.kernels.paged_decode import paged_decode_attention
    from tinyvllm.runtime.contracts import SingleQueryMetadata

    g = torch.Generator().manual_seed(dim)
    contexts = [longest, 17, 64]
    cache, k, v, blocks, offsets = _setup(g, contexts, 2, dim, dtype, False, device,
                                          "token_major")
    slot = int(blocks[(contexts[0] - 1) // 16]) * 16 + (contexts[0] - 1) % 16
    for t in (v, cache.value[0]):
        t[slot, 1, 3] = float("inf")
    q = torch.randn(3, 2 * group, dim, generator=g).to(dtype)
    rows, lengths = torch.arange(3), torch.tensor(contexts)
    meta = SingleQueryMetadata(rows.to(device), blocks.to(device), offsets.to(device),
                               lengths.to(device), longest)
    out = torch.zeros(q.shape, dtype=q.dtype, device=device)
    paged_decode_attention(q.to(device), cache, 0, meta, out, scale=dim ** -0.5)
    expect = torch.zeros(q.shape, dtype=q.dtype)
    OA.decode_attention(q, k, v, rows, blocks, offsets, lengths, 16, dim ** -0.5, expect)
    out = out.cpu()
    assert bool((expect[0, group:, 3] == float("inf")).all())
    assert torch.equal(torch.isinf(out), torch.isinf(expect))
    finite = torch.isfinite(expect)
    assert_bf16_close(out[finite], expect[finite])


def _sink_case(g, lengths, kv_heads, heads, dim, dtype, fp8, gap, device):
    """Key 0 of every item scores ``gap`` octaves above the others and has
    V = 0, as an attention sink; the others' scores differ by up to one
    octave. Stored values, and the context's attention in 64 bits."""
    pool, blocks, offsets = _pool(g, lengths)
    k = torch.rand(pool * 16, kv_heads, dim, generator=g)
    k[..., 1:] *= 0.0
    v = 64 + 64 * torch.rand(pool * 16, kv_heads, dim, generator=g)
    a = 4.0  # q = a in dim 0: scores a * k[..., 0], in octaves with this scale
    scale = math.log(2) / a
    for i in range(len(lengths)):
        slot = int(blocks[offsets[i]]) * 16
        k[slot, :, 0], v[slot] = float(gap), 0.0
    if fp8:
        cache, k, v = _fp8_cache(k, v, 16, device, 0.25, 0.5, "head_major")
    else:
        k, v = k.to(dtype), v.to(dtype)
        cache = _Cache(k.to(device), v.to(device), 16, layout="head_major")
    return cache, k.double(), v.double(), blocks, offsets, a, scale


def _sink_bound(dtype, gap):
    # The result's own rounding; a weight's rounding, at most 2^-36 of the
    # largest in fp16 and 2^-17 of itself in bf16; exponentials and fp32 sums.
    own = torch.finfo(dtype).eps / 2
    return own + (2.0 ** (gap - 36) if dtype == torch.float16 else 2.0 ** -17) + 2.0 ** -15


@pytest.mark.parametrize("gap", [12, 20, 24])
@pytest.mark.parametrize("dim,group,dtype,fp8", [
    (64, 4, torch.float16, False), (256, 2, torch.float16, False), (32, 1, torch.float16, True),
    (256, 2, torch.float16, True), (128, 20, torch.float16, False), (64, 4, torch.bfloat16, False)])
def test_small_weights_beside_a_sink(device, dim, group, dtype, fp8, gap):
    """Weights far below the row's largest count in full where that one's V is
    zero: decode (split and unsplit rows) and prefill tiles."""
    from tinyvllm.kernels.paged_decode import paged_decode_attention
    from tinyvllm.kernels.paged_prefill import paged_prefill_attention
    from tinyvllm.runtime.contracts import MultiQueryMetadata, SingleQueryMetadata

    g = torch.Generator().manual_seed(dim + gap)
    lengths, kv_heads = [3000, 90, 1], 2
    heads = kv_heads * group
    cache, k, v, blocks, offsets, a, scale = _sink_case(g, lengths, kv_heads, heads, dim, dtype,
                                                        fp8, gap, device)

    def exact(item, end):
        slots = blocks[offsets[item]:offsets[item + 1]].repeat_interleave(16) * 16 \
            + torch.arange(16).repeat(int(offsets[item + 1] - offsets[item]))
        slots = slots[:end]
        w = torch.softmax(k[slots, :, 0] * a * scale, 0)  # [keys, kv_heads]
        return torch.einsum("kh,khd->hd", w, v[slots]).repeat_interleave(group, 0)

    q = torch.zeros(3, heads, dim, dtype=dtype)
    q[..., 0] = a
    rows = torch.arange(3)
    meta = SingleQueryMetadata(rows.to(device), blocks.to(device), offsets.to(device),
                               torch.tensor(lengths).to(device), max(lengths))
    out = torch.zeros_like(q, device=device)
    paged_decode_attention(q.to(device), cache, 0, meta, out, scale=scale)
    bound = _sink_bound(dtype, gap)
    for i in range(3):
        e = exact(i, lengths[i])
        assert bool(((out[i].cpu().double() - e).abs() <= bound * e).all()), (i, lengths[i])
    if dim == 128:
        return  # prefill at that head dim has a kernel of its own
    queries = [70, 90, 1]
    q = torch.zeros(sum(queries), heads, dim, dtype=dtype)
    q[..., 0] = a
    starts = torch.tensor([0] + queries).cumsum(0)
    meta = MultiQueryMetadata(starts.to(device), blocks.to(device), offsets.to(device),
                              torch.tensor(lengths).to(device), max(queries))
    out = torch.zeros_like(q, device=device)
    paged_prefill_attention(q.to(device), cache, 0, meta, out, scale=scale)
    for i in range(3):
        for j in (0, queries[i] // 2, queries[i] - 1):
            e = exact(i, lengths[i] - queries[i] + j + 1)
            got = out[int(starts[i]) + j].cpu().double()
            assert bool(((got - e).abs() <= bound * e).all()), (i, j)


def _with_specials(cache, specials, contexts, blocks, offsets, device, run):
    """Two runs over the same cache: V zero at the special elements (item, key,
    kv head, dim, value), then holding them; the plain run's output with what
    the specials make of it, and the special run's."""
    value = cache.value[0]

    def place(zero):
        for item, key, head, d, x in specials:
            slot = int(blocks[offsets[item] + key // 16]) * 16 + key % 16
            value[slot, head, d] = torch.tensor(0.0 if zero else x).to(value.dtype).to(device)

    place(True)
    plain = run()
    place(False)
    return plain, run()


def _expect(plain, specials, rows_seeing, group):
    """rows_seeing(item, key): the output rows whose queries see the key."""
    expect = plain.clone().float()
    for item, key, head, d, x in specials:
        for r in rows_seeing(item, key):
            expect[r, head * group:(head + 1) * group, d] += x
    return expect.to(plain.dtype)


def _assert_same(out, expect):
    assert torch.equal(out.isnan(), expect.isnan())
    finite_or_inf = ~expect.isnan()
    assert torch.equal(out[finite_or_inf], expect[finite_or_inf])


INF, NAN = float("inf"), float("nan")


@pytest.mark.parametrize("dtype,fp8", [(torch.bfloat16, False), (torch.float16, False),
                                       (torch.float16, True)])
@pytest.mark.parametrize("dim,kv_heads,group,items", [
    (64, 2, 2, [(8, 31), (5, 60)]),          # up to 16 rows: rows kernel, several queries each
    (256, 2, 1, [(30, 400), (3, 3)]),        # rows kernel
    (32, 1, 1, [(64, 64), (129, 400)]),      # 64-row tiles, two halves
    (64, 2, 3, [(65, 97), (70, 300)]),       # two halves
    (256, 2, 2, [(40, 40), (100, 333)]),     # two halves
    (64, 8, 1, [(100, 150)] * 18),           # 64-row tiles, one half
    (256, 8, 4, [(60, 130)] * 9),            # one half
    (32, 8, 8, [(77, 200)] * 7 + [(2, 65)]), # 128-row tiles
    (64, 8, 8, [(77, 200)] * 7 + [(40, 40)])])
def test_prefill_with_infinities_and_nans(device, dim, kv_heads, group, items, dtype, fp8):
    """Queries before a key whose V holds an infinity or a NaN keep their bits;
    later ones get it in its dim alone."""
    g = torch.Generator().manual_seed(dim + group)
    queries, contexts = [list(x) for x in zip(*items)]
    cache, k, v, blocks, offsets = _setup(g, contexts, kv_heads, dim, dtype, fp8, device,
                                          "token_major")
    q = torch.randn(sum(queries), kv_heads * group, dim, generator=g).to(dtype)
    starts = [0]
    for n in queries:
        starts.append(starts[-1] + n)

    def middle(item):  # a key that about half of the item's queries see
        return contexts[item] - 1 - queries[item] // 2

    specials = [(0, middle(0), 0, 3, NAN), (1, middle(1), kv_heads - 1, dim - 1, NAN)]
    if not fp8:
        specials = [(0, middle(0), 0, 3, INF), (0, middle(0), 0, 17, -INF),
                    (0, contexts[0] - 1, 0, 17, INF), (1, middle(1), kv_heads - 1, dim - 1, NAN),
                    (1, 0, 0, 0, -INF)]

    def run():
        return _prefill(device, q, cache, k, v, blocks, offsets, queries, contexts, dim)[0]

    def seeing(item, key):
        first = max(0, key - (contexts[item] - queries[item]))
        return range(starts[item] + first, starts[item + 1])

    plain, out = _with_specials(cache, specials, contexts, blocks, offsets, device, run)
    _assert_same(out, _expect(plain, specials, seeing, group))


@pytest.mark.parametrize("dim,group,dtype,fp8", [
    (32, 2, torch.bfloat16, True), (64, 4, torch.bfloat16, False), (64, 4, torch.float16, False),
    (256, 3, torch.float16, True), (256, 16, torch.bfloat16, False),
    (128, 20, torch.bfloat16, False)])
@pytest.mark.parametrize("contexts", [[30, 17], [5000, 300, 1], [700] * 40])
def test_decode_with_infinities_and_nans(device, dim, group, dtype, fp8, contexts):
    from tinyvllm.kernels.paged_decode import paged_decode_attention
    from tinyvllm.runtime.contracts import SingleQueryMetadata

    g = torch.Generator().manual_seed(dim)
    cache, _, _, blocks, offsets = _setup(g, contexts, 2, dim, dtype, fp8, device, "head_major")
    n = len(contexts)
    q = torch.randn(n, 2 * group, dim, generator=g).to(dtype).to(device)
    meta = SingleQueryMetadata(torch.arange(n).to(device), blocks.to(device), offsets.to(device),
                               torch.tensor(contexts).to(device), max(contexts))
    x = NAN if fp8 else -INF
    specials = [(0, contexts[0] - 1, 0, 3, x), (1, 0, 1, dim - 1, NAN),
                (1, contexts[1] // 2, 0, dim // 2, x)]

    def run():
        out = torch.zeros_like(q)
        paged_decode_attention(q, cache, 0, meta, out, scale=dim ** -0.5)
        return out.cpu()

    plain, out = _with_specials(cache, specials, contexts, blocks, offsets, device, run)
    _assert_same(out, _expect(plain, specials, lambda item, key: [item], group))


@pytest.mark.parametrize("dim", [32, 64, 256])
def test_a_cache_of_nans_gives_nans(device, dim):
    """V all NaN in one item's pages, decode and prefill; the others' rows stay."""
    g = torch.Generator().manual_seed(dim)
    queries, contexts = [70, 33], [300, 90]
    cache, k, v, blocks, offsets = _setup(g, contexts, 2, dim, torch.bfloat16, False, device,
                                          "token_major")
    q = torch.randn(sum(queries), 8, dim, generator=g).to(torch.bfloat16)
    args = (device, q, cache, k, v, blocks, offsets, queries, contexts, dim)
    plain = _prefill(*args)[0]
    for b in blocks[:offsets[1]].tolist():
        cache.value[0][16 * b:16 * b + 16] = NAN
    out = _prefill(*args)[0]
    assert bool(out[:70].isnan().all()) and torch.equal(out[70:], plain[70:])
