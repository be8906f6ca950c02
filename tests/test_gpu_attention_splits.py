"""Context splits of the fused attention: each sequence takes the splits its own
context needs. Batches of very different lengths (one token beside tens of
thousands, more splits than one combine pass merges, the split cap, two launches of
unequal batches), every head's rows against attention over the original words in
float64 on the GPU. Tolerance: 1e-2 of each output row's largest magnitude (bf16
output and bf16 softmax weights), as for the kernel's other tests."""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

HEAD_DIM = 128
TOL = 1e-2


@pytest.fixture(scope="module")
def sz():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")
    from unchainkv_amd import splitzip_cuda

    assert splitzip_cuda.available(), splitzip_cuda.load_error()
    return splitzip_cuda


def make_batch(sz, kv_heads, contexts, seed, edit=None):
    from unchainkv_amd import workloads

    shape = workloads.Shape(layers=1, kv_heads=kv_heads, head_dim=HEAD_DIM)
    blocks = [-(-c // 16) for c in contexts]
    kv = workloads.make_kv_layer(torch, shape, sum(blocks), seed=seed, layer=0, device="cuda",
                                 outlier_rate=0.001)
    tables = workloads.random_block_tables(torch, sum(blocks), blocks, seed=seed)
    if edit:
        edit(kv, tables)
    books = workloads.fit_codebook(torch, kv, tables)
    batch = sz.PagedBatch(tables, shape.block_words, "cuda")
    payloads = batch.new_payload_buffer()
    assert sz.encode_top16_paged(kv, batch, payloads, batch.new_workspace(), codebooks=books)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    q = torch.randn((len(contexts), 4 * kv_heads, HEAD_DIM), generator=g,
                    device="cuda").to(torch.bfloat16)
    return kv, tables, books, batch, payloads, q


def reference(kv, ids, tokens, q, kv_heads):
    index = torch.tensor(ids, dtype=torch.int64, device=kv.device)
    k, v = kv.index_select(1, index).reshape(2, -1, kv_heads, HEAD_DIM)[:, :tokens].double()
    rows = q.double().reshape(kv_heads, 4, HEAD_DIM)
    p = torch.softmax((rows[:, :, None, :] * k.permute(1, 0, 2)[:, None]).sum(-1)
                      / HEAD_DIM ** 0.5, dim=-1)
    return (p[..., None] * v.permute(1, 0, 2)[:, None]).sum(2).reshape(4 * kv_heads, HEAD_DIM)


@pytest.mark.parametrize("kv_heads,contexts", [
    (1, [1, 15, 16, 17, 33, 20000]),             # one token beside the longest
    (1, [40000]),                                # a single sequence: the split cap
    (2, [2113]),                                 # more splits than one combine pass
    (3, [700, 5000, 64]),                        # odd head count
    (8, [1500]),                                 # a single user's decode step
    (5, [17 + 61 * i for i in range(40)]),       # more workgroups than one round
    (1, [1 + (i * 977) % 3000 for i in range(67)]),  # two launches, 64 and 3 sequences
])
def test_splits_follow_each_context(sz, kv_heads, contexts):
    print("[case] attention splits", kv_heads, contexts[:8], flush=True)
    kv, tables, books, batch, payloads, q = make_batch(sz, kv_heads, contexts, 7)
    out = sz.decode_attention_top16(q, payloads, batch.out_offsets, contexts, kv_heads,
                                    codebooks=books)
    torch.cuda.synchronize()
    assert out is not None
    got = out.double()
    for b, (ids, tokens) in enumerate(zip(tables, contexts)):
        ref = reference(kv, ids, tokens, q[b], kv_heads)
        err = (got[b] - ref).abs().amax(dim=-1)
        scale = ref.abs().amax(dim=-1).clamp_min(1e-6)
        assert (err <= TOL * scale).all(), (b, tokens, float((err / scale).max()))


def test_workspace_of_the_largest_batch_serves_smaller_ones(sz):
    """The workspace size grows with the batch and with the longest context, so one
    workspace can be kept while a batch shrinks and its contexts grow."""
    sizes = [[sz.decode_attention_workspace_bytes(b, heads, ctx) for ctx in
              (1, 17, 500, 1500, 8192, 8193, 40000)] for heads in (1, 8) for b in (1, 3, 32, 64, 90)]
    for row in sizes:
        assert row == sorted(row)
    for heads_rows in (sizes[:5], sizes[5:]):
        for column in zip(*heads_rows):
            assert list(column) == sorted(column)


@pytest.mark.parametrize("kv_heads,context", [(8, 1500), (1, 4000), (3, 700)])
@pytest.mark.parametrize("first,count", [(0, 16), (0, 128), (192, 64), (256, 128)])
@pytest.mark.parametrize("value", [float("nan"), float("-inf")])
def test_keys_that_are_not_finite(sz, kv_heads, context, first, count, value):
    """A NaN in the keys of a head makes its rows NaN, also where the NaN tokens fill whole
    ranges and splits; tokens whose scores are all -inf have no weight. Other heads keep
    their results."""
    print("[case] attention not finite", kv_heads, context, first, count, value, flush=True)
    head = kv_heads // 2

    def edit(kv, tables):
        for t in range(first, first + count):
            kv[0, tables[0][t // 16], t % 16, head, 5] = value

    kv, tables, books, batch, payloads, q = make_batch(sz, kv_heads, [context], 11, edit)
    q[:, :, 5] = q[:, :, 5].abs() + 0.5
    assert int(payloads[batch.out_offsets[0]]) == 5
    out = sz.decode_attention_top16(q, payloads, batch.out_offsets, [context], kv_heads,
                                    codebooks=books)
    got = out[0].double()
    ref = reference(kv, tables[0], context, q[0], kv_heads)
    rows = range(4 * head, 4 * head + 4)
    if value != value:
        assert torch.isnan(ref[rows]).all() and torch.isnan(got[rows]).all()
        keep = [r for r in range(4 * kv_heads) if r not in rows]
        got, ref = got[keep], ref[keep]
    if len(got):
        err, scale = (got - ref).abs().amax(dim=-1), ref.abs().amax(dim=-1).clamp_min(1e-6)
        assert (err <= TOL * scale).all(), float((err / scale).max())


def test_repeated_calls_give_the_same_bits(sz):
    """Whatever the workspace and the output held before."""
    contexts = [1, 300, 2113, 9000]
    kv, tables, books, batch, payloads, q = make_batch(sz, 2, contexts, 3)
    need = sz.decode_attention_workspace_bytes(len(contexts), 2, max(contexts))
    bits = []
    for fill in (0, 255, 0x7F):
        workspace = torch.full((need,), fill, dtype=torch.uint8, device="cuda")
        out = torch.full_like(q, float("nan"))
        assert sz.decode_attention_top16(q, payloads, batch.out_offsets, contexts, 2,
                                         codebooks=books, out=out, workspace=workspace) is out
        bits.append(out.view(torch.int16).clone())
    assert torch.equal(bits[0], bits[1]) and torch.equal(bits[0], bits[2])


@pytest.mark.parametrize("kv_heads,contexts,least,most", [
    (8, [256] * 32, 128, 256),       # 2 to 4 workgroups per CU: 16 us; one per CU: 18 us
    (8, [8192] * 32, 256, 256),      # 4 per CU: 144 us; 3: 150 us, 2: 164 us
    (1, [16384], 64, 128),           # 2 to 4 steps per range: 14 to 15 us; 1: 16.7 us
    (8, [32768], 96, 192),           # 2 or 3 per CU: 34 us; 1: 39 us, 4: 41 us
])
def test_number_of_splits(sz, kv_heads, contexts, least, most):
    """The splits a launch takes (partials written to the workspace), within those that
    measured best."""
    tokens = sum(contexts)
    kv, tables, books, batch, payloads, q = make_batch(sz, kv_heads, contexts, 5)
    need = sz.decode_attention_workspace_bytes(len(contexts), kv_heads, max(contexts))
    workspace = torch.full((need,), 0x7E, dtype=torch.uint8, device="cuda")
    assert sz.decode_attention_top16(q, payloads, batch.out_offsets, contexts, kv_heads,
                                     codebooks=books, workspace=workspace) is not None
    # a partial starts with its running max, never the filler
    maxima = workspace.view(torch.int32)[::4 * (HEAD_DIM + 2)]
    written = int((maxima != 0x7E7E7E7E).sum())
    print("[case] attention splits", kv_heads, tokens, written / kv_heads, flush=True)
    assert written % kv_heads == 0 and least <= written // kv_heads <= most


def test_rejected_payloads_with_more_splits_than_one_merge_pass(sz):
    """An overflowed payload and an escape list out of order make all rows of their own
    sequences NaN, also where four thread groups merge a sequence's splits."""
    heads, contexts = 2, [9000, 9000, 9000]
    kv, tables, books, batch, payloads, q = make_batch(sz, heads, contexts, 17)
    payloads[batch.out_offsets[0]] = 255
    at, n = batch.out_offsets[2], batch.count_words[2]
    count = int.from_bytes(bytes(payloads[at + 1:at + 5].cpu().numpy()), "little")
    assert count > 100
    last = at + 5 + n + n // 2 + 5 * (count - 2)  # the last two entries swapped
    pair = payloads[last:last + 10].clone()
    payloads[last:last + 5], payloads[last + 5:last + 10] = pair[5:], pair[:5]
    need = sz.decode_attention_workspace_bytes(len(contexts), heads, max(contexts))
    workspace = torch.full((need,), 0x7E, dtype=torch.uint8, device="cuda")
    out = sz.decode_attention_top16(q, payloads, batch.out_offsets, contexts, heads,
                                    codebooks=books, workspace=workspace)
    written = int((workspace.view(torch.int32)[::4 * (HEAD_DIM + 2)] != 0x7E7E7E7E).sum())
    assert written > 16 * heads * len(contexts)  # splits of a sequence: more than one pass
    assert torch.isnan(out[0]).all() and torch.isnan(out[2]).all()
    ref = reference(kv, tables[1], contexts[1], q[1], heads)
    err, scale = (out[1].double() - ref).abs().amax(dim=-1), ref.abs().amax(dim=-1)
    assert (err <= TOL * scale).all()
