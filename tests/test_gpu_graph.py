"""The batched codec calls under HIP graph capture.

The library's entry points only launch kernels with by-value arguments on the
caller's stream (no allocation, no memset, no host synchronisation), so a layer's
encode and decode can be captured once and replayed. Each replay here follows
eager work that changes the KV layer, and is checked byte for byte against the
oracle's payloads for the new contents and against the exact round trip.
"""

import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sz():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")
    from unchainkv_amd import splitzip_cuda

    assert splitzip_cuda.available(), splitzip_cuda.load_error()
    return splitzip_cuda


def say(*parts):
    print("[case]", *parts, flush=True)


def layer_words(rng, books, n, escape_rate):
    half = n // 2
    exps = np.empty(n, np.uint16)
    exps[:half] = np.frombuffer(books[:16], np.uint8)[rng.integers(0, 16, half)]
    exps[half:] = np.frombuffer(books[16:], np.uint8)[rng.integers(0, 16, n - half)]
    outside = np.array(sorted(set(range(256)) - set(books)), np.uint16)
    esc = rng.random(n) < escape_rate
    exps[esc] = outside[rng.integers(0, outside.size, int(esc.sum()))]
    return ((rng.integers(0, 2, n).astype(np.uint16) << 15) | (exps << 7)
            | rng.integers(0, 128, n).astype(np.uint16))


def test_paged_encode_decode_replay(sz, codebooks):
    books = codebooks[6 * 32:7 * 32]
    tab = oracle.top16_tables(books)
    bw, pool = 2048, 96
    rng = np.random.default_rng(4)
    perm = rng.permutation(pool).tolist()
    tables = [perm[0:9], perm[9:30], perm[30:34]]
    recv_tables = [perm[40:49], perm[49:70], perm[70:74]]
    batch = sz.PagedBatch(tables, bw, "cuda")
    recv = sz.PagedBatch(recv_tables, bw, "cuda")
    device_tables = sz.top16_tables_for(books, torch.device("cuda"), torch)
    kv = torch.zeros((2, pool, bw), dtype=torch.bfloat16, device="cuda")
    out = batch.new_payload_buffer()
    ws = batch.new_workspace()
    target = torch.zeros_like(kv)

    def step():
        assert sz.encode_top16_paged(kv, batch, out, ws, tables=device_tables)
        assert sz.decode_top16_paged(out, batch.out_offsets, batch.encoded_bytes, target, recv,
                                     tables=device_tables)

    step()  # warm-up outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    torch.cuda.synchronize()
    for replay in range(3):
        say("graph replay", replay)
        words = layer_words(rng, books, 2 * pool * bw, 0.002 * replay)
        # eager work between replays: new layer contents, receiver cleared
        kv.copy_(torch.from_numpy(words.view(np.int16)).cuda().view(torch.bfloat16).view(2, pool, bw))
        target.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        host = out.cpu().numpy()
        kv_host = words.reshape(2, pool, bw)
        got = target.view(torch.int16).cpu().numpy().view(np.uint16).reshape(2, pool, bw)
        for r, t in enumerate(tables):
            ref = oracle.top16_encode(kv_host[:, t].reshape(-1), tab)
            a = batch.out_offsets[r]
            assert bytes(host[a:a + batch.encoded_bytes[r]]) == bytes(ref), (replay, r)
            assert np.array_equal(got[:, recv_tables[r]], kv_host[:, t]), (replay, r)


@pytest.mark.parametrize("bw", [640, 1024])
def test_every_codec_replays(sz, bw):
    """Top-16, fixed6 and the torch-op formats of 70 requests (more than one launch of the
    small argument struct) in both geometries: each replay's payloads and restored layer
    are those of eager calls on the same contents."""
    books = bytes(range(0x78, 0x88)) * 2
    rng = np.random.default_rng(bw)
    requests, pool = 70, 150
    ids = rng.permutation(pool).tolist()
    batch = sz.PagedBatch([ids[2 * r:2 * r + 2] for r in range(requests)], bw, "cuda")
    recv = sz.PagedBatch([ids[::-1][2 * r:2 * r + 2] for r in range(requests)], bw, "cuda")
    device_tables = sz.top16_tables_for(books, torch.device("cuda"), torch)
    kv = torch.zeros((2, pool, bw), dtype=torch.bfloat16, device="cuda")
    # 8 high bytes (16 exponents, the codebook's) that every request holds, so that the
    # torch-op plans stay the same
    high = np.tile(np.arange(0x3C, 0x44, dtype=np.uint16), 2 * pool * bw // 8)

    def fill():
        words = (high << 8) | rng.integers(0, 256, high.size).astype(np.uint16)
        kv.copy_(torch.from_numpy(words.view(np.int16)).cuda().view(torch.bfloat16)
                 .view(2, pool, bw))

    fill()
    fields = sz.read_torchop_plans(sz.plan_torchop_paged(kv, batch).cpu().numpy())
    sizes = [size for _, size in fields]
    assert min(sizes) > 0
    starts = np.cumsum([0] + sizes)[:-1].tolist()
    six_offsets, six_sizes, _ = batch.palette_layout(6)

    class Buffers:
        def __init__(self):
            self.out, self.six = batch.new_payload_buffer().zero_(), batch.new_palette_buffer(6).zero_()
            self.torchop = torch.zeros(sum(sizes), dtype=torch.uint8, device="cuda")
            self.plans = torch.zeros(64 * requests, dtype=torch.uint8, device="cuda")
            self.layers = [torch.zeros_like(kv) for _ in range(3)]

        def all(self):
            return [self.out, self.six, self.torchop, self.plans] + \
                [layer.view(torch.int16) for layer in self.layers]

    workspace, six_workspace = batch.new_workspace(), batch.new_palette_workspace()

    def step(b):
        assert sz.encode_top16_paged(kv, batch, b.out, workspace, tables=device_tables)
        assert sz.decode_top16_paged(b.out, batch.out_offsets, batch.encoded_bytes, b.layers[0],
                                     recv, tables=device_tables)
        assert sz.encode_bf16_paged(kv, batch, b.six, six_workspace, 6)
        assert sz.decode_bf16_paged(b.six, six_offsets, six_sizes, b.layers[1], recv, 6)
        assert sz.plan_torchop_paged(kv, batch, b.plans) is not None
        assert sz.encode_torchop_paged(kv, batch, b.plans, b.torchop, starts, sizes)
        assert sz.decode_torchop_paged(b.torchop, starts, sizes, b.layers[2], recv)

    captured, eager = Buffers(), Buffers()
    step(captured)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(captured)
    torch.cuda.synchronize()
    for replay in range(3):
        say("graph replay of every codec", bw, replay)
        fill()
        for t in captured.all():
            t.zero_()
        torch.cuda.synchronize()
        graph.replay()
        step(eager)
        torch.cuda.synchronize()
        for k, (got, want) in enumerate(zip(captured.all(), eager.all())):
            assert torch.equal(got, want), (replay, k)
        sent = kv.view(torch.int16)[:, batch.ids]
        for layer in captured.layers:
            assert torch.equal(layer.view(torch.int16)[:, recv.ids], sent), replay


@pytest.mark.parametrize("contexts", [[300] * 5, [1, 17, 900, 4000, 64, 2113] * 11])
def test_attention_replays(sz, codebooks, contexts):
    """Equal contexts, and mixed ones in two launches."""
    books = codebooks[:32]
    rng = np.random.default_rng(len(contexts))
    heads, bw = 2, 16 * 2 * 128
    counts = [-(-c // 16) for c in contexts]
    pool = sum(counts)
    ids = rng.permutation(pool).tolist()
    ends = np.cumsum([0] + counts)
    batch = sz.PagedBatch([ids[a:b] for a, b in zip(ends, ends[1:])], bw, "cuda")
    device_tables = sz.top16_tables_for(books, torch.device("cuda"), torch)
    kv = torch.zeros((2, pool, bw), dtype=torch.bfloat16, device="cuda")
    payloads, workspace = batch.new_payload_buffer(), batch.new_workspace()
    q = torch.zeros((len(contexts), 4 * heads, 128), dtype=torch.bfloat16, device="cuda")
    out = torch.zeros_like(q)
    partials = torch.empty(sz.decode_attention_workspace_bytes(len(contexts), heads, max(contexts)),
                           dtype=torch.uint8, device="cuda")

    def step(target):
        assert sz.decode_attention_top16(q, payloads, batch.out_offsets, contexts, heads,
                                         tables=device_tables, out=target,
                                         workspace=partials) is target

    def fill():
        words = layer_words(rng, books, 2 * pool * bw, 0.0)
        kv.copy_(torch.from_numpy(words.view(np.int16)).cuda().view(torch.bfloat16).view(2, pool, bw))
        q.copy_(torch.from_numpy(rng.standard_normal(tuple(q.shape)).astype(np.float32)))
        assert sz.encode_top16_paged(kv, batch, payloads, workspace, tables=device_tables)

    fill()
    step(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(out)
    torch.cuda.synchronize()
    for replay in range(3):
        say("graph replay of attention", len(contexts), replay)
        fill()
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = torch.zeros_like(out)
        step(want)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), replay
        assert torch.isfinite(out).all() and out.float().abs().amax() > 0
