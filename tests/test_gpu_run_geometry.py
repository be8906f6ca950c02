"""Layers whose block words are a multiple of 8 but not of 1024 (the run geometry of the
tile kernels): every codec's payloads byte for byte with the oracle's and the decode
into other blocks word for word. Requests end on both sides of a 512-word run row, a
1024-word wave and a 4096-word tile; exponents are natural, escape-dense (a tile of each
plane past the staged escapes is scanned again) or overflow the Top-16 capacity. Blocks
of the layer outside the requests stay untouched."""

import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

BLOCK_WORDS = [8, 24, 520, 1016, 1032, 1280, 4104, 7680]
# blocks that end inside a 128-byte line, multiples of 16 words on both sides of the rule
# that decodes the short ones by 16-word lanes
SHORT_BLOCK_WORDS = [16, 48, 144, 160, 176, 272]


@pytest.fixture(scope="module")
def sz():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")
    from unchainkv_amd import splitzip_cuda

    assert splitzip_cuda.available(), splitzip_cuda.load_error()
    return splitzip_cuda


def make(bw, kind, seed):
    """(layer words, sender tables, receiver tables, codebook)."""
    rng = np.random.default_rng(seed)
    # 'dense': a longest request with room for more escapes than one tile stages
    counts = [max(3, t // bw) for t in (500, 1024, 4096, 4608, 64000 if kind == "dense" else 13000)]
    pool = sum(counts) + 4
    values = rng.standard_normal((2, pool, bw)).astype(np.float32)
    words = (values.view(np.uint32) >> 16).astype(np.uint16)

    def tables():
        ids, at, out = rng.permutation(pool).tolist(), 0, []
        for c in counts:
            out.append(ids[at:at + c])
            at += c
        return out

    send, recv = tables(), tables()
    if kind != "natural":
        hit = rng.random(words.shape) < (0.003 if kind == "dense" else 0.05)
        if kind == "dense":
            hit[:, send[-1]] = False
        words[hit] = (rng.integers(0x60, 0x7F, hit.sum()) << 8).astype(np.uint16)
    if kind == "dense":
        # one tile of each plane with more escapes than are staged, in two places of it
        request = words[:, send[-1]].reshape(2, -1)
        request[:, 4096 + 300:4096 + 400] = 0x7F00
        request[:, 4096 + 3900:4096 + 3980] = 0xFF00
        words[:, send[-1]] = request.reshape(2, -1, bw)
    book = b""
    for plane in range(2):
        count = np.bincount((words[plane].reshape(-1) >> 7) & 0xFF, minlength=256)
        count[0xC0:] = 0
        book += bytes(sorted(range(256), key=lambda e: (-count[e], e))[:16])
    return words, send, recv, book


def escapes_of_tiles(words, book):
    """Escapes of every 4096-word tile of a request (2, words of a plane)."""
    counts = []
    for plane in range(2):
        miss = ~np.isin((words[plane] >> 7) & 0xFF, np.frombuffer(book[16 * plane:16 * plane + 16],
                                                                  dtype=np.uint8))
        counts += [int(miss[at:at + 4096].sum()) for at in range(0, miss.size, 4096)]
    return counts


def to_gpu(words):
    return torch.from_numpy(words.view(np.int16).copy()).cuda().view(torch.bfloat16)


def check_restored(words, send, recv, target, payload_ok):
    got = target.view(torch.int16).cpu().numpy().view(np.uint16)
    for r, (t, u) in enumerate(zip(send, recv)):
        want = words[:, t] if payload_ok[r] else np.zeros_like(words[:, t])
        assert np.array_equal(got[:, u], want), r
    rest = sorted(set(range(words.shape[1])) - {b for u in recv for b in u})
    assert not got[:, rest].any()


@pytest.mark.parametrize("kind", ["natural", "dense", "overflow"])
@pytest.mark.parametrize("bw", BLOCK_WORDS + SHORT_BLOCK_WORDS)
def test_top16(sz, bw, kind):
    print("[case] runs top16", bw, kind, flush=True)
    words, send, recv, book = make(bw, kind, bw)
    layer = to_gpu(words)
    batch = sz.PagedBatch(send, bw, "cuda")
    assert batch.directory_bytes() == 0
    out = batch.new_payload_buffer().fill_(0x5A)
    assert sz.encode_top16_paged(layer, batch, out, batch.new_workspace(), codebooks=book) == \
        batch.total_encoded_bytes
    host = out.cpu().numpy()
    tab = oracle.top16_tables(book)
    ok = []
    for r, t in enumerate(send):
        a = batch.out_offsets[r]
        want = oracle.top16_encode(words[:, t].reshape(-1), tab)
        assert bytes(host[a:a + batch.encoded_bytes[r]]) == bytes(want), r
        ok.append(want[0] == 5)
    assert (host[:batch.out_offsets[0]] == 0x5A).all()
    if kind == "dense":
        # scanned again and placed: more escapes than a tile stages (128), no overflow
        assert max(escapes_of_tiles(words[:, send[-1]].reshape(2, -1), book)) > 128 and ok[-1]
    target = torch.zeros_like(layer)
    assert sz.decode_top16_paged(out, batch.out_offsets, batch.encoded_bytes, target,
                                 sz.PagedBatch(recv, bw, "cuda"), codebooks=book) == \
        batch.total_raw_bytes
    check_restored(words, send, recv, target, ok)
    # the drop-in pair over the longest request, a workspace's room past the payload
    words_r = np.ascontiguousarray(words[:, send[-1]])
    size = batch.encoded_bytes[-1]
    buf = torch.zeros(2 * words_r.size + (1 << 20), dtype=torch.uint8, device="cuda")
    assert sz.encode_top16(to_gpu(words_r), buf, 0, codebooks=book) == size
    want = oracle.top16_encode(words_r.reshape(-1), tab)
    assert bytes(buf[:size].cpu().numpy()) == bytes(want)
    target = torch.zeros_like(layer)
    assert sz.decode_top16(buf[:size], target, recv[-1], 2 * words_r.size, 0, codebooks=book)
    got = target.view(torch.int16).cpu().numpy().view(np.uint16)
    assert np.array_equal(got[:, recv[-1]], words_r if want[0] == 5 else np.zeros_like(words_r))


@pytest.mark.parametrize("blocks", [2, 256, 257])
@pytest.mark.parametrize("bw", [24, 48, 1032, 1280])
def test_dropin_block_table(sz, bw, blocks):
    """Shuffled tables of up to 256 ids ride in the kernel arguments, longer ones in a
    device copy: the drop-in decodes of both codecs restore the same words."""
    print("[case] runs drop-in table", bw, blocks, flush=True)
    rng = np.random.default_rng(bw + blocks)
    pool = blocks + 5
    values = rng.standard_normal((2, blocks, bw)).astype(np.float32)
    words = (values.view(np.uint32) >> 16).astype(np.uint16)
    ids = rng.permutation(pool)[:blocks].tolist()
    if blocks == 2:
        ids = [pool - 1, 0]
    book = b""
    for plane in range(2):
        count = np.bincount((words[plane].reshape(-1) >> 7) & 0xFF, minlength=256)
        book += bytes(sorted(range(256), key=lambda e: (-count[e], e))[:16])
    source = to_gpu(words)
    lib = sz._load()
    tab = sz.top16_tables_for(book, source.device, torch)
    buf = torch.zeros(4 * words.size + (1 << 20), dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for codec in ("top16", "fixed6"):
        size = sz.encode_top16(source, buf, 0, codebooks=book) if codec == "top16" else \
            sz.encode_bf16(source, buf)
        if not size:  # too short for fixed6 to be smaller
            assert codec == "fixed6" and words.size < 300
            continue
        target = torch.zeros((2, pool, bw), dtype=torch.bfloat16, device="cuda")
        payload = buf[:size]
        got = sz.decode_top16(payload, target, ids, 2 * words.size, 0, codebooks=book) \
            if codec == "top16" else sz.decode_fixed6(payload, target, ids, 2 * words.size)
        assert got == 2 * words.size
        restored = target.view(torch.int16).cpu().numpy().view(np.uint16)
        assert np.array_equal(restored[:, ids], words), codec
        rest = sorted(set(range(pool)) - set(ids))
        assert not restored[:, rest].any()
        # the entries' own rules: each takes its geometry and at most 256 blocks
        table = np.array(ids, dtype=np.int64)
        args = (payload.data_ptr(), size, target.data_ptr(), words.size, blocks, bw,
                target.stride(0), target.stride(1), table.ctypes.data) + \
            ((tab.data_ptr(),) if codec == "top16" else ()) + (stream,)
        tile = getattr(lib, f"kvq_splitzip_bf16_decode_{codec}_host_blocks")
        runs = getattr(lib, f"kvq_splitzip_bf16_decode_{codec}_host_runs")
        assert tile(*args) == 0
        assert runs(*args) == (2 * words.size if blocks <= 256 else 0)
    torch.cuda.synchronize()


@pytest.mark.parametrize("bits", [6, 5])
@pytest.mark.parametrize("bw", BLOCK_WORDS + SHORT_BLOCK_WORDS)
def test_palette(sz, bw, bits):
    print("[case] runs palette", bw, bits, flush=True)
    words, send, recv, _ = make(bw, "natural", bw + bits)
    # at most 31 high bytes, so that both palettes hold them; a request needs about
    # 300 words to be smaller than its raw bytes
    words = (((words >> 8) % 31 << 8) | (words & 0xFF)).astype(np.uint16)
    keep = [r for r, t in enumerate(send) if 2 * len(t) * bw >= 512]
    send, recv = [send[r] for r in keep], [recv[r] for r in keep]
    layer = to_gpu(words)
    batch = sz.PagedBatch(send, bw, "cuda")
    offsets, sizes, _ = batch.palette_layout(bits)
    out = batch.new_palette_buffer(bits).fill_(0x5A)
    assert sz.encode_bf16_paged(layer, batch, out, batch.new_palette_workspace(), bits) == \
        sum(sizes)
    host = out.cpu().numpy()
    for r, t in enumerate(send):
        want = oracle.palette_encode(words[:, t].reshape(-1), bits)
        assert bytes(host[offsets[r]:offsets[r] + sizes[r]]) == bytes(want), r
    target = torch.zeros_like(layer)
    assert sz.decode_bf16_paged(out, offsets, sizes, target, sz.PagedBatch(recv, bw, "cuda"),
                                bits) == batch.total_raw_bytes
    check_restored(words, send, recv, target, [True] * len(send))


@pytest.mark.parametrize("formats", ["signmag", "mixed"])
@pytest.mark.parametrize("bw", BLOCK_WORDS + SHORT_BLOCK_WORDS)
def test_torchop(sz, bw, formats):
    print("[case] runs torchop", bw, formats, flush=True)
    words, send, recv, _ = make(bw, "natural", bw + 1)
    if formats == "mixed":
        rng = np.random.default_rng(bw)
        # every third request's high bytes over the whole range (palette), another's
        # with few low nibbles (nibble planes)
        for r, t in enumerate(send):
            if r % 3 == 1:
                high = rng.choice(np.concatenate([[0, 0x7F], np.arange(0x80, 0x98)]),
                                  (2, len(t), bw))
                words[:, t] = ((high << 8) | (words[:, t] & 0xFF)).astype(np.uint16)
            elif r % 3 == 2:
                words[:, t] = (rng.integers(0, 256, (2, len(t), bw)) << 8 |
                               rng.integers(0, 2, (2, len(t), bw))).astype(np.uint16)
    layer = to_gpu(words)
    batch = sz.PagedBatch(send, bw, "cuda")
    plans = sz.plan_torchop_paged(layer, batch)
    fields = sz.read_torchop_plans(plans.cpu().numpy())
    sizes = [size for _, size in fields]
    offsets = (np.cumsum([0] + [s + 3 for s in sizes])[:-1] + 1).tolist()  # odd starts
    out = torch.full((sum(sizes) + 3 * len(sizes) + 8,), 0x5A, dtype=torch.uint8, device="cuda")
    assert sz.encode_torchop_paged(layer, batch, plans, out, offsets, sizes) == sum(sizes)
    host = out.cpu().numpy()
    keep = []
    for r, t in enumerate(send):
        want = oracle.encode_torchop(words[:, t].reshape(-1))
        if want is None:
            assert fields[r] == (255, 0), r
            continue
        keep.append(r)
        assert fields[r] == (int(want[0]), want.size), r
        end = offsets[r] + sizes[r]
        assert bytes(host[offsets[r]:end]) == want.tobytes(), r
        assert (host[end:end + 3] == 0x5A).all()
    assert keep
    target = torch.zeros_like(layer)
    assert sz.decode_torchop_paged(out, [offsets[r] for r in keep], [sizes[r] for r in keep],
                                   target, sz.PagedBatch([recv[r] for r in keep], bw, "cuda")) \
        == sum(batch.raw_bytes[r] for r in keep)
    check_restored(words, [send[r] for r in keep], [recv[r] for r in keep], target,
                   [True] * len(keep))


def time_of(call, n=20):
    """Median time of a call among n (us)."""
    times = []
    for _ in range(7):
        begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        begin.record()
        for _ in range(n):
            call()
        end.record()
        torch.cuda.synchronize()
        times.append(begin.elapsed_time(end) / n * 1e3)
    return sorted(times)[3]


@pytest.mark.parametrize("bw", [8, 16, 24, 48])
def test_short_blocks_decode_no_slower_than_they_encode(sz, bw):
    """64 MiB in 64 requests with shuffled tables, encode / decode: 90 / 93, 53 / 38, 47 / 48
    and 35 / 30 us. Written through, each part of a line shared between blocks by itself,
    the decode took 187, 102, 92 and 61 us. A quarter of room for noise."""
    blocks = (1 << 24) // bw
    per = blocks // 64
    g = torch.Generator(device="cuda")
    g.manual_seed(bw)
    layer = torch.randn((2, blocks, bw), generator=g, device="cuda").to(torch.bfloat16)

    def batch():
        ids = torch.randperm(blocks, generator=g, device="cuda").tolist()
        return sz.PagedBatch([ids[r * per:(r + 1) * per] for r in range(64)], bw, "cuda")

    send, recv = batch(), batch()
    tables = sz.top16_tables_for(bytes(range(114, 130)) * 2, layer.device, torch)
    out, workspace, target = send.new_payload_buffer(), send.new_workspace(), torch.zeros_like(layer)

    def encode():
        return sz.encode_top16_paged(layer, send, out, workspace, tables=tables)

    def decode():
        return sz.decode_top16_paged(out, send.out_offsets, send.encoded_bytes, target, recv,
                                     tables=tables)

    assert encode() == send.total_encoded_bytes and decode() == send.total_raw_bytes
    assert torch.equal(target[:, recv.ids].view(torch.int16), layer[:, send.ids].view(torch.int16))
    times = time_of(encode), time_of(decode)
    print("[case] runs short blocks", bw, "encode, decode (us)", times, flush=True)
    assert times[1] <= 1.25 * times[0], times


@pytest.mark.parametrize("bw", [24, 48, 640, 1024])
def test_code_table_off_four_byte_alignment(sz, bw):
    """Such a table takes the 16-word lanes (block words a multiple of 16) or the generic
    kernels."""
    print("[case] code table at byte offset 1", bw, flush=True)
    words, send, recv, book = make(bw, "natural", bw + 3)
    layer = to_gpu(words)
    batch = sz.PagedBatch(send, bw, "cuda")
    room = torch.zeros(545, dtype=torch.uint8, device="cuda")
    tables = room[1:]
    tables.copy_(sz.top16_tables_for(book, layer.device, torch))
    assert tables.data_ptr() % 4 == 1
    out = batch.new_payload_buffer().fill_(0x5A)
    assert sz.encode_top16_paged(layer, batch, out, batch.new_workspace(), tables=tables) == \
        batch.total_encoded_bytes
    host = out.cpu().numpy()
    tab = oracle.top16_tables(book)
    for r, t in enumerate(send):
        a = batch.out_offsets[r]
        want = oracle.top16_encode(words[:, t].reshape(-1), tab)
        assert want[0] == 5 and bytes(host[a:a + batch.encoded_bytes[r]]) == bytes(want), r
    target = torch.zeros_like(layer)
    assert sz.decode_top16_paged(out, batch.out_offsets, batch.encoded_bytes, target,
                                 sz.PagedBatch(recv, bw, "cuda"), tables=tables) == \
        batch.total_raw_bytes
    check_restored(words, send, recv, target, [True] * len(send))
