"""Presence spans of the palette encode (a workgroup's mask covers 2^k tiles, the encode
forms the palette from a payload's masks): span sizes on both sides of the rule, spans
that cross from the K to the V plane, planes that end inside a tile, and high bytes
present in a single word (a request's first, last, plane-border or a random one), which
a span that skipped a chunk would lose. Payloads byte for byte with the oracle's, a
payload with one high byte too many as 255 alone, and the decode word for word."""

import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = {
    # blocks of 1024 words (four per tile and plane) of each request: at most 512 tiles
    # -> spans of two tiles
    "two_tiles": [1, 2, 3, 4, 5, 9, 1023, 1024],
    # 514 tiles at most -> four tiles, with enough spans in all
    "four_tiles": [1027] * 2 + [1, 6, 15],
    # 514 tiles alone -> the tile presence pass and its reduce
    "tile_pass": [1027],
    # 2050 tiles at most -> sixteen tiles
    "sixteen_tiles": [4099] * 2 + [37],
}
# the run geometry: blocks of 1032 words (a chunk in two blocks, planes that end inside
# a chunk) and of 3848 (most chunks in one)
BLOCK_WORDS = {1024: CASES, 1032: ["two_tiles", "four_tiles", "tile_pass"], 3848: ["two_tiles"]}


@pytest.fixture(scope="module")
def sz():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")
    from unchainkv_amd import splitzip_cuda

    assert splitzip_cuda.available(), splitzip_cuda.load_error()
    return splitzip_cuda


@pytest.mark.parametrize("bits", [6, 5])
@pytest.mark.parametrize("bw,name", [(bw, n) for bw, names in BLOCK_WORDS.items() for n in names])
def test_spans(sz, bw, name, bits):
    print("[case] palette spans", bw, name, bits, flush=True)
    counts = CASES[name]
    limit = 64 if bits == 6 else 32
    rng = np.random.default_rng(len(counts) + bits)
    pool = sum(counts) + 3
    words = rng.integers(0, 1 << 16, (2, pool, bw), dtype=np.uint16)
    words = ((0x40 + (words >> 8) % (limit - 5)) << 8 | (words & 0xFF)).astype(np.uint16)
    ids = rng.permutation(pool).tolist()
    send, at = [], 0
    for c in counts:
        send.append(ids[at:at + c])
        at += c
    overflow = len(counts) - 3 if len(counts) > 1 else -1
    for r, t in enumerate(send):
        flat = words[:, t].reshape(-1)
        n = flat.size
        places = [0, n // 2 - 1, n // 2, n - 1, int(rng.integers(1, n // 2 - 1))]
        for k, place in enumerate(places):
            flat[place] = (k << 8) | 7  # high bytes 0 to 4 once each
        if r == overflow:
            # a request too short for limit - 5 more high bytes overflows by its own
            flat[1:1 + limit - 5] = (0x40 + np.arange(limit - 5)) << 8
            flat[int(rng.integers(n // 2 + 1, n - 1))] = 0xFF00
        words[:, t] = flat.reshape(2, len(t), bw)
    layer = torch.from_numpy(words.view(np.int16)).cuda().view(torch.bfloat16)
    batch = sz.PagedBatch(send, bw, "cuda")
    offsets, sizes, _ = batch.palette_layout(bits)
    out = batch.new_palette_buffer(bits).fill_(0x5A)
    assert sz.encode_bf16_paged(layer, batch, out, batch.new_palette_workspace(), bits) == \
        sum(sizes)
    host = out.cpu().numpy()
    for r, t in enumerate(send):
        got = host[offsets[r]:offsets[r] + sizes[r]]
        if r == overflow:
            assert got[0] == 255 and (got[1:] == 0x5A).all(), r
        else:
            assert bytes(got) == bytes(oracle.palette_encode(words[:, t].reshape(-1), bits)), r
    recv = [[ids[(b + 1) % pool] for b in range(at - len(t), at)]
            for t, at in zip(send, np.cumsum(counts))]
    target = torch.zeros_like(layer)
    assert sz.decode_bf16_paged(out, offsets, sizes, target, sz.PagedBatch(recv, bw, "cuda"),
                                bits) == batch.total_raw_bytes
    restored = target.view(torch.int16).cpu().numpy().view(np.uint16)
    for r, (t, u) in enumerate(zip(send, recv)):
        want = words[:, t] if r != overflow else np.zeros_like(words[:, t])
        assert np.array_equal(restored[:, u], want), r
