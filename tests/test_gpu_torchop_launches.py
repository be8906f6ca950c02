"""Torch-op plan, encode and decode at the edges of a tile launch's payloads (64 in
the small argument struct, 256 in the large one), with equal payloads (the payload by
a division) and ragged ones (by the search of the first tiles): plans and payload
bytes are the oracle's, and the decode restores every word."""

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


@pytest.mark.parametrize("ragged", [False, True])
@pytest.mark.parametrize("requests", [1, 64, 65, 256, 257])
def test_payloads_of_a_launch(sz, requests, ragged):
    print("[case] torchop launch", requests, ragged, flush=True)
    rng = np.random.default_rng(requests + 1000 * ragged)
    bw = 1024
    counts = [1 + (r * 7) % 5 if ragged else 2 for r in range(requests)]
    pool = sum(counts) + 3
    layer_np = (rng.standard_normal((2, pool, bw)).astype(np.float32)
                * 10.0 ** rng.integers(-2, 3, (2, pool, 1))).astype(np.float32)
    words = (layer_np.view(np.uint32) >> 16).astype(np.uint16)
    layer = torch.from_numpy(words.view(np.int16)).cuda().view(torch.bfloat16)

    def tables(seed):
        ids = np.random.default_rng(seed).permutation(pool).tolist()
        ends = np.cumsum([0] + counts)
        return [ids[a:b] for a, b in zip(ends, ends[1:])]

    send, recv = tables(1), tables(2)
    batch = sz.PagedBatch(send, bw, "cuda")
    fields = sz.read_torchop_plans(sz.plan_torchop_paged(layer, batch).cpu().numpy())
    plans = sz.plan_torchop_paged(layer, batch)
    sizes = [size for _, size in fields]
    offsets = np.cumsum([0] + sizes)[:-1].tolist()
    out = torch.zeros(sum(sizes), dtype=torch.uint8, device="cuda")
    assert sz.encode_torchop_paged(layer, batch, plans, out, offsets, sizes) == sum(sizes)
    host = out.cpu().numpy()
    for r, t in enumerate(send):
        expected = oracle.encode_torchop(words[:, t].reshape(-1))
        assert fields[r] == (int(expected[0]), expected.size), r
        assert bytes(host[offsets[r]:offsets[r] + sizes[r]]) == expected.tobytes(), r
    target = torch.zeros_like(layer)
    assert sz.decode_torchop_paged(out, offsets, sizes, target, sz.PagedBatch(recv, bw, "cuda")) \
        == sum(batch.raw_bytes)
    got = target.view(torch.int16).cpu().numpy().view(np.uint16)
    for r, (t, u) in enumerate(zip(send, recv)):
        assert np.array_equal(got[:, u], words[:, t]), r
