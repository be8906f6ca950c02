"""The host module's conversion of per-request numbers to u64 arrays, and the attention
call's bounds check in the library: the same answers as the plain Python forms."""

import ctypes

import numpy as np
import pytest

from unchainkv_amd import codec_format, splitzip_cuda as sz


@pytest.mark.parametrize("values", [
    [0, 1, (1 << 64) - 1], [3], [True, 7], [], [5.9, 2], [-1, 4], [1 << 64, 3],
    np.array([4, 9], dtype=np.int64), np.array([4.5, 9.0]), bytes(range(16)), (8, 16)])
def test_u64_array(values):
    want = (ctypes.c_ulonglong * len(values))(*map(int, values))
    got = sz._u64_array(values)
    assert len(got) == len(want) and list(got) == list(want)


def fits(offsets, contexts, block_tokens, heads, size, head_dim=128):
    lib = sz._load()
    need = ctypes.c_ulonglong(123)
    ok = lib.kvq_splitzip_top16_decode_attention_fits(
        sz._u64_array(offsets), sz._u64_array(contexts), len(offsets), block_tokens, heads,
        head_dim, size, ctypes.byref(need))
    return bool(ok), need.value


@pytest.mark.parametrize("contexts", [[1], [16, 17], [300, 5, 4096], [32768]])
@pytest.mark.parametrize("heads,block_tokens", [(1, 16), (3, 8), (8, 32)])
def test_attention_bounds(contexts, heads, block_tokens):
    if not sz.available():
        pytest.skip(sz.load_error())
    offsets, end = [], 11
    for ctx in contexts:
        offsets.append(end)
        span = -(-ctx // block_tokens) * block_tokens
        end += codec_format.top16_encoded_size(2 * span * heads * 128)
    assert fits(offsets, contexts, block_tokens, heads, end)[0]
    assert not fits(offsets, contexts, block_tokens, heads, end - 1)[0]
    assert not fits(offsets[:-1] + [end + 1], contexts, block_tokens, heads, end)[0]
    assert not fits([-5] + offsets[1:], contexts, block_tokens, heads, end)[0]
    assert not fits(offsets, [-3] + contexts[1:], block_tokens, heads, end)[0]
    assert not fits(offsets, contexts, 0, heads, end)[0]
    assert not fits(offsets, contexts, block_tokens, 0, end)[0]
    assert not fits(offsets, contexts, block_tokens, heads, end, head_dim=64)[0]


class RecordingLibrary:
    """Stands in for the C library: notes which entry is called, with what result."""

    def __init__(self, results):
        self.results, self.calls = results, []

    def __getattr__(self, name):
        if name not in self.results:
            raise AttributeError(name)

        def entry(*args):
            self.calls.append(name)
            return self.results[name]

        return entry


@pytest.mark.parametrize("block_words,blocks,entries", [
    (1024, 3, ["tile"]), (16384, 256, ["tile"]), (640, 3, ["runs"]), (8, 256, ["runs"]),
    (1032, 2, ["runs"]), (12, 3, []), (1024, 257, []), (640, 257, [])])
@pytest.mark.parametrize("answer", [64, 0, -1])
def test_one_host_table_entry_per_geometry(block_words, blocks, entries, answer):
    """A host block table is offered to the entry of its geometry and to no other."""
    torch = pytest.importorskip("torch")
    name = {"tile": "decode_x_host_blocks", "runs": "decode_x_host_runs"}
    lib = RecordingLibrary({n: answer for n in name.values()})
    source, out = torch.zeros(4, dtype=torch.uint8), torch.zeros((2, 4, 4), dtype=torch.bfloat16)
    got = sz._decode_with_table(lib, name["tile"], "decode_x_blocks", list(range(blocks))[::-1],
                                source, out, 2 * blocks * block_words, block_words, 0, (), torch)
    assert lib.calls == [name[e] for e in entries]
    # (a decline goes on to the device table, which this library does not have)
    assert got == (answer if entries and answer else None)


@pytest.mark.parametrize("offset,context", [
    (1 << 64, 16), ((1 << 64) + 11, 16), (11 - (1 << 64), 16), (-1, 16),
    (11, (1 << 64) + 16), (11, 16 - (1 << 64)), (11.0, 1e30)])
def test_attention_declines_numbers_outside_64_bits(monkeypatch, offset, context):
    """They reach the library neither as they are nor modulo 2^64."""
    torch = pytest.importorskip("torch")
    lib = RecordingLibrary({"kvq_splitzip_top16_decode_attention": 1,
                            "kvq_splitzip_top16_decode_attention_fits": 1})
    monkeypatch.setattr(sz, "_load", lambda: lib)
    monkeypatch.setattr(sz, "_is_cuda", lambda tensor: True)
    q = torch.zeros((2, 4, 128), dtype=torch.bfloat16)
    payloads = torch.zeros(1 << 16, dtype=torch.uint8)
    got = sz.decode_attention_top16(q, payloads, [11, offset], [16, context], 1,
                                    tables=torch.zeros(544, dtype=torch.uint8))
    assert got is None and lib.calls == []
