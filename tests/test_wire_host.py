"""Host side of the wire form (no GPU): the Python header reader and checks agree with the
oracle's layout, and malformed headers are rejected before anything is launched.

No counterpart in the reference (a byte form of buffers(), cache.py:121-123, is this
package's own)."""
import ctypes
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from exactkv_amd import _lib, wire
from exactkv_amd.cache import CompressedKV
from oracle import wire as owire


class _Cache:
    H, D = 2, 128


def _blob(T=37, H=2, seed=3):
    x = np.random.default_rng(seed).permutation(65536).astype(np.uint16)[:T * H * 128].reshape(T, H, 128)
    return torch.from_numpy(owire.pack(x))


def test_header_reader_matches_the_oracle():
    b = _blob()
    assert wire.header(b) == owire.header(b.numpy())
    assert wire._check_blob(b, _Cache)["tokens"] == 37
    assert wire.nbytes(2, 37, wire.header(b)["raw_rows"]) == b.numel()


def test_malformed_blobs_are_rejected():
    b = _blob()
    with pytest.raises(ValueError, match="1-D uint8"):
        wire.header(b[:100])
    bad = b.clone()
    bad[4] = 2                                          # version 2
    with pytest.raises(ValueError, match="not an exactkv"):
        wire._check_blob(bad, _Cache)
    bad = b.clone()
    bad[16] = 38                                        # tokens no longer match the layout
    with pytest.raises(ValueError, match="inconsistent"):
        wire._check_blob(bad, _Cache)
    with pytest.raises(ValueError, match="shorter"):
        wire._check_blob(b[:-256].clone(), _Cache)

    class Four(_Cache):
        H = 4
    with pytest.raises(ValueError, match="heads"):
        wire._check_blob(b, Four)

    bad = b.clone()
    h = wire.header(b)
    assert h["full_pages"] > 0
    rm = bad[h["off_rowmask"]: h["off_rowmask"] + 4 * h["full_pages"] * 2].view(torch.int32)
    rm[0] ^= 1 << 15                                    # one more (or one less) raw row than declared
    with pytest.raises(ValueError, match="declares"):
        wire._check_blob(bad, _Cache)


class _TwoGpus:
    """Stands in for torch.cuda and the library: which GPU is current, and the (entry point, current
    GPU, stream) of every call and upload. GPU i's stream is 100 + i."""

    def __init__(self, monkeypatch, words):
        self.current, self.log = 0, []
        two = self

        class device:
            def __init__(self, dev):
                self.dev = torch.device(dev).index

            def __enter__(self):
                self.was, two.current = two.current, self.dev

            def __exit__(self, *e):
                two.current = self.was

        monkeypatch.setattr(torch.cuda, "current_device", lambda: self.current)
        monkeypatch.setattr(torch.cuda, "device", device)
        monkeypatch.setattr(_lib, "stream", lambda index=None: 100 + (self.current if index is None else index))
        monkeypatch.setattr(_lib, "ptr", lambda t, *a, **k: 0)
        monkeypatch.setattr(_lib, "call", lambda name, *a: self.log.append((name, self.current, a[-1])))
        monkeypatch.setattr(_lib, "fetch", lambda index, w, st: self.log.append(("fetch", index, st)))
        monkeypatch.setattr(_lib, "host_words", lambda index, n: SimpleNamespace(addr=0, view=words))
        monkeypatch.setattr(wire, "_upload", lambda host, dev: self._upload(host, dev))
        monkeypatch.setattr(wire, "_scratch", lambda *a: (torch.empty(1), 3, 5))
        empty = torch.empty
        monkeypatch.setattr(torch, "empty", lambda *a, device=None, **k: empty(*a, **k))

    def _upload(self, host, dev):
        self.log.append(("upload", self.current, 100 + dev.index))     # torch: on the current stream of dev
        return {k: wire._Part(torch.zeros(1), 0) for k in host}


def _cache_of_gpu(index, T):
    c = CompressedKV.__new__(CompressedKV)
    c.B, c.H, c.D, c.TS, c.T, c.cap, c._pending, c._step_rows = 1, 2, 128, 64, T, 1000, None, 32
    for k in ("sm", "code", "base", "rowmask", "rowoff", "raw", "cnt", "_before"):
        setattr(c, k, SimpleNamespace(device=torch.device("cuda", index), shape=(1032,)))
    c.state = [T]
    return c


@pytest.mark.parametrize("gpu", [0, 1])
def test_batches_run_on_the_caches_own_gpu(monkeypatch, gpu):
    """Uploads, launches and waits of a pack and an unpack all go to one stream, that of the cache's
    GPU, with that GPU current, whichever GPU the caller has current."""
    blob = _blob(T=5)
    head = np.frombuffer(blob[:256].numpy().tobytes(), np.int32).tolist()
    words = (ctypes.c_int32 * 68)()                     # flag, then no raw rows for the pack
    two = _TwoGpus(monkeypatch, words)
    cache = _cache_of_gpu(gpu, 5)
    wire.pack_many(cache, [0])
    words[1:65] = head                                  # and header, raw rows, counter for the unpack
    on_gpu = SimpleNamespace(dtype=blob.dtype, dim=blob.dim, numel=blob.numel, stride=blob.stride, device=cache.sm.device)
    wire.unpack_many([on_gpu], cache, [0])
    assert [n for n, _, _ in two.log] == ["upload", "exkv_wire_count", "fetch", "upload", "exkv_wire_pack",
                                          "upload", "exkv_wire_check", "fetch", "upload", "exkv_wire_unpack"]
    assert {(d, st) for _, d, st in two.log} == {(gpu, 100 + gpu)} and two.current == 0
