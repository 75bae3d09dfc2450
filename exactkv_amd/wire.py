"""Wire form of a sequence's compressed cache: pack it into one contiguous byte blob
(KV offload to host memory or disk, transfer between pools, processes or GPUs) and
unpack it into a contiguous or paged cache, on the GPU.

No counterpart in the reference: its caches hand out their six tensors (buffers(),
cache.py:121-123); a byte form of them is this package's own. The blob keeps the
reference format's fields (codec.py:1-25) for one sequence, about 200 bytes per
(token, head) against 256 for bf16. Layout (little-endian, sections at multiples of
256 bytes, gaps zero):

  header   256 B: u32 magic "EXKV", version 1, heads, head_dim, tokens, full_pages,
           tail_rows, raw_rows; u64 off_tail, off_rowmask, off_base, off_sm, off_code,
           off_raw, total
  tail     bf16 [T % 16, H, 128]       the open page's tokens
  rowmask  i32  [T // 16, H]
  base     u8   [T // 16, H, 128]
  sm       u8   [16 * (T // 16), H, 128]
  code     u8   [16 * (T // 16), H, 64]
  raw      bf16 [N, 128]               raw rows in (page, head, token) order

rowoff is implicit (the running count of raw rows in (page, head) order), so a blob
does not depend on where its rows sat in the source pool.
"""
import struct
from array import array

import numpy as np
import torch

from . import _lib
from .cache import CompressedKV
from .kernels import P
from .paged import PagedCompressedKV, _popc16

_NO_WORDS = array("Q")
HEADER = 256
MAGIC = 0x564B5845
VERSION = 1
_KEYS = ("magic", "version", "heads", "head_dim", "tokens", "full_pages", "tail_rows", "raw_rows",
         "off_tail", "off_rowmask", "off_base", "off_sm", "off_code", "off_raw", "total")


def nbytes(H, T, raw_rows):
    """Blob size for H heads, T tokens and raw_rows raw rows."""
    n = _lib.load().exkv_wire_bytes(int(H), int(T), int(raw_rows))
    if n < 0:
        raise ValueError(f"bad wire size arguments H={H} T={T} raw_rows={raw_rows}")
    return n


class _Read:
    """A blob on the GPU with its header and the raw rows of its rowmask section, as
    exkv_wire_check has read them."""
    __slots__ = ("blob", "head", "rows")

    def __init__(self, blob, head, rows):
        self.blob, self.head, self.rows = blob, head, rows

    def numel(self):
        return self.blob.numel()


def _blob_shape(blob):
    if blob.dtype != torch.uint8 or blob.dim() != 1 or blob.numel() < HEADER:
        raise ValueError("a wire blob is a 1-D uint8 tensor of at least 256 bytes")


def header(blob):
    """The header fields of a blob (a uint8 tensor on any device) as a dict."""
    if isinstance(blob, _Read):
        return dict(zip(_KEYS, struct.unpack_from("<8I7Q", blob.head)))
    _blob_shape(blob)
    vals = struct.unpack_from("<8I7Q", bytes(blob[:HEADER].cpu().numpy()))
    return dict(zip(_KEYS, vals))


def _sequence(cache, seq):
    """(T, pool page of each sequence page, first tail row, pool pages, open page exists)."""
    H = cache.H
    if isinstance(cache, PagedCompressedKV):
        t = cache.table
        if not 0 <= seq < t.max_seqs or t._pages[seq] is None:
            raise ValueError(f"slot {seq} is not in use")
        T = t.length(seq)
        return T, t._pages[seq], cache.cap + seq * H * P, t.num_pages, T // P < t.max_pages
    if isinstance(cache, CompressedKV):
        if not 0 <= seq < cache.B:
            raise ValueError(f"sequence {seq} outside the cache's {cache.B}")
        NP = cache.TS // P
        T = cache.T
        return T, range(seq * NP, seq * NP + NP), cache.cap + seq * H * P, cache.B * NP, T < cache.TS
    raise TypeError(type(cache))


class _Part:
    """A part of a device buffer, by its address."""
    __slots__ = ("buf", "off")

    def __init__(self, buf, off):
        self.buf, self.off = buf, off

    def data_ptr(self):
        return self.buf.data_ptr() + self.off


def _upload(host, dev):
    """Numpy arrays (a dict) on the GPU, in one buffer and one copy that waits for nothing."""
    offs, size = {}, 0
    for k, v in host.items():
        offs[k] = size
        size += -(-v.nbytes // 16) * 16
    pin = torch.empty(size, dtype=torch.uint8, pin_memory=True)
    view = pin.numpy()
    for k, v in host.items():
        view[offs[k]:offs[k] + v.nbytes] = v.reshape(-1).view(np.uint8)
    buf = torch.empty(size, dtype=torch.uint8, device=dev)
    buf.copy_(pin, non_blocking=True)
    return {k: _Part(buf, o) for k, o in offs.items()}


def _host_pages(cache, infos):
    """The sequences' page lists, token counts, first tail rows and open flags as arrays."""
    width = max(max(len(i[1]) for i in infos), 1)
    pages = np.zeros((len(infos), width), np.int32)
    for row, i in zip(pages, infos):
        row[:len(i[1])] = np.arange(i[1].start, i[1].stop) if isinstance(i[1], range) else i[1]
    return dict(pages=pages, tokens=np.array([i[0] for i in infos], np.int32),
                tails=np.array([i[2] for i in infos], np.int64), open=np.array([int(i[4]) for i in infos], np.int32))


def _host_blobs(blobs):
    return dict(blobs=np.array([_lib.ptr(b, align=256, what="blob") for b in blobs], np.int64),
                sizes=np.array([b.numel() for b in blobs], np.int64))


def _scratch(cache, infos, dev):
    """(ws, its row stride, the most tokens) of a pack or unpack call."""
    max_t = max(i[0] for i in infos)
    ws_stride = (max_t // P) * cache.H + 3
    return torch.empty(len(infos), ws_stride, dtype=torch.int32, device=dev), ws_stride, max_t


def _batch_args(cache, seqs, infos, blobs, dev):
    """Device arrays of one pack / unpack call."""
    host = _host_pages(cache, infos)
    d = _upload(dict(host, **_host_blobs(blobs)), dev)
    d["ws"], ws_stride, max_t = _scratch(cache, infos, dev)
    return d, host["pages"].shape[1], max_t, ws_stride


def pack(cache, seq):
    """Sequence `seq` (a CompressedKV slot b, or a PagedCompressedKV slot) -> uint8 blob on
    the cache's GPU. Synchronises once (to size the blob)."""
    return pack_many(cache, [seq])[0]


def pack_many(cache, seqs):
    """Blobs of several sequences of one cache, packed by one call (two launches)."""
    if cache._pending is not None:
        raise RuntimeError("call check_overflow() before packing")
    seqs = list(seqs)
    if not seqs:
        return []
    H, dev = cache.H, cache.sm.device
    if dev.index != torch.cuda.current_device():       # uploads and launches on one stream, the cache's GPU's
        with torch.cuda.device(dev):
            return pack_many(cache, seqs)
    infos = [_sequence(cache, s) for s in seqs]
    host, n = _host_pages(cache, infos), len(seqs)
    d, width = _upload(host, dev), host["pages"].shape[1]
    d["ws"], ws_stride, max_t = _scratch(cache, infos, dev)
    st = _lib.stream()
    hw = _lib.host_words(dev.index, n + 1)
    _lib.call("exkv_wire_count", _lib.ptr(cache.rowmask), infos[0][3], n, d["pages"].data_ptr(), width,
              d["tokens"].data_ptr(), max_t, H, hw.addr + 4, st)
    _lib.fetch(dev.index, _NO_WORDS, st)
    blobs = [torch.empty(nbytes(H, i[0], c), dtype=torch.uint8, device=dev) for i, c in zip(infos, hw.view[1:n + 1])]
    d.update(_upload(_host_blobs(blobs), dev))
    _lib.call("exkv_wire_pack", _lib.ptr(cache.sm), _lib.ptr(cache.code), _lib.ptr(cache.base),
              _lib.ptr(cache.rowmask), _lib.ptr(cache.rowoff), _lib.ptr(cache.raw), cache.raw.shape[0], infos[0][3],
              len(seqs), d["pages"].data_ptr(), width, d["tokens"].data_ptr(), d["tails"].data_ptr(),
              d["blobs"].data_ptr(), d["sizes"].data_ptr(), max_t, H, cache.D, d["ws"].data_ptr(), ws_stride, st)
    return blobs


def _check_blob(blob, cache):
    h = header(blob)
    if h["magic"] != MAGIC or h["version"] != VERSION:
        raise ValueError(f"not an exactkv wire blob (magic {h['magic']:#x}, version {h['version']})")
    if h["head_dim"] != cache.D or h["heads"] != cache.H:
        raise ValueError(f"blob holds {h['heads']} heads of dim {h['head_dim']}, the cache {cache.H} of {cache.D}")
    T, N = h["tokens"], h["raw_rows"]
    if h["total"] != nbytes(cache.H, T, N) or h["full_pages"] != T // P or h["tail_rows"] != T % P:
        raise ValueError("inconsistent wire header")
    if blob.numel() < h["total"]:
        raise ValueError(f"blob of {blob.numel()} bytes is shorter than its header's {h['total']}")
    npf = h["full_pages"] * cache.H
    if npf:
        if isinstance(blob, _Read):
            rows = blob.rows
        else:
            rm = blob[h["off_rowmask"]: h["off_rowmask"] + 4 * npf].view(torch.int32)
            rows = int(_popc16(rm & 0xFFFF).sum().item())
        if rows != N:
            raise ValueError(f"blob's rowmask marks {rows} raw rows, its header declares {N}")
    return h


def unpack(blob, cache, seq):
    """Write a blob into sequence `seq` of `cache`: a CompressedKV slot b (the cache then
    holds the blob's T tokens, as after prefill_slot) or a PagedCompressedKV slot already
    added with table.add(T) for the blob's T. The raw pool grows first if needed."""
    unpack_many([blob], cache, [seq])


def unpack_many(blobs, cache, seqs):
    """unpack for several blobs and sequences of one cache in one call (two launches)."""
    seqs = list(seqs)
    if len(blobs) != len(seqs) or len(set(seqs)) != len(seqs):
        raise ValueError("one distinct sequence per blob")
    if not seqs:
        return
    dev, n = cache.sm.device, len(seqs)
    if dev.index != torch.cuda.current_device():       # uploads and launches on one stream, the cache's GPU's
        with torch.cuda.device(dev):
            return unpack_many(blobs, cache, seqs)
    for b in blobs:
        _blob_shape(b)
        # the GPU reads a blob through its address; one that is copied there first comes out dense, and
        # has been taken strided where it holds no whole page, whose masks need dense words
        if b.stride(0) != 1 and (b.device == dev or header(b)["full_pages"]):
            raise ValueError("a wire blob must be contiguous")
    blobs = [b if b.device == dev else b.to(dev) for b in blobs]
    up = _upload(_host_blobs(blobs), dev)
    st = _lib.stream()
    hw = _lib.host_words(dev.index, 65 * n + 2)
    _lib.call("exkv_wire_check", n, up["blobs"].data_ptr(), up["sizes"].data_ptr(), cache.H, _lib.ptr(cache.cnt, align=4),
              hw.addr + 4, st)
    _lib.fetch(dev.index, _NO_WORDS, st)
    head, rows, cnt = bytes(hw.view)[4:4 + HEADER * n], hw.view[1 + 64 * n:1 + 65 * n], hw.view[1 + 65 * n]
    heads = [_check_blob(_Read(b, head[HEADER * i:HEADER * (i + 1)], rows[i]), cache) for i, b in enumerate(blobs)]
    if cache._pending is not None:
        raise RuntimeError("call check_overflow() before unpacking")
    Ts = [h["tokens"] for h in heads]
    if isinstance(cache, CompressedKV):
        if len(set(Ts)) != 1 or Ts[0] > cache.TS:
            raise ValueError(f"blobs of {sorted(set(Ts))} tokens into a cache of {cache.TS} (one length per cache)")
        cache.T = Ts[0]
        cache.state[0] = Ts[0]
    else:
        for s, T in zip(seqs, Ts):
            if cache.table.length(s) != T:
                raise ValueError(f"blob of {T} tokens into a slot of {cache.table.length(s)}")
    N = sum(h["raw_rows"] for h in heads)
    if cnt + N > cache.cap:
        cache._grow(cnt + N)
    infos = [_sequence(cache, s) for s in seqs]                 # tail rows after any growth
    host = _host_pages(cache, infos)
    d, width = _upload(host, dev), host["pages"].shape[1]
    d["ws"], ws_stride, max_t = _scratch(cache, infos, dev)
    _lib.call("exkv_wire_unpack", _lib.ptr(cache.sm), _lib.ptr(cache.code), _lib.ptr(cache.base),
              _lib.ptr(cache.rowmask), _lib.ptr(cache.rowoff), _lib.ptr(cache.raw), cache.raw.shape[0], cache.cap,
              _lib.ptr(cache.cnt, align=4), _lib.ptr(cache._before, align=4), infos[0][3], len(seqs),
              d["pages"].data_ptr(), width, d["tokens"].data_ptr(), d["open"].data_ptr(), d["tails"].data_ptr(),
              up["blobs"].data_ptr(), up["sizes"].data_ptr(), max_t, cache.H, cache.D, d["ws"].data_ptr(), ws_stride, st)
    cache._keep_headroom(cnt + N)
