"""GPU encoder and decoder vs the CPU oracle (reference codec.py:31-73; reference GPU
test tests/test_exactkv.py:52-58, here with all six tensors byte-identical)."""
import json
import os

import numpy as np
import pytest
import torch

import exactkv_amd as exactkv
from exactkv_amd import synthetic
from exactkv_amd import kernels
from oracle import codec as ocodec
from tests.conftest import same_bits, u16
from tests.golden import cases

pytestmark = pytest.mark.gpu
DEV = "cuda"
GOLD = os.path.join(os.path.dirname(__file__), "golden")


def _say(*a):
    print("[case]", *a, flush=True)


def _gpu_encode(x):
    """Encode [B,T,H,D] with the HIP encoder into fresh cache buffers (reference tests:19-26)."""
    B, T, H, D = x.shape
    c = exactkv.CompressedKV(B, T, H, D, reserve=1.0)
    st = (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2))
    kernels.encode_pages(x, st, c._buf(), 0, 0, B, T // 16)
    assert int(c.cnt.item()) <= c.cap
    return c


def _compare(c, ref, name):
    for k in ("sm", "code", "base", "rowmask", "rowoff"):
        assert np.array_equal(getattr(c, k).cpu().numpy(), ref[k]), (name, k)
    n = int(c.cnt.item())
    assert n == ref["raw"].shape[0], name
    assert np.array_equal(u16(c.raw[:n]), ref["raw"]), (name, "raw")


@pytest.mark.parametrize("name", list(cases.CASES))
def test_encoder_bytes_equal_oracle_and_decode_exact(name):
    x = cases.CASES[name][0]()
    _say("encoder", name, tuple(x.shape))
    ref = ocodec.encode(u16(x))
    xd = x.to(DEV)
    c = _gpu_encode(xd)
    _compare(c, ref, name)
    assert same_bits(kernels.decode_to_bf16(c.buffers(), x.shape[1]), xd), name


def test_encode_reference_api_matches_golden_bytes():
    z = np.load(os.path.join(GOLD, "codec_vectors.npz"))
    for name, (make, stored) in cases.CASES.items():
        if not stored:
            continue
        _say("encode_reference", name)
        x = make()
        c = exactkv.encode_reference(x)                 # CPU in, CPU out, computed on the GPU
        for k in ("sm", "code", "base", "rowmask", "rowoff", "raw"):
            got = c[k].numpy() if k != "raw" else u16(c[k])
            assert np.array_equal(got, z[f"{name}/{k}"]), (name, k)
        assert same_bits(exactkv.decode_reference(c), x), name
        cg = exactkv.encode_reference(x.to(DEV))        # GPU in, GPU out
        assert cg["sm"].is_cuda and same_bits(exactkv.decode_reference(cg), x.to(DEV))


def test_encode_reference_hashed_cases():
    import hashlib
    h = json.load(open(os.path.join(GOLD, "codec_hashes.json")))["cases"]
    for name, (make, stored) in cases.CASES.items():
        if stored:
            continue
        _say("encode_reference hashed", name)
        c = exactkv.encode_reference(make().to(DEV))
        for k in ("sm", "code", "base", "rowmask", "rowoff", "raw"):
            a = u16(c[k]) if k == "raw" else c[k].cpu().numpy()
            assert hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest() == h[name][k]["sha256"], (name, k)


def test_encoder_strided_source_and_offsets():
    """Encode pages [pg0, pg0+npg) of sequences [b0, b0+nb) from a strided view."""
    big = synthetic.make_kv(3, 96, 8, kind="k", seed=4).to(DEV)
    src = big[:, :, ::2]                                  # heads 0, 2, 4, 6: head stride 256
    B, T, H, D = src.shape
    _say("strided encode", tuple(src.shape), src.stride())
    c = exactkv.CompressedKV(4, 128, H, D, reserve=1.0)
    st = (src.stride(0), 16 * src.stride(1), src.stride(1), src.stride(2))
    kernels.encode_pages(src[1:], st, c._buf(), 2, 1, 2, T // 16)        # sequences 2,3 pages 1..6
    ref = ocodec.encode(u16(src[1:].contiguous()))
    NP = T // 16
    assert np.array_equal(c.sm[2:4, 16:16 + T].cpu().numpy(), ref["sm"])
    assert np.array_equal(c.code[2:4, 16:16 + T].cpu().numpy(), ref["code"])
    assert np.array_equal(c.base[2:4, 1:1 + NP].cpu().numpy(), ref["base"])
    assert np.array_equal(c.rowmask[2:4, 1:1 + NP].cpu().numpy(), ref["rowmask"])
    assert np.array_equal(c.rowoff[2:4, 1:1 + NP].cpu().numpy(), ref["rowoff"])
    assert not c.sm[:2].any() and not c.sm[2:4, :16].any()              # nothing else written


def test_encoder_overflow_skips_rows_past_cap():
    x = synthetic.stress_pages(1, 64, 2, seed=9).to(DEV)       # many raw rows
    ref = ocodec.encode(u16(x))
    n = ref["raw"].shape[0]
    B, T, H, D = x.shape
    c = exactkv.CompressedKV(B, T, H, D, reserve=0.0)                   # cap 64 < n
    assert n > c.cap
    sentinel = torch.full_like(c.raw, 7.0)
    c.raw.copy_(sentinel)
    st = (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2))
    kernels.encode_pages(x, st, c._buf(), 0, 0, B, T // 16)
    assert int(c.cnt.item()) == n and int(c._before.item()) == 0
    assert np.array_equal(u16(c.raw[: c.cap]), ref["raw"][: c.cap])
    assert same_bits(c.raw[c.cap:], sentinel[c.cap:])                  # tail area untouched


@pytest.mark.parametrize("T", [1, 15, 16, 17, 100, 128])
def test_decode_partial_lengths(T):
    x = cases.CASES["allpat_perm"][0]().to(DEV)
    c = _gpu_encode(x)
    _say("decode T", T)
    assert same_bits(kernels.decode_to_bf16(c.buffers(), T), x[:, :T])


@pytest.mark.parametrize("width,offset", [(128, 0), (130, 0), (136, 2)])
def test_encoder_row_alignment(width, offset):
    """Source rows inside wider rows: 16-byte aligned rows (width 128) take the wide raw-row
    copy, 4-byte aligned ones (row pitch 130, or a 2-element offset) the narrow one; the
    bytes equal the oracle's either way."""
    x = synthetic.stress_pages(2, 64, 4, seed=21)
    big = torch.zeros(2, 64, 4, width + offset, dtype=torch.bfloat16)
    big[..., offset:offset + 128] = x
    src = big.to(DEV)[..., offset:offset + 128]
    _say("aligned encode", width, offset, src.stride())
    ref = ocodec.encode(u16(x))
    c = exactkv.CompressedKV(2, 64, 4, 128, reserve=1.0)
    st = (src.stride(0), 16 * src.stride(1), src.stride(1), src.stride(2))
    kernels.encode_pages(src, st, c._buf(), 0, 0, 2, 4)
    assert ref["raw"].shape[0] > 0
    _compare(c, ref, f"width {width} offset {offset}")


def _popc16(t):
    t = t.to(torch.int32)
    return sum((t >> i) & 1 for i in range(16))


@pytest.mark.parametrize("chained", [True, False])
@pytest.mark.parametrize("B,T,H", [(8, 8208, 16), (5, 8192, 32)])
def test_encoder_slot_scan_full_size(B, T, H, chained):
    """65,664 and 81,920 units, 5% outlier rows, counter starting at 7, through the
    chained scan (look-back over 65 and 80 blocks) and the three-launch scan:
    every rowoff is 7 + the raw rows of the units before it in (sequence, page, head)
    order, the counter ends at 7 + all of them, and decoding gives back every bit."""
    x = synthetic.make_kv(B, T, H, kind="k", seed=31, raw_row_rate=0.05, device=DEV)
    _say("slot scan", B, T, H, "units", B * (T // 16) * H, "chained", chained)
    c = exactkv.CompressedKV(B, T, H, 128, reserve=0.08)
    c.cnt.fill_(7)
    st = (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2))
    kernels.encode_pages(x, st, c._buf(), 0, 0, B, T // 16, chained=chained)
    per = _popc16(c.rowmask).flatten().to(torch.int64)
    n = int(per.sum().item())
    assert n > 0.04 * B * T * H
    assert int(c.cnt.item()) == 7 + n and int(c._before.item()) == 7 and 7 + n <= c.cap
    want = 7 + torch.cumsum(per, 0) - per
    assert torch.equal(c.rowoff.flatten().to(torch.int64), want)
    assert same_bits(kernels.decode_to_bf16(c.buffers(), T), x)


def test_encoder_chained_equals_multi_launch():
    """Encodes of different sizes one after another on one stream (the chained scan's
    workspace is shared: its generation advances between calls), each byte-identical to
    the three-launch scan on the same input and counter, including a raw pool too small for
    every raw row (slots past cap skipped, counter past cap), head dims 64 and 256, a unit
    with every row raw, and source rows 4-byte but not 16-byte aligned (the raw-row copy's
    word path). All but the last have masks that are not read by fours, so that 12,289 units
    are enough for these scans."""
    cases = [(3, 16 * 1367, 3, 0.05, 0.5, 128), (2, 16 * 2051, 5, 0.02, 0.5, 128), (3, 16 * 1389, 3, 0.3, 0.5, 128),
             (5, 16 * 839, 3, 0.05, 0.002, 128), (3, 16 * 1367, 3, 0.05, 0.5, 128), (7, 16 * 1795, 1, 0.05, 0.5, 64),
             (2, 16 * 2051, 3, 0.05, 0.5, 256), (8, 8208, 16, 0.01, 0.5, 64)]
    kernels.release_workspaces()
    for i, (B, T, H, rate, reserve, D) in enumerate(cases):
        x = synthetic.make_kv(B, T, H, D=D, kind="k", seed=40 + i, raw_row_rate=rate, device=DEV)
        if i == 2:
            x[0, 16:32, 1] *= 2.0 ** 100                   # a floor >= 128 in every channel: all 16 rows raw
        if i == 4:                                         # rows 4-byte aligned but not 16
            xx = torch.empty(B, T, H, D + 2, dtype=x.dtype, device=DEV)
            xx[..., 2:] = x
            x = xx[..., 2:]
        st = (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2))
        out = []
        for chained in (True, False):
            c = exactkv.CompressedKV(B, T, H, D, reserve=reserve)
            c.cnt.fill_(3)
            kernels.encode_pages(x, st, c._buf(), 0, 0, B, T // 16, chained=chained)
            out.append(c)
        ws, = kernels._SCAN.values()
        assert ws[:2].tolist() == [0, i + 1]               # no ticket out, a generation for each chained call
        a, b = out
        _say("chained vs three-launch scan", B, T, H, D, "counter", int(a.cnt.item()), "cap", a.cap)
        for f in ("sm", "code", "base", "rowmask", "rowoff", "cnt", "_before"):
            assert torch.equal(getattr(a, f), getattr(b, f)), f
        n = min(int(a.cnt.item()), a.cap)
        assert torch.equal(a.raw[:n], b.raw[:n])
        if i == 2:
            assert int(b.rowmask[0, 1, 1].item()) == 0xFFFF
            assert same_bits(kernels.decode_to_bf16(b.buffers(), T), x)


@pytest.mark.parametrize("B,npg,H,b0,pg0,D,paged", [
    (1, 1, 1, 0, 0, 64, False),         # one unit
    (1, 8, 8, 0, 0, 128, False),        # 64 units: one block full
    (1, 13, 5, 0, 1, 128, False),       # 65 units, masks not 16-byte aligned
    (3, 41, 8, 1, 2, 64, False),        # masks of several sequences, aligned
    (3, 41, 3, 1, 1, 64, False),        # and not
    (2, 37, 3, 0, 0, 256, True),
    (4, 512, 8, 0, 0, 64, False),       # 16,384 units: the last size of 64-unit blocks
    (1, 5462, 3, 0, 0, 64, False),      # 16,386: 128-unit blocks
    (8, 512, 8, 0, 0, 64, False),       # 32,768
    (3, 3641, 3, 0, 0, 64, False),      # 32,769: 256-unit blocks
    (8, 1024, 8, 0, 0, 64, False),      # 65,536: the last direct scan
    (1, 65537, 1, 0, 0, 64, False),     # the first chained one
    (1, 65536, 1, 0, 0, 64, True),
])
def test_encoder_slot_scan_block_edges(B, npg, H, b0, pg0, D, paged):
    """Raw-row slots at the edges of the slot scan's block sizes and mask layouts: every unit's
    rowoff is the counter plus the raw rows of the units before it, the raw rows are in their
    slots, and the counter and its value before are right."""
    _say("slot scan edges", B, npg, H, b0, pg0, D, paged)
    g = torch.Generator(device=DEV).manual_seed(B * npg + H)
    x = torch.randn(B, npg * 16, H, D, generator=g, device=DEV).bfloat16()
    rows = torch.rand(B, npg * 16, H, generator=g, device=DEV) < 0.02
    x[rows, 3] *= 2.0 ** -30
    c = exactkv.CompressedKV(b0 + B, (pg0 + npg) * 16, H, D, reserve=0.2)
    c.cnt.fill_(5)
    c.raw.zero_()
    st = (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2))
    if paged:
        NP = c.TS // 16
        order = torch.randperm(c.B * NP, generator=g, device=DEV)[:B * npg].view(B, npg)
        kernels.encode_pages_paged(x, st, c._buf(), order.to(torch.int32), B, npg)
        pick = order.reshape(-1)
        rm, off = (t.view(-1, H)[pick].view(B, npg, H) for t in (c.rowmask, c.rowoff))
    else:
        kernels.encode_pages(x, st, c._buf(), b0, pg0, B, npg)
        rm, off = (t[b0:, pg0:] for t in (c.rowmask, c.rowoff))
    bits = ((rm[..., None] >> torch.arange(16, device=DEV)) & 1).bool()        # [B, npg, H, 16]
    assert bool((bits.permute(0, 1, 3, 2).reshape(rows.shape) | ~rows).all())
    per = bits.sum(-1).reshape(-1)
    excl = torch.cumsum(per, 0) - per + 5
    assert torch.equal(off.reshape(-1).long(), excl)
    n = int(per.sum())
    assert int(c.cnt.item()) == 5 + n and int(c._before.item()) == 5
    want = x.view(B, npg, 16, H, D).permute(0, 1, 3, 2, 4)[bits]               # (sequence, page, head, token) order
    assert 5 + n <= c.cap and torch.equal(c.raw[5:5 + n].view(torch.int16), want.view(torch.int16))
    assert not bool(c.raw[:5].view(torch.int16).any()) and not bool(c.raw[5 + n:c.cap].view(torch.int16).any())


def _source(B, T, H, D, rate, g, shift=0):
    """bf16 [B, T, H, D], a share of rows raw, its memory `shift` elements off an allocation's start."""
    x = torch.empty(B * T * H * D + shift, dtype=torch.bfloat16, device=DEV)[shift:].view(B, T, H, D)
    for b in range(B):
        x[b] = torch.randn(T, H, D, generator=g, device=DEV)
    x[torch.rand(B, T, H, generator=g, device=DEV) < rate, 3] *= 2.0 ** -30
    return x


def _check_slots(x, rm, off, raw, cap, cnt0, cnt):
    """Raw-row slots of pages encoded from x [B, T, H, D], masks and offsets [B, T / 16, H]: each unit's
    offset is cnt0 plus the raw rows of the units before it, those below cap are in their slots, the
    counter is past all of them."""
    B, T, H, D = x.shape
    bits = ((rm[..., None] >> torch.arange(16, device=DEV)) & 1).bool()          # [B, pages, H, 16]
    per = bits.sum(-1).reshape(-1)
    assert torch.equal(off.reshape(-1).long(), torch.cumsum(per, 0) - per + cnt0)
    n = int(per.sum())
    assert cnt == cnt0 + n
    want = x.view(B, T // 16, 16, H, D).permute(0, 1, 3, 2, 4)[bits]             # (sequence, page, head, token) order
    m = min(cap - cnt0, n)
    assert torch.equal(raw[cnt0:cnt0 + m].view(torch.int16), want[:m].view(torch.int16))
    return n


@pytest.mark.parametrize("npg,H,pg0,paged,prefill,direct", [
    (8192, 8, 0, False, False, True), (8193, 8, 0, False, False, False),      # 65,536 units of masks read by fours
    (4096, 3, 1, False, False, True), (4097, 3, 1, False, False, False),      # 12,288 and 12,291 of masks off 16 bytes
    (21845, 3, 0, False, False, True),                                        # as many heads, aligned
    (1024, 8, 0, True, False, True), (1025, 8, 0, True, False, False),        # 8,192 through a table
    (2048, 8, 0, True, True, True), (2049, 8, 0, True, True, False),          # 16,384, the scan with a prefill's end
])
def test_slot_scan_by_mask_layout(npg, H, pg0, paged, prefill, direct):
    """Which slot scan an encode takes, seen by whether the chained one's workspace was used, and its
    slots, on both sides of each limit."""
    g = torch.Generator(device=DEV).manual_seed(npg + H)
    x = _source(1, npg * 16, H, 64, 0.02, g)
    _say("slot scan by layout", npg, H, pg0, paged, prefill)
    kernels.release_workspaces()
    if paged:
        table = exactkv.PageTable(npg + 1, 1, npg + 1)
        table._free = torch.randperm(npg + 1, generator=torch.Generator().manual_seed(1)).tolist()
        table.add(npg * 16)
        c = exactkv.PagedCompressedKV(table, H, D=64, reserve=0.2)
        pages = torch.tensor(table.pages(0)[:npg], device=DEV)
    else:
        c = exactkv.CompressedKV(1, (pg0 + npg) * 16, H, 64, reserve=0.2)
        pages = torch.arange(pg0, pg0 + npg, device=DEV)
    c.cnt.fill_(5)
    if prefill:
        assert kernels.prefill_pages(x, c, table=table) == int(c.cnt.item())
    elif paged:
        c._encode_pages(x, (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2)), table.block_table, npg)
    else:
        kernels.encode_pages(x, (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2)), c._buf(), 0, pg0, 1, npg)
    assert any(bool(ws.any()) for ws in kernels._SCAN.values()) != direct
    rm, off = (t.view(-1, H)[pages].view(1, npg, H) for t in (c.rowmask, c.rowoff))
    assert int(c._before.item()) == 5
    assert _check_slots(x, rm, off, c.raw, c.cap, 5, int(c.cnt.item())) > 0.01 * npg * 16 * H


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("shift", [0, 2])
@pytest.mark.parametrize("reserve", [0.3, 0.01])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("chained", [True, False])
def test_chained_and_three_launch_scans(D, shift, reserve, paged, chained):
    """The scans above the direct one's limits, contiguous and through a block table, with rows 16- and
    4-byte aligned and a pool with and without room: masks as the direct scan's encode of the same
    pages, slots, raw rows and counter; nothing behind cap."""
    B, npg, H = (2, 1367, 3) if paged else (3, 1367, 3)        # 8,202 and 12,303 units
    g = torch.Generator(device=DEV).manual_seed(D + shift)
    x = _source(B, npg * 16, H, D, 0.05, g, shift)
    st = (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2))
    _say("scans above the limits", D, shift, reserve, paged, chained)
    kernels.release_workspaces()
    c = exactkv.CompressedKV(B, (npg + 1) * 16, H, D, reserve=reserve)
    c.cnt.fill_(5)
    c.raw.fill_(7.0)
    old = c.raw.clone()
    if paged:
        order = torch.randperm(B * (npg + 1), generator=g, device=DEV)[:B * npg].view(B, npg)
        kernels.encode_pages_paged(x, st, c._buf(), order.to(torch.int32), B, npg, chained=chained)
        rm, off = (t.view(-1, H)[order] for t in (c.rowmask, c.rowoff))
    else:
        kernels.encode_pages(x, st, c._buf(), 0, 1, B, npg, chained=chained)
        rm, off = (t[:, 1:] for t in (c.rowmask, c.rowoff))
    assert len(kernels._SCAN) == chained
    one = exactkv.CompressedKV(1, npg * 16, H, D, reserve=0.3)     # a sequence alone: 4,101 units
    for b in range(B):
        kernels.encode_pages(x[b:b + 1], st, one._buf(), 0, 0, 1, npg)
        assert torch.equal(one.rowmask[0], rm[b])
    n = _check_slots(x, rm, off, c.raw, c.cap, 5, int(c.cnt.item()))
    assert int(c._before.item()) == 5 and (5 + n > c.cap) == (reserve < 0.1)
    end = min(5 + n, c.cap)
    assert same_bits(c.raw[:5], old[:5]) and same_bits(c.raw[end:], old[end:])


@pytest.mark.parametrize("B,T,H,D,rate", [(1, 16, 1, 64, 1.0), (2, 160, 3, 128, 0.2), (3, 1040, 5, 256, 0.02),
                                          (1, 4096, 8, 128, 1.0), (4, 2048, 8, 64, 0.0)])
@pytest.mark.parametrize("shift", [0, 2])
def test_store_raw_rows_equals_a_second_encode(B, T, H, D, rate, shift):
    """Raw rows stored after an encode that had no room for them are those of an encode that
    had; the ones past cap are left out."""
    g = torch.Generator(device=DEV).manual_seed(T + H)
    x = torch.empty(B * T * H * D + shift, dtype=torch.bfloat16, device=DEV)[shift:].view(B, T, H, D)
    x.copy_(torch.randn(B, T, H, D, generator=g, device=DEV))
    x[torch.rand(B, T, H, generator=g, device=DEV) < rate, 1] *= 2.0 ** -30
    st = (x.stride(0), 16 * x.stride(1), x.stride(1), x.stride(2))
    c = exactkv.CompressedKV(B, T, H, D, reserve=1.0)
    kernels.encode_pages(x, st, c._buf(), 0, 0, B, T // 16)
    n = int(c.cnt.item())
    for cap in {n, n // 2}:
        buf = dict(c._buf(), cap=cap, raw=torch.zeros(n + 1, D, dtype=torch.bfloat16, device=DEV))
        kernels.store_raw_rows(x, st, buf, 0, 0, B, T // 16)
        assert same_bits(buf["raw"][:cap], c.raw[:cap]) and not bool(buf["raw"][cap:].view(torch.int16).any())
