"""CompressedKV on the GPU: append, page encode, raw-pool growth (reference cache.py:17-158;
reference test tests/test_exactkv.py:81-104), checked against the plain bf16 cache and,
byte for byte, against the CPU model of the protocol (oracle/cache.py)."""
import numpy as np
import pytest
import torch

import exactkv_amd as exactkv
from exactkv_amd import kernels
from oracle import cache as ocache
from tests.conftest import same_bits, u16

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _say(*a):
    print("[case]", *a, flush=True)


def _make(g, B, n, H, D, rate):
    x = torch.randn(B, n, H, D, generator=g).to(torch.bfloat16)
    x[torch.rand(B, n, H, generator=g) < rate, 7] = 1e-30          # forces raw rows
    return x


def _state_equal(c, m, tag):
    for k in ("sm", "code", "base", "rowmask", "rowoff"):
        assert np.array_equal(getattr(c, k).cpu().numpy(), getattr(m, k)), (tag, k)
    assert np.array_equal(u16(c.raw), m.raw), (tag, "raw")
    assert int(c.cnt.item()) == m.cnt and c.cap == m.cap and c.T == m.T and c.grows == m.grows, tag
    assert int(c.state[0].item()) == c.T, tag


@pytest.mark.parametrize("B,H,T0,TS,rate,reserve", [(2, 4, 1000, 1200, 0.1, 0.001), (3, 2, 33, 160, 0.02, 0.01),
                                                    (1, 8, 0, 96, 0.3, 0.0)])
def test_append_and_pool_growth(B, H, T0, TS, rate, reserve):
    g = torch.Generator().manual_seed(2)
    D = 128
    _say("append", B, H, T0, TS, rate, reserve)
    c, r = exactkv.CompressedKV(B, TS, H, D, reserve=reserve), exactkv.BF16KV(B, TS, H, D)
    m = ocache.CacheModel(B, TS, H, D, reserve=reserve)
    x0 = _make(g, B, T0, H, D, rate)
    q = torch.randn(B, 32, D, generator=g).to(torch.bfloat16).to(DEV)
    if T0:
        for b in range(B):
            c.prefill_slot(b, x0[b:b + 1].to(DEV).contiguous())
            r.prefill_slot(b, x0[b:b + 1].to(DEV).contiguous())
            m.prefill_slot(b, u16(x0[b]))
        _state_equal(c, m, "prefill")
    xs = _make(g, B, TS - T0, H, D, rate)
    for t in range(TS - T0):
        xt = xs[:, t].to(DEV).contiguous()
        c.append(xt)
        r.append(xt)
        m.append(u16(xs[:, t]))
        if c.T % 16 == 0:                      # the page encode inside the step never overflows
            assert int(c.cnt.item()) <= c.cap
        exactkv.check_overflow([c])
        m.check_overflow()
        if t % 37 == 0 or t == TS - T0 - 1:
            _state_equal(c, m, t)
            assert same_bits(kernels.decode_to_bf16(c.buffers(), c.T), r.buf[:, :c.T]), t
            assert same_bits(exactkv.decode_attention(q, c, c), exactkv.decode_attention(q, r, r)), t
    assert int(r.state[0].item()) == TS
    assert c.grows > 0 or reserve >= 0.01


def test_prefill_overflow_regrows_and_matches_codec():
    """A prefill whose raw rows exceed the pool: grow, rewind, re-encode (cache.py:77-84)."""
    from oracle import codec as ocodec
    from exactkv_amd import synthetic
    x = synthetic.stress_pages(2, 128, 2, seed=17)
    B, T, H, D = x.shape
    c = exactkv.CompressedKV(B, T, H, D, reserve=0.0)
    for b in range(B):
        c.prefill_slot(b, x[b:b + 1].to(DEV).contiguous())
    ref = ocodec.encode(u16(x))
    n = int(c.cnt.item())
    assert c.grows > 0 and n == ref["raw"].shape[0]
    for k in ("sm", "code", "base", "rowmask", "rowoff"):
        assert np.array_equal(getattr(c, k).cpu().numpy(), ref[k]), k
    assert np.array_equal(u16(c.raw[:n]), ref["raw"])


@pytest.mark.parametrize("B,H,T0,TS,rate", [(600, 8, 13, 48, 0.5), (1040, 8, 9, 48, 0.05)])
def test_append_page_ends_with_many_units_and_raw_rows(B, H, T0, TS, rate):
    """The one-launch append's page end with many (sequence, head) units: 4,800 units with
    half the rows raw (the raw rows, several per thread of the last workgroup, found through
    its LDS table of ranks), and 8,320 units, more than that table holds (each thread moves
    its own units' rows). Byte-equal to the CPU model of the protocol at every page end; the
    arrival counter state[1] is zero after every append."""
    g = torch.Generator().manual_seed(5)
    D = 128
    _say("append many units", B, H, T0, TS, rate)
    c = exactkv.CompressedKV(B, TS, H, D, reserve=0.6)
    m = ocache.CacheModel(B, TS, H, D, reserve=0.6)
    x0 = _make(g, B, T0, H, D, rate)
    x0d = x0.to(DEV)
    for b in range(B):
        c.prefill_slot(b, x0d[b:b + 1].contiguous())
        m.prefill_slot(b, u16(x0[b]))
    xs = _make(g, B, TS - T0, H, D, rate)
    xsd = xs.to(DEV)
    ends = 0
    for t in range(TS - T0):
        c.append(xsd[:, t].contiguous())
        m.append(u16(xs[:, t]))
        exactkv.check_overflow([c])
        m.check_overflow()
        assert int(c.state[1].item()) == 0, t
        if c.T % 16 == 0:
            _state_equal(c, m, t)
            ends += 1
    assert ends >= 2


def _layout(x, kind):
    """x [1, T, H, D] with other strides or alignment, same values."""
    if kind == "heads":                                  # [1, H, T, D] as the attention modules give it
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if kind == "pairs":                                  # rows 4-byte aligned
        flat = torch.empty(x.numel() + 2, dtype=x.dtype, device=x.device)[2:].view(x.shape)
        return flat.copy_(x)
    if kind == "odd":                                    # rows 2-byte aligned (less than a page only)
        flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view(x.shape)
        return flat.copy_(x)
    if kind == "wide":                                   # a slice of more heads and channels
        big = torch.zeros(1, x.shape[1], x.shape[2] + 3, x.shape[3] + 8, dtype=x.dtype, device=x.device)
        big[:, :, 1:1 + x.shape[2], :x.shape[3]] = x
        return big[:, :, 1:1 + x.shape[2], :x.shape[3]]
    return x


@pytest.mark.parametrize("T,H,D,kind,reserve", [
    (1, 8, 128, "plain", 0.5), (15, 3, 64, "odd", 0.5), (16, 8, 128, "plain", 0.5), (17, 5, 256, "heads", 0.5),
    (95, 8, 128, "heads", 0.5), (96, 8, 128, "plain", 0.5), (250, 3, 64, "pairs", 0.5), (333, 2, 128, "wide", 0.5),
    (8191, 9, 64, "heads", 0.3),                         # 4,599 units
    (1000, 8, 128, "heads", 0.0),                        # the pool overflows and grows
])
@pytest.mark.parametrize("paged", [False, True])
def test_prefill_in_one_call_equals_its_parts(T, H, D, kind, reserve, paged, monkeypatch):
    """prefill_slot's one call (pages, open page, token count, counter) leaves every array as
    the encoder, the page opening and the row copy leave it one after the other."""
    from exactkv_amd import cache as mcache, paged as mpaged
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(1, T, H, D, generator=g, device=DEV).bfloat16()
    x[0, torch.rand(T, H, generator=g, device=DEV) < 0.1, 5] *= 2.0 ** -30
    x = _layout(x, kind)
    got = []
    for parts in (False, True):
        if parts:
            monkeypatch.setattr(mcache, "prefill_ready", lambda *a: False)
            monkeypatch.setattr(mpaged, "prefill_ready", lambda *a: False)
        if paged:
            table = exactkv.PageTable(3 * (T // 16 + 2), 3, T // 16 + (1 if T % 16 else 0) or 1)
            c = exactkv.PagedCompressedKV(table, H, D=D, reserve=reserve)
            for other in (40, T):
                c.prefill(table.add(min(other, T)), x[:, :min(other, T)])
        else:
            c = exactkv.CompressedKV(2, -(-T // 16) * 16, H, D, reserve=reserve)
            c.prefill_slot(0, x)
            c.prefill_slot(1, x.flip(1) if kind == "plain" else x)
            got.append((c.T, c.state))
        got.append((c.cap, c.grows, c.sm, c.code, c.base, c.rowmask, c.rowoff, c.cnt, c._before,
                    c.raw.view(torch.int16)))
    half = len(got) // 2
    for a, b in zip(sum(got[:half], ()), sum(got[half:], ())):
        assert torch.equal(a, b) if isinstance(a, torch.Tensor) else a == b


def test_appends_follow_moved_buffers():
    """Every append and prefill reads the addresses of the cache's arrays anew: storage that moves
    under the same tensor objects is written where it is now."""
    g = torch.Generator().manual_seed(3)
    B, H, D, T0 = 2, 4, 128, 20
    x = _make(g, B, 64, H, D, 0.1).to(DEV)
    a, c = exactkv.CompressedKV(B, 64, H, D, reserve=0.6), exactkv.CompressedKV(B, 64, H, D, reserve=0.6)
    for k in (a, c):
        for b in range(B):
            k.prefill_slot(b, x[b:b + 1, :T0].contiguous())
        k.append(x[:, T0].contiguous())
    old = {n: getattr(c, n).data for n in ("sm", "code", "base", "rowmask", "rowoff", "raw", "cnt", "state")}
    was = {n: t.clone() for n, t in old.items()}
    for n in old:
        getattr(c, n).data = old[n].clone()
    for t in range(T0 + 1, 40):
        for k in (a, c):
            k.append(x[:, t].contiguous())
        exactkv.check_overflow([a, c])
    for n in old:
        assert torch.equal(getattr(a, n), getattr(c, n)), n
        assert torch.equal(old[n], was[n]), n


@pytest.mark.parametrize("T", [7, 40])
def test_prefill_takes_any_index_type(T):
    """Slots as Python ints, numpy ints and one-element tensors alike."""
    g = torch.Generator().manual_seed(4)
    x = _make(g, 3, T, 2, 128, 0.1).to(DEV)
    a, c = exactkv.CompressedKV(3, 64, 2, 128, reserve=0.6), exactkv.CompressedKV(3, 64, 2, 128, reserve=0.6)
    for b, same in enumerate((0, np.int64(1), torch.tensor(2))):
        a.prefill_slot(b, x[b:b + 1])
        c.prefill_slot(same, x[b:b + 1])
    for n in ("sm", "code", "base", "rowmask", "rowoff", "raw", "cnt", "state"):
        assert torch.equal(getattr(a, n), getattr(c, n)), n


@pytest.mark.parametrize("T", [7, 40])
def test_prefill_refuses_a_truth_value_as_slot(T):
    c = exactkv.CompressedKV(3, 64, 2, 128, reserve=0.6)
    with pytest.raises(RuntimeError):
        c.prefill_slot(True, torch.ones(1, T, 2, 128, dtype=torch.bfloat16, device=DEV))


@pytest.mark.parametrize("T,H,D,kind", [
    (T, H, D, kind) for T, H, D in ((1, 1, 64), (15, 128, 256), (31, 128, 256), (31, 33, 128), (20, 64, 128), (31, 70, 64))
    for kind in ("plain", "heads", "pairs", "odd") if kind != "odd" or T < 16])    # full pages need 4-byte aligned rows
@pytest.mark.parametrize("paged", [False, True])
def test_prefill_open_rows(T, H, D, kind, paged):
    """A prompt's last rows in the open page, in 16-, 4- and 2-byte pieces, a few and more than the
    block has in flight at once."""
    g = torch.Generator(device=DEV).manual_seed(T + H)
    x = torch.randn(1, T, H, D, generator=g, device=DEV).bfloat16()
    if paged:
        table = exactkv.PageTable(8, 2, 3)
        c = exactkv.PagedCompressedKV(table, H, D=D, reserve=3.0)
        c.prefill(table.add(17), torch.ones(1, 17, H, D, dtype=torch.bfloat16, device=DEV))
        slot = table.add(T)
        first = c.cap + slot * H * 16
    else:
        slot, c = 1, exactkv.CompressedKV(2, 48, H, D, reserve=3.0)
        first = c.cap + H * 16
    before = c.raw.clone()
    (c.prefill if paged else c.prefill_slot)(slot, _layout(x, kind))
    assert c.grows == 0
    got = kernels.decode_to_bf16(c.buffers(), T, block_table=table.block_table if paged else None)
    assert same_bits(got[slot], x[0])
    rows = c.raw[first:first + H * 16].view(H, 16, D)
    assert same_bits(rows[:, :T % 16], x[0, T - T % 16:].transpose(0, 1))
    rows[:, :T % 16] = before[first:first + H * 16].view(H, 16, D)[:, :T % 16]
    assert same_bits(c.raw[c.cap:], before[c.cap:])        # no other row


@pytest.mark.parametrize("B,H,D", [(1, 1, 64), (2, 8, 128), (9, 8, 128), (3, 5, 256), (300, 4, 64)])
@pytest.mark.parametrize("offset,pitch", [(0, 0), (2, 0), (0, 2), (4, 4), (0, 6)])
@pytest.mark.parametrize("paged", [False, True])
def test_append_row_alignment(B, H, D, offset, pitch, paged):
    """Token rows inside wider ones, 16-, 8- and 4-byte aligned, one block of units and more: after
    every append the cache decodes to the tokens given so far."""
    g = torch.Generator(device=DEV).manual_seed(B + D + offset)
    T0, N = 10, 9                                          # appends before, at and after a page end
    x = torch.randn(B, T0 + N, H, D, generator=g, device=DEV).bfloat16()
    x[torch.rand(B, T0 + N, H, generator=g, device=DEV) < 0.1, 5] *= 2.0 ** -30
    if paged:
        table = exactkv.PageTable(2 * B, B, 2)
        c = exactkv.PagedCompressedKV(table, H, D=D, reserve=1.0)
    else:
        table, c = None, exactkv.CompressedKV(B, 32, H, D, reserve=1.0)
    for b in range(B):
        c.prefill_slot(b if table is None else table.add(T0), x[b:b + 1, :T0].contiguous())
    for t in range(T0, T0 + N):
        flat = torch.full((B * H * (D + pitch) + offset,), 3.0, dtype=torch.bfloat16, device=DEV)
        row = flat[offset:].view(B, H, D + pitch)[..., :D]
        row.copy_(x[:, t])
        if paged:
            table.begin_step()
        c.append(row)
        exactkv.check_overflow([c])
        got = kernels.decode_to_bf16(c.buffers(), t + 1, block_table=table.block_table if paged else None)
        assert same_bits(got, x[:, :t + 1]), t


def test_misaligned_cache_arrays_are_refused():
    """array_ptrs names what is at fault: an array off 16 bytes, a word off 4, a tensor not on the GPU."""
    buf = torch.zeros(64, dtype=torch.uint8, device=DEV)
    word = torch.zeros(1, dtype=torch.int32, device=DEV)
    assert kernels.array_ptrs((buf, buf[16:]), (word,)) == [buf.data_ptr(), buf.data_ptr() + 16, word.data_ptr()]
    for arrays, words in (((buf[8:],), (word,)), ((buf,), (buf[2:],)), ((buf.cpu(),), (word,))):
        with pytest.raises(ValueError):
            kernels.array_ptrs(arrays, words)


@pytest.mark.parametrize("T,H", [(1, 8), (15, 2), (16, 1), (1040, 1), (1040, 8), (65536, 16), (32769, 33)])
@pytest.mark.parametrize("paged", [False, True])
def test_prefill_returns_the_counter(T, H, paged):
    """The counter that a prefill's last block (without full pages, or above the direct scan's limit,
    its last launch) gives the host, call after call: one block, several, 257 and a launch of its own."""
    from exactkv_amd import kernels as k
    g = torch.Generator(device=DEV).manual_seed(T)
    x = (1 + torch.rand(1, T, H, 64, generator=g, device=DEV)).bfloat16()        # no raw rows by chance
    raw = torch.rand(T, H, generator=g, device=DEV) < 0.02
    x[0, raw, 9] = 1e-30
    full = T - T % 16
    n = int(raw[:full].sum())
    pages = -(-(T + 1) // 16)
    if paged:
        table = exactkv.PageTable(pages, 1, pages)
        table.add(T)
        c = exactkv.PagedCompressedKV(table, H, D=64, reserve=0.2)
    else:
        table, c = None, exactkv.CompressedKV(1, 16 * pages, H, 64, reserve=0.2)
    word = c._arrivals[0] if paged else c.state[1]
    for i in range(1, 4):
        assert k.prefill_pages(x, c, table=table) == i * n == int(c.cnt.item())
        assert int(word.item()) == 0
