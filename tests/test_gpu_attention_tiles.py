"""Attention over more than 512 rows. Short lists run item by item; lists of more than
32768 items and groups in tiles of sixteen rows that share their pages, as fp32 MFMAs, and
what shares nothing item by item (stride_amd/csrc/tc_aux.hip). Bit for bit against the
oracle, bf16 and fp32 KV, either side of that line, at the edges of the tile form:
sequences that end inside a tile, positions around page ends, tiles of one row, rows that
share nothing, rows of two sequences in turn; then lists other than the engine's, whose
unlisted pages come from scratch, and values (infinities, NaN, -0) that must not reach
rows that do not see them."""
import numpy as np
import pytest
import torch

from stride_amd import exact as E
from stride_amd import harness, layout, tc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def bf16_bits(a):
    return (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)


def prompts(*spans):
    """(slots, positions) of consecutive rows: one (first, last + 1) span per sequence."""
    slots = [s for s, (a, b) in enumerate(spans) for _ in range(a, b)]
    return np.array(slots, np.int32), np.array([p for a, b in spans for p in range(a, b)], np.int32)


def make(seed, slots, pos, n_kv, hd, page, k=None, v=None):
    rng = np.random.default_rng(seed)
    m, cap, ns = len(slots), int(pos.max()) + 1, int(slots.max()) + 1
    q = rng.standard_normal((m, n_kv * 4, hd)).astype(np.float32)
    k = bf16_bits(rng.standard_normal((ns, n_kv, cap, hd))) if k is None else k
    v = bf16_bits(rng.standard_normal((ns, n_kv, cap, hd))) if v is None else v
    kv = harness.PagedKv.create(ns, cap, n_kv, hd, 1, page, DEV, shuffle_seed=seed + 1)
    kv.fill_dense(0, 0, torch.from_numpy(k.view(np.int16)))
    kv.fill_dense(0, 1, torch.from_numpy(v.view(np.int16)))
    return q, k, v, kv, -(-cap // 64)


def run(q, kv, slots, pos, n_kv, hd, pages, **kw):
    out = harness.attention(torch.from_numpy(q.reshape(len(slots), -1)).to(DEV), kv, torch.from_numpy(slots).to(DEV),
                            torch.from_numpy(pos).to(DEV), n_kv, hd, hd ** -0.5, max_pages=pages, **kw)
    torch.cuda.synchronize()
    return layout.untile_lanes(out.cpu(), len(slots)).numpy().view(np.uint16)


def interleaved(a, b):
    s, p = prompts(a, b)
    order = np.argsort(p, kind="stable")
    return s[order], p[order]


CASES = [prompts((0, 513)), prompts((0, 250), (3, 210), (190, 300)),                # sequences ending inside tiles
         prompts(*[(40 + i, 90 + i) for i in range(11)]),                           # 50 rows each: three in a tile
         interleaved((0, 300), (1, 290)),                                           # two sequences in turn
         (np.arange(530, dtype=np.int32) % 37, (np.arange(530) * 7 % 200).astype(np.int32)),  # nothing shared
         prompts((100, 612), (0, 1))]                                               # a tile of one row


# The same forms past the line (8 groups: more than 4096 items).
LONG = [prompts((300, 900)), prompts((500, 750), (3, 210), (600, 803)),
        prompts(*[(500 + 7 * i, 550 + 7 * i) for i in range(11)]),
        interleaved((300, 620), (310, 600)),
        (np.arange(530, dtype=np.int32) % 37, (500 + np.arange(530) * 7 % 200).astype(np.int32)),
        (np.zeros(530, np.int32), (500 + np.arange(530) * 37 % 400).astype(np.int32)),  # one sequence, far apart
        prompts((420, 932), (0, 1))]


def item_list(pos):
    return [(j, c) for j in range(len(pos)) for c in range((pos[j] >> 6) + 1)]


class Long:
    """A call on inputs of its own, in both kinds of KV (fp32 of the same values). One of
    all rows has to take the tiles."""

    def __init__(self, seed, slots, pos, hd, page, n_kv=8):
        rng = np.random.default_rng(seed)
        m, ns = len(slots), int(slots.max()) + 1
        self.slots, self.pos, self.hd, self.page, self.n_kv = slots, pos, hd, page, n_kv
        self.pages = int(pos.max()) // 64 + 1
        self.blocks = -(-(int(pos.max()) + 1) // page)
        self.q = rng.standard_normal((m, n_kv * 4, hd)).astype(np.float32)
        self.k, self.v = (bf16_bits(rng.standard_normal((ns, n_kv, self.blocks * page, hd))) for _ in range(2))
        self.order = rng.permutation(ns * self.blocks).astype(np.int32).reshape(ns, self.blocks)
        self.items = item_list(pos)

    def want(self, exact):
        return exact.tc_attention(self.q, self.k, self.v, self.slots, self.pos, self.hd ** -0.5)

    def run(self, fp32, lists=None, rows=None):
        """Output [row][head * hd + d], of the rows `rows`, after a call for each list."""
        lo, hi = rows or (0, len(self.pos))
        m, n_kv, hd, page = hi - lo, self.n_kv, self.hd, self.page
        lists = lists or [[(j - lo, c) for j, c in self.items if lo <= j < hi]]
        for items in lists if rows is None else []:
            assert len(items) * n_kv > 32768 and 128 <= m <= 8192, "not a list that the tiles take"
        d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
        blocked = lambda a: d(a.view(np.int16)).view(-1, n_kv, self.blocks, page, hd).transpose(1, 2)  # noqa: E731
        arena = torch.empty((self.order.size, 2, n_kv, page, hd), dtype=torch.int16, device=DEV)
        arena[d(self.order).long(), 0], arena[d(self.order).long(), 1] = blocked(self.k), blocked(self.v)
        if fp32:
            arena = arena.view(torch.bfloat16).float()
        table, q, slots, pos = d(self.order), d(self.q[lo:hi]), d(self.slots[lo:hi]), d(self.pos[lo:hi])
        scratch = torch.zeros(m * n_kv * self.pages * (8 + 4 * hd), device=DEV)
        cols, block = n_kv * 4 * hd, arena[0].numel()
        if fp32:
            out, l = torch.zeros((cols, E.lane_shape(m)[2]), device=DEV), E.lanes(m)
        else:
            out, l = torch.zeros(((m + 15) // 16, cols // 16, 16, 16), dtype=torch.int16, device=DEV), tc.lanes(m)
        for items in lists:
            it = d(np.array(items, np.int32).reshape(-1))
            p = tc.AttentionParams()
            p.l, p.q, p.q_stride, p.out, p.out_cols = l, tc.ptr(q), cols, tc.ptr(out), cols
            p.kv = tc.KvRef(tc.ptr(arena), tc.ptr(table), block, block, block // 2, page * hd, self.blocks, hd)
            p.row_slot, p.row_pos, p.items, p.item_count = tc.ptr(slots), tc.ptr(pos), tc.ptr(it), len(items)
            p.scratch, p.max_pages, p.rec_floats = tc.ptr(scratch), self.pages, 8 + 4 * hd
            p.layer, p.n_kv, p.n_q, p.head_dim, p.scale = 0, n_kv, 4, hd, hd ** -0.5
            (E.k_attention if fp32 else tc.tc_attention)(p)
        torch.cuda.synchronize()
        if fp32:
            return out[:, :m].T.contiguous().cpu().numpy()
        return layout.untile_lanes(out.cpu(), m).numpy().view(np.uint16)


_prompt = {}


def long_prompt(exact, hd):
    """One prompt's last 800 rows of 1100, and the oracle's output."""
    if hd not in _prompt:
        a = Long(hd, *prompts((300, 1100)), hd, 16)
        _prompt[hd] = a, a.want(exact)
    return _prompt[hd]


def to_bf16(a):
    """fp32 to bf16 bits, nearest even."""
    return torch.from_numpy(a).bfloat16().view(torch.int16).numpy().view(np.uint16)


@pytest.mark.parametrize("case", range(len(LONG)))
@pytest.mark.parametrize("hd,page", [(64, 16), (128, 64), (32, 32)])
def test_long_lists(exact, case, hd, page):
    print("attention tiles, long list", case, hd, page, flush=True)
    a = Long(case + hd, *LONG[case], hd, page)
    want = a.want(exact)
    assert np.array_equal(a.run(False), want)
    whole = a.run(True)
    assert np.array_equal(to_bf16(whole), want)
    # all bits of the fp32 output: the same rows in short calls, which take one kernel
    m = len(a.pos)
    parts = np.concatenate([a.run(True, rows=(lo, min(lo + 400, m))) for lo in range(0, m, 400)])
    assert np.array_equal(whole.view(np.uint32), parts.view(np.uint32))


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("n_kv,hd,page", [(2, 64, 16), (1, 128, 64), (1, 32, 32)])
def test_short_lists_fp32(exact, case, n_kv, hd, page):
    """The page + combine pair and the one-kernel form over fp32 KV."""
    print("attention, short list, fp32", case, n_kv, hd, page, flush=True)
    a = Long(case + hd, *CASES[case], hd, page, n_kv)
    m = len(a.pos)
    assert m > 512 and len(a.items) * n_kv <= 32768
    pair = a.run(True, rows=(0, m))
    assert np.array_equal(to_bf16(pair), a.want(exact))
    parts = np.concatenate([a.run(True, rows=(lo, min(lo + 400, m))) for lo in range(0, m, 400)])
    assert np.array_equal(pair.view(np.uint32), parts.view(np.uint32))


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("form", ["alternate items", "alternate tiles", "reversed", "two rows swapped"])
@pytest.mark.parametrize("hd", [64, 128])
def test_long_lists_not_the_engines(exact, form, fp32, hd):
    """Lists that do not hold each tile's items where the engine's does: they are summed
    item by item, and a call's unlisted pages come from scratch."""
    print("attention tiles, long lists not the engine's", form, fp32, hd, flush=True)
    a, want = long_prompt(exact, hd)
    if form == "alternate items":
        lists = [a.items[::2], a.items[1::2]]
    elif form == "alternate tiles":
        lists = [[(j, c) for j, c in a.items if j // 16 % 2 == half] for half in (0, 1)]
    elif form == "reversed":
        lists = [a.items[::-1]]
    else:
        order = [{100: 101, 101: 100}.get(j, j) for j in range(len(a.pos))]
        lists = [[(j, c) for j in order for c in range((a.pos[j] >> 6) + 1)]]
    got = a.run(fp32, lists)
    assert np.array_equal(to_bf16(got) if fp32 else got, want)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("hd", [32, 64, 128])
def test_unseen_positions_stay_out_of_tiles(exact, fp32, hd):
    """As test_unseen_positions_stay_out, past the line."""
    print("attention tiles, long list, unseen values", fp32, hd, flush=True)
    a = Long(6, *prompts((0, 900)), hd, 16)
    a.v[0, :, ::3] = 0x8000  # -0
    want = a.run(fp32)
    assert np.array_equal(to_bf16(want) if fp32 else want, a.want(exact))
    for at, bits in ((70, 0x7F80), (201, 0xFF80), (333, 0x7FC0), (450, 0x7F80), (777, 0xFF80)):
        a.v[0, :, at, ::5] = bits
        a.k[0, :, at, 1::7] = bits
    got = a.run(fp32)
    u = np.uint32 if fp32 else np.uint16
    assert np.array_equal(got[:70].view(u), want[:70].view(u))
    assert not np.array_equal(got[70].view(u), want[70].view(u))
    # rows that see them: as the one-kernel form gives them (NaN where it does)
    parts = np.concatenate([a.run(fp32, rows=(lo, lo + 300)) for lo in (0, 300, 600)])
    f = lambda x: x if fp32 else (x.astype(np.uint32) << 16).view(np.float32)  # noqa: E731
    nan = np.isnan(f(got))
    assert nan.any() and np.array_equal(nan, np.isnan(f(parts)))
    assert np.array_equal(got.view(u)[~nan], parts.view(u)[~nan])


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("n_kv,hd,page", [(2, 64, 16), (1, 128, 64), (1, 32, 32)])
def test_tiles(exact, case, n_kv, hd, page):
    print("attention tiles", case, n_kv, hd, page, flush=True)
    slots, pos = CASES[case]
    q, k, v, kv, pages = make(case + hd, slots, pos, n_kv, hd, page)
    got = run(q, kv, slots, pos, n_kv, hd, pages)
    assert np.array_equal(got, exact.tc_attention(q, k, v, slots, pos, hd ** -0.5))


def test_partial_lists(exact):
    """Listed pages are summed and stored, the others combined from scratch: two calls
    that list a page each in turn give the whole list's bits, for tiles that share."""
    print("attention tiles, partial lists", flush=True)
    slots, pos = prompts((60, 610))
    q, k, v, kv, pages = make(5, slots, pos, 1, 64, 16)
    items = [(j, c) for j in range(len(pos)) for c in range((pos[j] >> 6) + 1)]
    scratch = torch.zeros(len(pos) * pages * 264, dtype=torch.float32, device=DEV)
    for half in (0, 1):
        part = torch.tensor([it for n, it in enumerate(items) if n % 2 == half], dtype=torch.int32, device=DEV).reshape(-1)
        got = run(q, kv, slots, pos, 1, 64, pages, items=part, scratch=scratch)
    assert np.array_equal(got, exact.tc_attention(q, k, v, slots, pos, 0.125))


def test_unseen_positions_stay_out(exact):
    """A row's result does not depend on later positions, whatever they hold, nor on
    the sign of zeros: rows before a non-finite position equal the same rows without it."""
    print("attention tiles, unseen values", flush=True)
    slots, pos = prompts((0, 520))
    q, k, v, kv, pages = make(6, slots, pos, 1, 64, 16)
    v[0, 0, ::3] = 0x8000  # -0
    k2, v2 = k.copy(), v.copy()
    for at, bits in ((70, 0x7F80), (201, 0xFF80), (333, 0x7FC0), (450, 0x7F80)):
        v2[0, 0, at, ::5] = bits
        k2[0, 0, at, 1::7] = bits
    want = run(q, make(6, slots, pos, 1, 64, 16, k, v)[3], slots, pos, 1, 64, pages)
    assert np.array_equal(want, exact.tc_attention(q, k, v, slots, pos, 0.125))
    got = run(q, make(6, slots, pos, 1, 64, 16, k2, v2)[3], slots, pos, 1, 64, pages)
    assert np.array_equal(got[:70], want[:70])
    assert not np.array_equal(got[70], want[70])
