"""The launches behind the native half of the Python launchers, at the sizes where they can go
wrong: row blocks of one row up to several workgroups, fp32 and strided sources, ring and whole
history; uploads around the block that one launch carries; group lists longer than one launch."""
import pytest
import torch

import oracle.ommx_oracle as O
from open_ommx_serve_amd.attention import CanonicalKVStore, MultiSeqKVPool, WindowSpec, _hip, ommx_pack_kv_canonical_block
from open_ommx_serve_amd.attention.kv_store_ops import ring_slot
from open_ommx_serve_amd.attention.pack import alloc_planes, store_pack_into, store_table

pytestmark = pytest.mark.gpu
DEV = "cuda"
RECIPE = dict(outliers_per_vector=6, outlier_repr="bitmap", use_pow2=True)


def _block(T, H, D, dtype, seed, strided=False):
    g = torch.Generator(device=DEV).manual_seed(seed)
    t = torch.randn(T, H, 2 * D if strided else D, generator=g, device=DEV).to(dtype)
    return t[..., D // 2:D // 2 + D] if strided else t


@pytest.mark.parametrize("ring", [False, True])
@pytest.mark.parametrize("T", [1, 7, 8, 9, 39, 71, 72, 73, 200, 1033])
@pytest.mark.parametrize("dtype,strided", [(torch.bfloat16, False), (torch.float32, False), (torch.bfloat16, True)])
def test_block_rows_reach_their_history_slots(ring, T, dtype, strided):
    H, D, win = 2, 128, WindowSpec()
    pool = MultiSeqKVPool(D, H, 3, 1100, window=win, device=DEV, kv_ring=ring, **RECIPE)
    K, V = _block(T, H, D, dtype, 1, strided), _block(T, H, D, dtype, 2, strided)
    assert pool.append_block(1, K, V) == win.num_groups(T)
    live = range(T) if not ring else [*range(min(8, T)), *range(min(T, max(8, win.boundary(T) - 32)), T)]
    for p in live:
        slot = ring_slot(p, pool._ring_sink, pool._ring_rec) if ring else p
        assert torch.equal(pool.k_hist[1, slot], K[p].to(torch.bfloat16)), p
        assert torch.equal(pool.v_hist[1, slot], V[p].to(torch.bfloat16)), p
    assert not pool.k_hist[0].any() and not pool.k_hist[2].any()
    if win.num_groups(T):
        edge = win.boundary(T)
        want = O.pack_kv(K[8:edge].to(torch.bfloat16).cpu(), V[8:edge].to(torch.bfloat16).cpu())
        got = pool.request_planes(1)
        for n in ("k_base", "k_scale", "k_obmp", "k_oval", "v_main", "v_scale"):
            assert torch.equal(got[n].cpu(), want[n]), n


@pytest.mark.parametrize("ring", [False, True])
@pytest.mark.parametrize("recent,D,gt", [(32600, 64, 32), (32800, 64, 32), (70000, 128, 32), (140000, 64, 32), (70000, 64, 128)])
def test_one_group_under_a_long_window(ring, recent, D, gt):
    """The rows that are copied along with a single group take a slice of the grid each: from as many slices on as a grid
    does not hold, they are copied by a launch of their own."""
    T, win = 8 + gt + recent, WindowSpec(recent_window=recent, group_tokens=gt)
    recipe = dict(RECIPE, outlier_select="signed", kv_outlier_map=True)
    if gt != 32:
        recipe.update(outlier_repr="relidx7", group_channels=gt // 2)
    assert win.num_groups(T) == 1
    pool = MultiSeqKVPool(D, 1, 1, T + 100, window=win, device=DEV, kv_ring=ring, **recipe)
    K, V = _block(T, 1, D, torch.bfloat16, 21), _block(T, 1, D, torch.bfloat16, 22)
    assert pool.append_block(0, K, V) == 1
    at = [ring_slot(p, pool._ring_sink, pool._ring_rec) if ring else p for p in range(T)]
    assert torch.equal(pool.k_hist[0, at], K) and torch.equal(pool.v_hist[0, at], V)
    want = ommx_pack_kv_canonical_block(K[8:8 + gt], V[8:8 + gt], page_size=16, device=DEV, group_tokens=gt, **recipe)
    got = pool.request_planes(0)
    for n in ("k_base", "k_scale", "k_oval", "v_main", "v_scale"):
        assert torch.equal(got[n], want[n]), n


@pytest.mark.parametrize("n", [1, 479, 480, 481, 960, 961, 2000])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_uploads_of_one_launch_and_more(n, dtype):
    values = [(-1) ** i * (i * 7919 % 2000003) for i in range(n)]
    out = torch.full((n + 1,), -5, dtype=dtype, device=DEV)
    assert _hip.host().upload(out[:n], values)
    assert out.tolist() == values + [-5]
    assert not _hip.host().upload(out, values)              # a list of another length is refused


@pytest.mark.parametrize("ring", [False, True])
def test_groups_of_many_requests_complete_in_one_step(ring):
    """490 requests complete a group in the same step: the group list takes two launches."""
    B, H, D, win = 490, 1, 32, WindowSpec()
    pool = MultiSeqKVPool(D, H, B, 80, window=win, device=DEV, kv_ring=ring, **RECIPE)
    K, V = _block(73 * B, H, D, torch.bfloat16, 3).view(73, B, H, D), _block(73 * B, H, D, torch.bfloat16, 4).view(73, B, H, D)
    for r in range(B):
        pool.append_block(r, K[:71, r], V[:71, r])
    assert pool.append_decode_batched(range(B), K[71], V[71]) == B
    for r in (0, 1, 479, 480, 489):
        want = O.pack_kv(K[8:40, r].cpu(), V[8:40, r].cpu())
        got = pool.request_planes(r)
        for n in ("k_base", "k_scale", "k_obmp", "k_oval", "v_main", "v_scale"):
            assert torch.equal(got[n].cpu(), want[n]), (r, n)


@pytest.mark.parametrize("gt,ps", [(32, 16), (32, 32), (32, 64), (64, 16), (128, 256), (16, 64)])
@pytest.mark.parametrize("groups", [2, 6, 34])
def test_a_block_carries_identity_tables(gt, ps, groups):
    """Each store kernel writes the tables of its block: pages shorter and longer than a group."""
    T, gc = 2 * gt * ps // 16 * groups, 32 if gt < 64 else gt
    K, V = _block(T, 2, 128, torch.bfloat16, 5), _block(T, 2, 128, torch.bfloat16, 6)
    out = ommx_pack_kv_canonical_block(K, V, outliers_per_vector=6, page_size=ps, device=DEV, outlier_select="signed",
                                       use_pow2=True, group_tokens=gt, group_channels=gc)
    assert torch.equal(out["req_to_token"], torch.arange(T // ps, dtype=torch.int32, device=DEV)[None])
    assert torch.equal(out["req_to_group"], torch.arange(T // gt, dtype=torch.int32, device=DEV)[None])


@pytest.mark.parametrize("recipe", [
    dict(outliers_per_vector=6, outlier_repr="bitmap"),
    dict(outliers_per_vector=6, outlier_repr="relidx7", group_tokens=64, group_channels=64, kv_outlier_map=False),
    dict(outliers_per_vector=4, outlier_repr="relidx7", group_tokens=128, group_channels=32)])
@pytest.mark.parametrize("H", [1, 3, 8])
@pytest.mark.parametrize("extra", [0, 1, 31, 127])
def test_live_rows_ride_along_with_the_groups(recipe, H, extra):
    """One launch of each store kernel packs the groups and copies the ring's rows: the same as two launches."""
    recipe = dict(recipe)
    gt = recipe.pop("group_tokens", 32)
    win = WindowSpec(page_size=16, group_tokens=gt)
    T = 40 + 3 * gt + extra
    K, V = _block(T, H, 128, torch.bfloat16, 7), _block(T, H, 128, torch.bfloat16, 8)
    pools = [MultiSeqKVPool(128, H, 2, T, window=win, device=DEV, kv_ring=True, use_pow2=True, **recipe) for _ in range(2)]
    for p in pools:
        for t in p.pool_planes().values():
            if torch.is_tensor(t) and t.dtype != torch.int32:
                t.view(torch.uint8).zero_()
    one, two = pools
    launches = []
    inner = two._pack_block_into_pool
    two._pack_block_into_pool = lambda *a, live=None, **kw: launches.append(inner(*a, **kw))       # without the rows
    assert one.append_block(1, K, V) == two.append_block(1, K, V) == win.num_groups(T) > 0
    assert launches == [False]
    assert torch.equal(one.k_hist, two.k_hist) and torch.equal(one.v_hist, two.v_hist)
    assert one.k_hist[1].any() and not one.k_hist[0].any()
    for n, t in one.pool_planes().items():
        if torch.is_tensor(t):
            assert torch.equal(t.view(torch.uint8), two.pool_planes()[n].view(torch.uint8)), n


@pytest.mark.parametrize("ring", [False, True])
def test_a_block_may_come_out_of_the_history_it_goes_to(ring):
    """Rows that overlap the slots they are written to: as from a copy of them."""
    H, D, T = 2, 128, 150
    pools = [MultiSeqKVPool(D, H, 2, 160, device=DEV, kv_ring=ring, **RECIPE) for _ in range(2)]
    for p in pools:
        for h, seed in ((p.k_hist, 9), (p.v_hist, 10)):
            h.copy_(_block(h.shape[0] * h.shape[1], H, D, torch.bfloat16, seed).view(h.shape))
    first = pools[0].k_hist.shape[1] - 60                    # from the first request's slots into the second's
    for p, own in zip(pools, (True, False)):
        K, V = (h.view(-1, H, D)[first:first + T] for h in (p.k_hist, p.v_hist))
        p.append_block(1, K if own else K.clone(), V if own else V.clone())
    for name in ("k_hist", "v_hist", "k_base", "k_scale", "v_main", "v_scale"):
        assert torch.equal(getattr(pools[0], name), getattr(pools[1], name)), name


def test_error_words_nobody_asks_for_stay_until_the_kernel_is_through():
    """The block goes back to torch's pinned allocator, which must not hand it on while a kernel may write to it."""
    K, V = _block(128, 2, 128, torch.bfloat16, 11), _block(128, 2, 128, torch.bfloat16, 12)

    def launch():
        return _hip.host().pack_block(K, V, 16, True, store_table(K.device), 6, 32, 32, "bitmap", "signed", True, True, "i2")[0]

    held = [launch() for _ in range(20)]                     # (more than are kept idle)
    torch.cuda.synchronize()
    torch.cuda._sleep(20_000_000)                            # some ten milliseconds
    flags = launch()
    at, words = flags.data_ptr(), flags.numel()
    del flags
    others = [torch.empty(words, dtype=torch.int32, pin_memory=True) for _ in range(4)]
    assert not torch.cuda.current_stream().query()           # (still asleep: the test means something)
    assert at not in [t.data_ptr() for t in others]
    torch.cuda.synchronize()
    del held


@pytest.mark.parametrize("H,D,kw,lens", [
    (8, 128, {}, [97, 1, 530, 39, 40, 71, 72, 73]), (1, 128, dict(outlier_repr="relidx7"), [700, 8, 104]),
    (4, 64, {}, [72, 71]), (2, 128, dict(group_tokens=64, group_channels=64, outlier_repr="relidx7", kv_outlier_map=False), [300, 111]),
    (3, 64, {}, [41, 200, 1, 1]), (2, 128, dict(outliers_per_vector=0), [260, 90]),
])
def test_prompts_of_several_requests_in_two_launches(H, D, kw, lens):
    """Every row and group where one append_block per request puts them: bit for bit, whatever the slots, from rows of a
    wider tensor that do not start at its first row; what the launches do not take is refused and leaves the pool alone."""
    kw = dict(kw)
    win = WindowSpec(group_tokens=kw.pop("group_tokens", 32))
    kw.setdefault("group_channels", min(32, D))
    g = torch.Generator(device="cuda").manual_seed(3)
    slots = [(5 * i + 2) % (len(lens) + 3) for i in range(len(lens))] if (len(lens) + 3) % 5 else list(range(len(lens)))[::-1]
    pools = [MultiSeqKVPool(D, H, len(lens) + 3, 720, window=win, device="cuda", **{"outlier_repr": "bitmap", **kw}) for _ in range(3)]
    for p in pools:
        for t in (p.k_hist, p.v_hist, *(v for k, v in p.pool_planes().items() if torch.is_tensor(v) and not k.startswith("req_"))):
            t.zero_()
    starts = [5]
    for n in lens:
        starts.append(starts[-1] + n)
    wide = torch.randn(starts[-1] + 3, 2 * H, D, generator=g, device="cuda").to(torch.bfloat16)
    K, V = wide[:, :H], wide[:, H:]
    assert pools[0].append_prompts(slots, starts, K, V)
    for r, a, b in zip(slots, starts, starts[1:]):
        pools[1].append_block(r, K[a:b], V[a:b])
    assert pools[0].seq_len == pools[1].seq_len and pools[0].packed_groups == pools[1].packed_groups
    for name, t in pools[0].pool_planes().items():
        if torch.is_tensor(t):
            assert torch.equal(t.view(torch.uint8), pools[1].pool_planes()[name].view(torch.uint8)), name
    assert torch.equal(pools[0].k_hist, pools[1].k_hist) and torch.equal(pools[0].v_hist, pools[1].v_hist)
    pools[0].check_errors()
    before = [list(pools[2].seq_len), pools[2].k_hist.clone()]
    assert not pools[2].append_prompts(slots, starts, K.float(), V.float())
    assert not pools[2].append_prompts(slots, [0, *[x + 721 for x in starts[1:]]], K, V)
    assert not pools[2].append_prompts([slots[0]] * len(slots), starts, K, V)
    rows = pools[2].k_hist.view(-1, H, D)
    assert not pools[2].append_prompts(slots, [0, *[x - 5 for x in starts[1:]]], rows, rows)
    assert before[0] == pools[2].seq_len and torch.equal(before[1], pools[2].k_hist)


@pytest.mark.parametrize("ring", [False, True])
def test_a_step_of_rows_and_cursors_in_one_call(ring):
    """append_step against append_decode_batched over steps that complete groups; a slot that is not one token behind,
    without room, named twice, or rows of another type or device are refused and nothing moves."""
    H, D, win, lens = 2, 64, WindowSpec(), [70, 9, 103, 71]
    pools = [MultiSeqKVPool(D, H, 6, 110, window=win, device=DEV, kv_ring=ring, **RECIPE) for _ in range(2)]
    slots = [3, 0, 5, 2]
    for i, (r, n) in enumerate(zip(slots, lens)):
        K, V = _block(n, H, D, torch.bfloat16, 10 + i), _block(n, H, D, torch.bfloat16, 20 + i)
        for p in pools:
            p.append_block(r, K, V)
    sel = torch.tensor(slots, device=DEV)
    for s in range(1, 6):
        K, V = _block(4, H, D, torch.bfloat16, 30 + s), _block(4, H, D, torch.bfloat16, 40 + s)
        seqs = [n + s for n in lens]
        cols = torch.tensor([n - 1 for n in seqs], device=DEV)
        assert pools[0].append_step(slots, seqs, sel, cols, K, V)
        pools[1].append_decode_batched(slots, K, V)
        assert pools[0].seq_len == pools[1].seq_len and pools[0].packed_groups == pools[1].packed_groups
        assert torch.equal(pools[0].k_hist[sel], pools[1].k_hist[sel]) and torch.equal(pools[0].v_hist[sel], pools[1].v_hist[sel])
    for r in slots:
        a, b = pools[0].request_planes(r), pools[1].request_planes(r)
        for n in ("k_base", "k_scale", "k_obmp", "k_oval", "v_main", "v_scale"):
            assert torch.equal(a[n], b[n]), (r, n)
    held, hist = list(pools[0].seq_len), pools[0].k_hist.clone()
    nxt = [n + 6 for n in lens]
    cols = torch.tensor([n - 1 for n in nxt], device=DEV)
    refused = [(slots, [n + 1 for n in nxt], K, V), (slots, [*nxt[:3], nxt[3] - 1], K, V), ([3, 0, 5, 5], [*nxt[:3], nxt[2]], K, V),
               (slots, nxt, K.float(), V.float()), (slots, nxt, K.cpu(), V.cpu()), (slots, nxt, K[:3], V[:3]),
               (tuple(slots), nxt, K, V), ([3, 0, 5, 9], nxt, K, V)]
    for sl, sq, k, v in refused:
        assert not pools[0].append_step(sl, sq, sel, cols, k, v)
    if not ring:
        pools[0].seq_len[5] = 110
        assert not pools[0].append_step(slots, [nxt[0], nxt[1], 111, nxt[3]], sel, cols, K, V)
        pools[0].seq_len[5] = held[5]
    assert held == pools[0].seq_len and torch.equal(hist, pools[0].k_hist)


@pytest.mark.parametrize("ring,B,D,view", [(False, 1, 64, False), (True, 4, 128, False), (True, 64, 64, False), (False, 5, 64, True),
                                           (True, 65, 64, False)])
def test_a_step_whose_places_go_with_the_launch(ring, B, D, view):
    """append_step_rows against append_step over steps that complete groups and turn the ring: histories, cursors, planes and
    the block for the step's other launches; rows of a strided view; 65 requests and what append_step refuses change
    nothing."""
    H, win = 2, WindowSpec()
    pools = [MultiSeqKVPool(D, H, B + 2, 210, window=win, device=DEV, kv_ring=ring, **RECIPE) for _ in range(2)]
    slots = [(3 * i + 1) % (B + 2) if (B + 2) % 3 else i for i in range(B)]
    lens = [60 + 7 * (i % 19) for i in range(B)]
    for i, (r, n) in enumerate(zip(slots, lens)):
        K, V = _block(n, H, D, torch.bfloat16, 10 + i), _block(n, H, D, torch.bfloat16, 200 + i)
        for p in pools:
            p.append_block(r, K, V)
    sel, block = torch.tensor(slots, device=DEV), torch.full((7 * B,), -1, dtype=torch.int32, device=DEV)
    for s in range(1, 9):
        K, V = _block(B, H, D, torch.bfloat16, 30 + s), _block(B, H, D, torch.bfloat16, 40 + s)
        if view:
            both = torch.stack([K, V], 2)                       # [B, H, 2, D]: a head stride of 2 D
            K, V = both[:, :, 0], both[:, :, 1]
        seqs = [n + s for n in lens]
        got = pools[0].append_step_rows(slots, seqs, K, V, block if s % 2 else None)
        assert pools[0].step_rows == 64
        if B > 64:
            assert got is None and pools[0].seq_len == pools[1].seq_len and bool((block == -1).all())
            return
        packed = [win.packed_len(n) for n in seqs]
        assert got == (max(packed), sum(packed))
        assert pools[1].append_step(slots, seqs, sel, torch.tensor([n - 1 for n in seqs], device=DEV), K, V)
        assert pools[0].seq_len == pools[1].seq_len and pools[0].packed_groups == pools[1].packed_groups
        assert torch.equal(pools[0].k_hist[sel], pools[1].k_hist[sel]) and torch.equal(pools[0].v_hist[sel], pools[1].v_hist[sel])
        if s % 2:
            wide = block[:6 * B].view(torch.int64).view(3, B)
            assert wide.tolist() == [slots, [n - 1 for n in seqs], seqs] and block[6 * B:].tolist() == packed
    for r in slots:
        a, b = pools[0].request_planes(r), pools[1].request_planes(r)
        for n in ("k_base", "k_scale", "k_obmp", "k_oval", "v_main", "v_scale"):
            assert torch.equal(a[n], b[n]), (r, n)
    held, hist, was = list(pools[0].seq_len), pools[0].k_hist.clone(), block.clone()
    nxt = [n + 9 for n in lens]
    refused = [(slots, [n + 1 for n in nxt], K, V, block), (slots, nxt, K.float(), V.float(), block), (slots, nxt, K.cpu(), V.cpu(), block),
               (slots, nxt, K[:0], V[:0], block), (tuple(slots), nxt, K, V, block), ([B + 7, *slots[1:]], nxt, K, V, block),
               (slots, nxt, K, V, block[:-1]), (slots, nxt, K, V, block.long()), (slots, nxt, K, V, block.cpu())]
    for sl, sq, k, v, to in refused:
        assert pools[0].append_step_rows(sl, sq, k, v, to) is None
    if not ring:
        pools[0].seq_len[slots[0]] = 210
        assert pools[0].append_step_rows(slots, [211, *nxt[1:]], K, V, block) is None
        pools[0].seq_len[slots[0]] = held[slots[0]]
    torch.cuda.synchronize()
    assert held == pools[0].seq_len and torch.equal(hist, pools[0].k_hist) and torch.equal(was, block)
    pools[0].check_errors()


@pytest.mark.parametrize("sink,span,wsink,count,H,ps", [
    (0, 0, 8, 3, 8, 16), (8, 96, 8, 3, 8, 16),            # whole history; groups that end where the ring turns
    (8, 83, 8, 2, 3, 8), (8, 41, 13, 1, 8, 32),           # groups that turn with it
    (8, 96, 8, 96, 2, 16), (8, 96, 8, 97, 2, 16), (0, 0, 8, 30, 70, 16)])   # as arguments, and through the tables
@pytest.mark.parametrize("rep", ["bitmap", "relidx7"])
def test_groups_of_a_history_as_arguments_of_their_store(sink, span, wsink, count, H, ps, rep):
    """pack_groups against the general entry with index tables, for the newest groups of many requests."""
    D, gt, per_seq, rows = 128, 32, 9, sink + span if span else 300
    g = torch.Generator(device=DEV).manual_seed(count + span)
    kh, vh = (torch.randn(count, rows, H, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    pairs = [(r, (5 * r + 3) % per_seq) for r in range(count)]
    pos = [[wsink + n * gt + i for i in range(gt)] for _, n in pairs]
    src = [r * rows + (ring_slot(p, sink, span) if span else p) for (r, _), ps_ in zip(pairs, pos) for p in ps_]
    pages = [(r * per_seq + n) * (gt // ps) + i for r, n in pairs for i in range(gt // ps)]
    groups = [r * per_seq + n for r, n in pairs]
    how = dict(outliers_per_vector=6, outlier_repr=rep)
    planes = [alloc_planes(count * per_seq * (gt // ps), count * per_seq, H, D, page_size=ps, device=DEV, **how) for _ in range(2)]
    for p in planes:
        for t in p.values():
            if torch.is_tensor(t):
                t.fill_(0x5A if t.dtype == torch.uint8 else 1)
    names = [n for n, t in planes[0].items() if torch.is_tensor(t)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    store_pack_into(kh.view(-1, H, D), vh.view(-1, H, D), planes[0], page_size=ps, src_rows=i32(src), dst_pages=i32(pages),
                    dst_groups=i32(groups), **how)
    err = torch.zeros(1, dtype=torch.int32, device=DEV)
    assert _hip.host().pack_groups(kh, vh, {n: planes[1].get(n) for n in ("k_base", "k_scale", "k_zp", "k_fp4_mapscale",
                                                                         "k_fp4_mapcenter", "k_obmp", "k_oidx", "k_oval",
                                                                         "v_main", "v_scale", "v_zp")},
                                   [x for pair in pairs for x in pair], ps, sink, span, wsink, per_seq, err,
                                   store_table(kh.device), 6, gt, 32, rep, "signed", True, True, "i2")
    assert int(err.item()) == 0
    for n in names:
        assert torch.equal(planes[0][n].view(torch.uint8), planes[1][n].view(torch.uint8)), n


@pytest.mark.parametrize("H,D", [(1, 8), (3, 40), (8, 128), (16, 256), (32, 256), (7, 12)])
def test_rows_of_any_width_reach_their_slot(H, D):
    """One piece of K or V a thread up to 1024 of them, several beyond, and rows without 16-byte pieces; positions past 32
    bits turn with the ring."""
    sink, span = 4, 24
    kh, vh = (torch.zeros(2, sink + span, H, D, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    for pos in ([3, 4], [27, 28], [2 ** 33 + 5, 2 ** 32 + 3]):
        K, V = _block(2, H, D, torch.bfloat16, pos[0] % 97), _block(2, H, D, torch.bfloat16, 7)
        at = torch.tensor(pos, dtype=torch.int64, device=DEV)
        assert _hip.host().ring_write(kh, vh, at, K, V, sink, span, None, at, None)
        assert at.tolist() == [p + 1 for p in pos]
        for b, p in enumerate(pos):
            slot = p if p < sink else sink + (p - sink) % span
            assert torch.equal(kh[b, slot], K[b]) and torch.equal(vh[b, slot], V[b])


@pytest.mark.parametrize("T,H,gt", [(105, 3, 32), (4096, 8, 32), (8300, 8, 32), (1100, 2, 64)])
@pytest.mark.parametrize("single", [False, True])
def test_rows_and_groups_of_a_fresh_block_in_one_launch(T, H, gt, single):
    """A fresh block against the same rows in two pieces, which take a launch for the rows and one for the groups: a full
    chip, one that is not, a block of one or two groups with more rows than that."""
    D, how = 128, dict(window=WindowSpec(group_tokens=gt), device=DEV, kv_ring=False, outliers_per_vector=6,
                       use_pow2=True, outlier_repr="bitmap" if gt == 32 else "relidx7")
    K, V = _block(T, H, D, torch.bfloat16, 1), _block(T, H, D, torch.bfloat16, 2)
    made = [CanonicalKVStore(D, H, T + 5, **how) if single else MultiSeqKVPool(D, H, 2, T + 5, **how) for _ in range(2)]
    put = (lambda s, a, b: s.append_block(a, b)) if single else (lambda s, a, b: s.append_block(1, a, b))
    for s in made:
        for t in [s.k_hist, s.v_hist, *(t for t in s._store_planes.values() if torch.is_tensor(t))]:
            t.zero_()
    put(made[0], K, V)
    put(made[1], K[:40], V[:40])
    put(made[1], K[40:], V[40:])
    assert made[0].seq_len == made[1].seq_len and made[0].packed_groups == made[1].packed_groups
    assert torch.equal(made[0].k_hist, made[1].k_hist) and torch.equal(made[0].v_hist, made[1].v_hist)
    for n, t in made[0]._store_planes.items():
        if torch.is_tensor(t):
            assert torch.equal(t.view(torch.uint8), made[1]._store_planes[n].view(torch.uint8)), n


@pytest.mark.parametrize("kw", [
    {}, dict(outlier_repr="relidx7", kv_outlier_map=False), dict(group_tokens=64, group_channels=64, outliers_per_vector=10, outlier_repr="relidx7"),
    dict(outliers_per_vector=0), dict(v_format="bf16", k_format="itf4"), dict(use_pow2=False, outlier_select="abs"),
    dict(kv_int8_scale=False, kv_outlier_map=None), dict(kv_int8_scale=True, outliers_per_vector=3)], ids=lambda k: "-".join(map(str, k.values())) or "serving")
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_one_call_of_a_block_gives_what_the_steps_give(kw, dtype):
    """Same keys in the same order, same values of the same types, same bits as arguments that take the way through Python
    (a device by its full name), and the same error for the same block."""
    call = dict(outliers_per_vector=6, outlier_repr="bitmap", outlier_select="signed", use_pow2=True, page_size=16) | kw
    K, V = _block(128, 2, 64, dtype, 31), _block(128, 2, 64, dtype, 32, strided=True)
    store_table(K.device)
    assert _hip.host().pack_whole_block(K, V, store_table(K.device), 16, "cuda:0", None, "i2f4", 6, 32, 32, "bitmap", "signed", True, None, "i2") is False
    want = ommx_pack_kv_canonical_block(K, V, device="cuda:0", **call)
    for device in ("cuda", torch.device("cuda"), torch.device("cuda", 0), K.device):
        got = ommx_pack_kv_canonical_block(K, V, device=device, **call)
        assert list(got) == list(want)
        for name, value in want.items():
            assert type(got[name]) is type(value), name
            if torch.is_tensor(value):
                assert got[name].dtype == value.dtype and got[name].device == value.device and got[name].is_contiguous(), name
                assert torch.equal(got[name].view(torch.uint8), value.view(torch.uint8)), name
            else:
                assert got[name] == value, name
    if kw.get("v_format") != "bf16":
        V = V.clone()
        V[5, 1, 3] = float("nan")
        for device in ("cuda", "cuda:0"):
            with pytest.raises(ValueError, match="V pack: non-finite"):
                ommx_pack_kv_canonical_block(K, V, device=device, **call)


@pytest.mark.parametrize("ring,B,H,win,repr_,form", [
    (False, 1, 1, {}, "bitmap", "plain"), (True, 1, 8, {}, "bitmap", "plain"), (False, 5, 8, {}, "relidx7", "view"), (True, 64, 2, {}, "bitmap", "plain"),
    (False, 64, 1, {}, "relidx7", "plain"), (True, 3, 2, {}, "relidx7", "odd"), (False, 4, 2, dict(recent_window=0), "bitmap", "plain"),
    (False, 4, 2, dict(sink_tokens=0, recent_window=1), "bitmap", "plain"), (True, 4, 2, dict(recent_window=1), "bitmap", "plain")])
def test_a_step_whose_rows_go_with_its_groups(ring, B, H, win, repr_, form, monkeypatch):
    """Steps that complete groups, rows and groups in one launch where that takes both, against rows first and groups behind them: histories,
    planes, cursors and the step's block are the same bits, step after step.  Not in one launch: a group that ends with the step's own token (no recent
    rows), rows that cannot be read 16 bytes at a time."""
    D, w = 128, WindowSpec(**win)
    pools = [MultiSeqKVPool(D, H, B + 2, 330, window=w, device=DEV, kv_ring=ring, outliers_per_vector=6, outlier_repr=repr_, use_pow2=True) for _ in range(2)]
    slots = [(3 * i + 1) % (B + 2) if (B + 2) % 3 else i for i in range(B)]
    lens = [35 + 11 * (i % 17) for i in range(B)]
    for i, (r, n) in enumerate(zip(slots, lens)):
        K, V = _block(n, H, D, torch.bfloat16, 10 + i), _block(n, H, D, torch.bfloat16, 200 + i)
        for p in pools:
            p.append_block(r, K, V)
    blocks = [torch.full((7 * B,), -1, dtype=torch.int32, device=DEV) for _ in pools]
    pools[1]._step_how = ()                                     # (nothing to pack with: a launch for the rows)
    groups_behind = []
    behind = pools[0]._pack_completed
    monkeypatch.setattr(pools[0], "_pack_completed", lambda full: groups_behind.append(full) or behind(full))
    completed = 0
    for s in range(1, 71):
        K, V = _block(B, H, D, torch.bfloat16, 30 + s), _block(B, H, D, torch.bfloat16, 140 + s)
        if form == "view":
            both = torch.stack([K, V], 2)
            K, V = both[:, :, 0], both[:, :, 1]
        elif form == "odd":
            K = torch.cat([K.flatten(), K.new_zeros(1)])[1:].view(B, H, D)
        seqs = [n + s for n in lens]
        was = list(pools[0].packed_groups)
        got = [p.append_step_rows(slots, seqs, K, V, t if s % 3 else None) for p, t in zip(pools, blocks)]
        assert got[0] == got[1] and got[0] is not None
        completed += pools[0].packed_groups != was
        assert pools[0].seq_len == pools[1].seq_len and pools[0].packed_groups == pools[1].packed_groups
        assert pools[0].packed_groups[slots[0]] == w.num_groups(seqs[0])
        for a, b in zip([*pools[0]._store_planes.values(), pools[0].k_hist, pools[0].v_hist, blocks[0]],
                        [*pools[1]._store_planes.values(), pools[1].k_hist, pools[1].v_hist, blocks[1]]):
            assert a is b is None or torch.equal(a.view(torch.uint8), b.view(torch.uint8)), s
    assert completed >= 2 and len(groups_behind) == (completed if form == "odd" or win.get("recent_window") == 0 else 0)
    for p in pools:
        p.check_errors()
