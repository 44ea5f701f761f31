"""The kernels of path preparation at the sizes where their tiles and packings end."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from eppgcn_amd import capi
    capi.load()
    assert torch.cuda.is_available()
    return capi


@pytest.mark.parametrize("n,length", [(1, 1), (31, 5), (32, 1023), (33, 1024), (8192, 1025), (8193, 40000),
                                      (70001, 4097), (1 << 18, 3), (5, 0)])
@pytest.mark.parametrize("shift", [0, 1])
def test_distinct_rows_with_and_without_scratch(api, n, length, shift):
    """`shift`: the list starts 4 bytes past a 16-byte boundary.  Half of the entries are one hub row."""
    rng = np.random.default_rng(n * 7 + length)
    rows = rng.integers(0, n, length + shift, dtype=np.int32)
    rows[rng.random(length + shift) < 0.5] = n // 2
    lst = torch.from_numpy(rows).cuda()[shift:]
    want = np.zeros((n + 31) // 32 * 32, np.uint8)
    want[rows[shift:]] = 1
    bits = np.packbits(want, bitorder="little").view(np.int32)
    got, count = api.mark_gathered_rows(lst, length, n)
    assert count == int(want.sum()) and np.array_equal(got.cpu().numpy(), bits)
    # the entry point without scratch memory
    lib, out = api.load(), torch.full(((n + 31) // 32 + 1,), -1, dtype=torch.int32, device="cuda")
    v = ctypes.c_int64(-1)
    rc = lib.eppgcn_mark_gathered_rows(lst.data_ptr() if length else None, length, n, out.data_ptr(), out[-1:].data_ptr(),
                                       ctypes.byref(v), torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and v.value == count and np.array_equal(out[:-1].cpu().numpy(), bits)


@pytest.mark.parametrize("n", [0, 1, 255, 4096, 4097, 300001])
def test_count_of_rows_with_kept_edges(api, n):
    deg = (np.arange(n) % 3).astype(np.int32)
    assert api.count_nonzero(torch.from_numpy(deg).cuda()) == int(np.count_nonzero(deg))


@pytest.mark.parametrize("n,slots_per_row,loops,ps", [
    (1, 3, True, 2), (33, 5, True, 4), (500, 9, False, 1),          # a single small tile
    (700, 0, True, 3),                                              # nothing but self-loops
    (3000, 11, True, 8), (3001, 11, False, 64),                     # several small tiles, with and without self-loops
    (9, 3000, True, 32),                                            # rows of several tiles
    (300000, 15, True, 16), (9, 600000, False, 32),                 # a thousand tiles
    (4300000, 0, True, 1)])                                         # as many groups in a tile as slots
@pytest.mark.parametrize("is_last", [False, True])
@pytest.mark.parametrize("shift", [0, 1])
def test_path_marking_in_one_pass(api, n, slots_per_row, loops, ps, is_last, shift):
    _check_marking(api, n, slots_per_row, loops, ps, is_last, shift)


@pytest.mark.parametrize("n,slots_per_row,loops,ps", [
    (2300000, 15, True, 16), (9, 6000000, False, 32),               # nine and thirteen thousand tiles (scanned from 2^25 slots on)
    (34000000, 0, True, 1)])                                        # as many groups in a tile as slots
@pytest.mark.parametrize("is_last", [False, True])
def test_path_marking_in_large_tiles(api, n, slots_per_row, loops, ps, is_last):
    assert _check_marking(api, n, slots_per_row, loops, ps, is_last, 1) >= 1 << 25


@pytest.mark.parametrize("n", [512 * 4096 - 1, 512 * 4096, 512 * 4096 + 1])
@pytest.mark.parametrize("is_last", [False, True])
def test_path_marking_where_the_workgroups_get_smaller(api, n, is_last):
    """512 and 513 tiles of 4096 slots, the last one full, one slot short and one slot long."""
    assert _check_marking(api, n, 0, True, 4, is_last, 0) == n


@pytest.mark.parametrize("slots", [(1 << 25) - 4096, (1 << 25) - 4095])
def test_path_marking_where_the_counts_are_scanned(api, slots):
    """8191 full tiles add up the counts before theirs, 8192 (the last one with a single slot) have them scanned."""
    assert _check_marking(api, slots, 0, True, 64, False, 0) == slots


@pytest.mark.parametrize("e", [40, 4096, 4097, 30000, 9000000])
@pytest.mark.parametrize("is_last", [False, True])
def test_path_marking_with_empty_groups_and_slots_of_no_group(api, e, is_last):
    """Runs of empty groups, also at the start of a tile and at both ends, and slots before the first group and behind the last
    one, which are never kept and mark nobody.  A row whose groups are all empty is not its own neighbour."""
    rng = np.random.default_rng(e)
    n = max(8, e // 9)
    cuts = np.unique(np.concatenate([rng.integers(3, e - 5, e // 7 + 1), [3, e - 5], np.arange(4096, e - 5, 4096)])).astype(np.int64)
    again = rng.integers(0, 4, cuts.size) * (rng.random(cuts.size) < 0.2)          # empty groups in front of a group
    again[[0, -1]] = 2
    pp = np.repeat(cuts, 1 + again)
    p2n = np.sort(rng.integers(0, n, pp.size - 1)).astype(np.int32)
    _check_groups(api, pp, p2n, e, n, is_last, rng)


def _check_groups(api, pp, p2n, e, n, is_last, rng):
    """Marking of e slots with random columns and sources against the groups' definition: slot s belongs to the group with slots
    that starts last at or before s."""
    slots = np.arange(e)
    row = np.full(e, -1)
    filled = np.flatnonzero(np.diff(pp) > 0)
    inside = (slots >= pp[0]) & (slots < pp[-1])
    row[inside] = p2n[filled[np.searchsorted(pp[filled], slots[inside], side="right") - 1]]
    col = rng.integers(0, n, e).astype(np.int32)
    src = rng.random(n) < 0.3
    keep = inside & src[col]
    ngh = np.zeros(n, bool)
    if not is_last:
        marked = inside & src[np.maximum(row, 0)]
        ngh[row[marked]] = True
        ngh[col[marked]] = True
    want = np.zeros((2, e), np.int32)
    v = int(keep.sum())
    want[0, :v], want[1, :v] = row[keep], col[keep]
    degs_want = np.bincount(row[keep], minlength=n)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for call in (api.mark_path, api.mark_compact):
        degs, got_ngh = torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.bool, device="cuda")
        got = call(d(p2n), d(pp.astype(np.int32)), d(col), d(src), None if is_last else got_ngh, degs, is_last)
        assert got[2] == v and np.array_equal(degs.cpu().numpy(), degs_want)
        assert np.array_equal(got[0].cpu().numpy(), want[0]) and np.array_equal(got[1].cpu().numpy(), want[1])
        assert np.array_equal(got_ngh.cpu().numpy(), ngh)


@pytest.mark.parametrize("at", [(4096,), (8192,), (5000,), (4096, 5000, 8192)])
@pytest.mark.parametrize("e", [12388, 3000000, 34000000])
@pytest.mark.parametrize("is_last", [False, True])
def test_path_marking_where_a_tile_has_more_groups_than_slots(api, at, e, is_last):
    """Five thousand empty groups at a slot: a tile's rows are not staged then.  Where they start with the next tile, no two
    groups of this one share a slot; in the middle they do.  In each of the three sizes of workgroups."""
    rng = np.random.default_rng(e + len(at))
    cuts = np.unique(np.concatenate([rng.integers(0, e, e // 5), [0, e], at])).astype(np.int64)
    pp = np.repeat(cuts, 1 + 5000 * np.isin(cuts, at))
    n = max(8, e // 9)
    p2n = np.sort(rng.integers(0, n, pp.size - 1)).astype(np.int32)
    _check_groups(api, pp, p2n, e, n, is_last, rng)


def _marking_us(api, p2n, pp, col, n, is_last):
    """Shortest of ten markings."""
    src = torch.arange(n, device="cuda") % 10 == 0
    best = float("inf")
    for _ in range(10):
        ngh, degs = torch.zeros(n, dtype=torch.bool, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        torch.cuda.synchronize()
        start.record()
        pending = api.mark_path_begin(p2n, pp, col, src, None if is_last else ngh, degs, is_last)
        end.record()
        pending()
        best = min(best, start.elapsed_time(end) * 1e3)
    return best


@pytest.mark.parametrize("is_last", [False, True])
def test_one_slot_groups_are_staged(api, is_last):
    """A tile of one-slot groups has 4097 of them, with the next tile's first.  With their rows staged, 33.5 M slots take 1.25 to
    1.3 times as long in groups of one slot as in groups of two; with a search per slot it is 2.06 to 2.27 times."""
    n = 1 << 22
    indptr = torch.arange(0, 8 * n + 1, 8, dtype=torch.int32, device="cuda")
    col = torch.randint(0, n, (8 * n,), dtype=torch.int32, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    one, two = (_marking_us(api, *reversed(api.build_part(ps, indptr, 8 * n)), col, n, is_last) for ps in (1, 2))
    print("groups of 1 and 2 slots:", one, two, "us")
    assert one < 1.6 * two


@pytest.mark.parametrize("tiles", [3, 4, 5, 6, 68, 69, 133])
@pytest.mark.parametrize("edge", [-1, 0, 1])
def test_path_marking_with_groups_of_many_tiles(api, tiles, edge):
    """A thread writes up to four tiles of a group, its wave the others: a group of `tiles` tiles behind one slot, in the middle of
    small groups, and as the last group in front of as many tiles of no group."""
    rng = np.random.default_rng(tiles)
    long = tiles * 4096 + edge
    small = np.arange(0, 40000, 5)
    pp = np.concatenate([[0, 1, 1 + long], 1 + long + small[1:], 40000 + 2 * long + np.array([0, long])]).astype(np.int64)
    e = int(pp[-1]) + long
    n = 3000
    p2n = np.sort(rng.integers(0, n, pp.size - 1)).astype(np.int32)
    _check_groups(api, pp, p2n, e, n, False, rng)


def test_one_group_is_marked_by_more_than_a_thread(api):
    """2^27 slots in one group, and in none but the first 4096: 32 thousand tiles whose group is the same.  They take 1.14 and 0.6
    times as long as 2^27 slots in groups of 32; written by one thread 2.2 and 1.8 times."""
    n, e = 1 << 20, 1 << 27
    col = torch.randint(0, n, (e,), dtype=torch.int32, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    rows = torch.zeros(1, dtype=torch.int32, device="cuda")
    many = torch.arange(0, e + 1, 32, dtype=torch.int32, device="cuda")
    usual = _marking_us(api, torch.arange(many.numel() - 1, device="cuda", dtype=torch.int32) % n, many, col, n, True)
    for end in (e, 4096):
        us = _marking_us(api, rows, torch.tensor([0, end], dtype=torch.int32, device="cuda"), col, n, True)
        print("groups of 32 slots, one group of", end, ":", usual, us, "us")
        assert us < 1.25 * usual


def _check_marking(api, n, slots_per_row, loops, ps, is_last, shift):
    """`shift`: the masks start one byte past a word boundary.  Vertex 0 is a neighbour of every third slot.  -> slots"""
    rng = np.random.default_rng(n + slots_per_row)
    deg = rng.integers(0, 2 * slots_per_row + 1, n) + (1 if loops else 0)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    e = int(indptr[-1])
    row = np.repeat(np.arange(n, dtype=np.int32), deg)
    col = rng.integers(0, n, e, dtype=np.int32)
    col[::3] = 0
    if loops:
        col[indptr[:-1]] = np.arange(n)
    src = rng.random(n) < 0.3
    keep = src[col]
    want_ngh = np.zeros(n, bool)
    if not is_last:
        want_ngh[row[src[row]]] = True
        want_ngh[col[src[row]]] = True
    degs_want = np.bincount(row[keep], minlength=n).astype(np.int32)
    gathered = np.zeros((n + 31) // 32 * 32, np.uint8)
    gathered[col[keep]] = 1

    pp, p2n = api.build_part(ps, torch.from_numpy(indptr).cuda(), e)
    hold = torch.zeros(2, n + 1, dtype=torch.bool, device="cuda")
    d_src, ngh = hold[0][shift:shift + n], hold[1][shift:shift + n]
    d_src.copy_(torch.from_numpy(src))
    degs = torch.zeros(n, dtype=torch.int32, device="cuda")
    ids, edges, kept, rows, bitmap, distinct = api.mark_path(p2n, pp, torch.from_numpy(col).cuda(), d_src,
                                                             None if is_last else ngh, degs, is_last)
    v = int(keep.sum())
    assert (kept, rows, distinct) == (v, int(np.count_nonzero(degs_want)), int(gathered.sum()))
    want = np.zeros((2, e), np.int32)
    want[0, :v], want[1, :v] = row[keep], col[keep]
    assert np.array_equal(ids.cpu().numpy(), want[0]) and np.array_equal(edges.cpu().numpy(), want[1])
    assert np.array_equal(degs.cpu().numpy(), degs_want)
    assert np.array_equal(ngh.cpu().numpy(), want_ngh)
    assert np.array_equal(bitmap.cpu().numpy(), np.packbits(gathered, bitorder="little").view(np.int32))
    # the entry point without the path's counts (it reads the mask byte by byte)
    again, ngh2 = torch.zeros_like(degs), torch.zeros_like(ngh)
    ids2, edges2, kept2 = api.mark_compact(p2n, pp, torch.from_numpy(col).cuda(), d_src, None if is_last else ngh2, again, is_last)
    assert kept2 == v and torch.equal(ids2, ids) and torch.equal(edges2, edges)
    assert torch.equal(again, degs) and torch.equal(ngh2, ngh)
    return e


@pytest.mark.parametrize("n,top,ps", [(1, 3, 2), (1023, 9, 4), (2048, 7, 1), (2049, 7, 1), (4097, 40, 8), (5000, 0, 3),
                                      (70000, 25, 4), (3, 200000, 5)])
def test_group_split_at_the_ends_of_tiles(api, n, top, ps):
    """Rows of 0 to `top` slots, a hub in the middle: both directions, with and without room to spare."""
    rng = np.random.default_rng(n + top)
    deg = rng.integers(0, top + 1, n).astype(np.int32)
    deg[n // 2] = 40 * top
    groups = (deg + ps - 1) // ps
    inside = np.arange(groups.sum()) - np.repeat(np.cumsum(groups) - groups, groups)
    first = np.cumsum(deg) - deg
    e = int(deg.sum())
    want = np.concatenate([np.repeat(first, groups) + inside * ps, [e]]).astype(np.int32)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    pp, p2n = api.build_part(ps, torch.from_numpy(indptr).cuda(), e)
    assert np.array_equal(pp.cpu().numpy(), want)
    assert np.array_equal(p2n.cpu().numpy(), np.repeat(np.arange(n, dtype=np.int32), groups))
    for room in (e, e + 37):
        got, parts, slots = api.split_back_part(torch.from_numpy(deg).cuda(), room, ps)
        assert (parts, slots) == (int(groups.sum()), e)
        got = got.cpu().numpy()
        assert np.array_equal(got[:parts + 1], want) and not got[parts + 1:].any()


@pytest.mark.parametrize("groups", [1, 4, 5, 63, 64, 65, 127, 128, 129, 5000])
@pytest.mark.parametrize("ps", [1, 3])
def test_groups_of_a_hub(api, groups, ps):
    """A wave writes the first 64 groups of a vertex in one step and those behind them in loops that end at the capacity."""
    deg = np.array([2, groups * ps - ps // 2, 0, 7], np.int32)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    count = (deg + ps - 1) // ps
    want = np.concatenate([start + ps * np.arange(c) for start, c in zip(indptr, count)] + [[indptr[-1]]]).astype(np.int32)
    pp, p2n = api.build_part(ps, torch.from_numpy(indptr).cuda(), int(indptr[-1]))
    assert np.array_equal(pp.cpu().numpy(), want) and np.array_equal(p2n.cpu().numpy(), np.repeat(np.arange(4), count))
    lib = api.load()
    nbytes = lib.eppgcn_split_workspace_bytes(4)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    for capacity in sorted({1, 2, 3, 66, 67, 68, groups, want.size - 1, want.size, want.size + 9}):
        whole = torch.full((capacity + 200,), 7, dtype=torch.int32, device="cuda")
        parts, slots = ctypes.c_int64(), ctypes.c_int64()
        rc = lib.eppgcn_split_back_part(torch.from_numpy(deg).cuda().data_ptr(), 4, ps, whole[100:].data_ptr(), capacity,
                                        ws.data_ptr(), nbytes, None, ctypes.byref(parts), ctypes.byref(slots),
                                        torch.cuda.current_stream().cuda_stream)
        got = whole.cpu().numpy()
        assert rc == (0 if capacity >= want.size else -4) and (got[:100] == 7).all() and (got[100 + capacity:] == 7).all()
        inside = min(capacity, want.size)
        assert np.array_equal(got[100:100 + inside], want[:inside]) and not got[100 + inside:100 + capacity].any()


@pytest.mark.parametrize("layers", [2, 6])
def test_preparing_several_layers_holds_one_build_workspace(api, layers):
    """All plans of a run are under way before the host waits for the first one, but their builds follow one another on the
    stream: beyond what stays, path preparation needs the workspace of the largest build and the marking of the layers (a
    bit per slot and a little over a byte per vertex), not a build workspace per layer."""
    from eppgcn_amd import graphs, workload
    g = graphs.rmat_graph(17, 8, seed=3, device="cuda")
    mask = graphs.bernoulli_mask(g.num_nodes, 0.9, 4, "cuda")
    run = lambda: workload.prepare(g, layers, train_mask=mask, widths=(16,), plan=True, part_size=2, backsize=2)
    run()                                            # whatever the first call loads and keeps
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    wl = run()
    torch.cuda.synchronize()
    over = torch.cuda.max_memory_allocated() - torch.cuda.memory_allocated()
    lib = api.load()
    build = max([lib.eppgcn_plan_workspace_bytes(wl.part2node.numel(), g.num_edges)] +
                [lib.eppgcn_plan_workspace_bytes(p.num_parts, p.valid_len) for p in wl.paths])
    marking = layers * lib.eppgcn_mark_path_workspace_bytes(g.num_edges, g.num_nodes)
    assert over <= 1.05 * build + marking, (over, build, marking)


def test_results_are_waited_for_on_the_stream_they_were_issued_on(api):
    """The three calls that are issued first and waited for later, issued behind other work on a side stream and waited for
    with the default stream current."""
    from eppgcn_amd import graphs
    g = graphs.rmat_graph(14, 8, seed=3, device="cuda")
    n, e = g.num_nodes, g.num_edges
    pp, p2n = api.build_part(16, g.row_pointers, e)
    src = graphs.bernoulli_mask(n, 0.2, 4, "cuda")
    degs, degs2 = torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
    want = api.mark_path(p2n, pp, g.column_index, src, None, degs, True)
    want_split = api.split_back_part(degs, e, 8)
    want_plan = api.build_plan(pp, g.column_index, p2n.numel(), e, n, 16, part2node=p2n)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)                 # some milliseconds
        marked = api.mark_path_begin(p2n, pp, g.column_index, src, None, degs2, True)
        split = api.split_back_part_begin(degs, e, 8)
        plan = api.build_plan_begin(pp, g.column_index, p2n.numel(), e, n, 16, part2node=p2n)
    plan, split, marked = plan(), split(), marked()
    assert marked[2:4] == want[2:4] and marked[5] == want[5]
    assert all(torch.equal(marked[i], want[i]) for i in (0, 1, 4)) and torch.equal(degs2, degs)
    assert split[1:] == want_split[1:] and torch.equal(split[0], want_split[0])
    assert plan.partial_rows == want_plan.partial_rows
    assert all(torch.equal(a, b) for a, b in zip(plan.view(), want_plan.view()))


def test_path_counts_of_other_sizes_are_refused(api):
    """The kept slots size a launch where a marked vertex has no self-loop: counts that cannot be those of the sizes given
    are an error before anything is launched."""
    from eppgcn_amd import graphs
    g = graphs.rmat_graph(12, 8, seed=3, device="cuda")
    n, e = g.num_nodes, g.num_edges
    lib = api.load()
    pp, p2n = api.build_part(16, g.row_pointers, e)
    src, degs = torch.ones(n, dtype=torch.bool, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
    out = torch.empty(2, e, dtype=torch.int32, device="cuda")
    bitmap = torch.empty((n + 31) // 32, dtype=torch.int32, device="cuda")
    ws = torch.empty(lib.eppgcn_mark_path_workspace_bytes(e, n), dtype=torch.uint8, device="cuda")
    stream, counts = torch.cuda.current_stream().cuda_stream, (ctypes.c_int64 * 3)()
    assert lib.eppgcn_mark_path(p2n.data_ptr(), pp.data_ptr(), g.column_index.data_ptr(), src.data_ptr(), None, degs.data_ptr(),
                                out[0].data_ptr(), out[1].data_ptr(), bitmap.data_ptr(), p2n.numel(), e, n, 1, ws.data_ptr(),
                                ws.numel(), None, stream) == 0
    ask = lambda edges, nodes: lib.eppgcn_mark_path_counts(out[1].data_ptr(), bitmap.data_ptr(), edges, nodes, ws.data_ptr(),
                                                           counts, stream)
    assert ask(e - 1, n) == -1 and b"finished eppgcn_mark_path" in lib.eppgcn_last_error()
    assert ask(e, n - 1) == -1
    assert ask(e, n) == 0 and list(counts) == [e, n, n]
