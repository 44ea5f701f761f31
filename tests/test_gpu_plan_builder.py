"""GPU tests of the plan builder where its tiles end: group counts around the tiles of its two scans, slot counts around
a fill tile and a wave, groups longer than a fill tile, empty rows between them, one block and several.  The stream arrays
are held, entry by entry, against the plain construction of tests/test_gpu_stream.py."""
import numpy as np
import pytest
import torch

from oracle import c_oracle as co
from tests.test_gpu_stream import check_stream_form, dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from eppgcn_amd import capi
    capi.load()
    assert torch.cuda.is_available(), "these tests need the MI355X"
    return capi


def csr_of(degrees, seed):
    """CSR with these row lengths, columns ascending inside a row (repeats allowed)."""
    degrees = np.asarray(degrees, np.int64)
    indptr = np.concatenate([[0], np.cumsum(degrees)]).astype(np.int32)
    n = degrees.size
    col = np.random.default_rng(seed).integers(0, n, int(indptr[-1]))
    rows = np.repeat(np.arange(n), degrees)
    col = col[np.lexsort((col, rows))].astype(np.int32)
    return indptr, col


def degrees_of(kind):
    rng = np.random.default_rng(17)
    if kind.startswith("ones"):                      # one group per row: exactly that many groups and slots
        return np.ones(int(kind[4:]), np.int64)
    if kind == "long":                               # groups and pieces longer than fill tiles and waves
        return np.array([5000, 0, 0, 1, 2047, 2049, 512, 511, 513, 0, 1, 4096], np.int64)
    if kind == "mixed":                              # several tiles of groups, empty rows, rows of one to many groups
        d = rng.integers(0, 40, 12000)
        d[rng.random(12000) < 0.3] = 0
        d[[7, 4000, 11999]] = [9000, 3000, 1500]
        return d
    raise ValueError(kind)


@pytest.mark.parametrize("kind,ps", [("ones1", 1), ("ones511", 3), ("ones512", 3), ("ones2047", 3), ("ones2048", 1),
                                     ("ones2049", 8), ("ones4095", 2), ("ones4096", 2), ("ones4097", 2), ("ones8193", 1),
                                     ("long", 4), ("long", 6000), ("mixed", 1), ("mixed", 7), ("mixed", 32)])
@pytest.mark.parametrize("shift", [0, 5, 31])
def test_stream_form_at_tile_edges(api, kind, ps, shift):
    indptr, col = csr_of(degrees_of(kind), 3)
    n = indptr.size - 1
    pp, p2n = co.build_part(ps, indptr)
    plan = api.build_plan(dev(pp), dev(col), p2n.size, col.size, n, 16, part2node=dev(p2n), block_shift=shift)
    check_stream_form(api, plan, n)


def test_slots_no_group_covers_gather_nothing(api):
    """A column array longer than what the groups cover: the slots behind the last group are padding."""
    indptr, col = csr_of(degrees_of("mixed"), 5)
    n = indptr.size - 1
    pp, p2n = co.build_part(16, indptr)
    longer = np.concatenate([col, np.zeros(3000, np.int32)])
    plan = api.build_plan(dev(pp), dev(longer), p2n.size, longer.size, n, 16, part2node=dev(p2n))
    got = plan.stream_view()["col"].cpu().numpy()
    assert np.all(got[col.size:] == (n + 4095) // 4096 * 4096)
    rng = np.random.default_rng(1)
    x = rng.integers(-4, 5, (n, 16)).astype(np.float32)
    ones = np.ones(n, np.float32)
    out = api.spmm_forward(dev(x), dev(longer), dev(ones), dev(pp), dev(p2n), part_size=16, plan=plan)
    assert api.last_call_used_stream()
    assert np.array_equal(out.cpu().numpy(), co.spmm_f64(x, indptr, col, ones).astype(np.float32))


@pytest.mark.parametrize("num_slots", [2 ** 31 - 2049, 2 ** 31 - 1025, 2 ** 31 - 513])
def test_the_largest_plans(api, num_slots):
    """Up to the slot counts that 32-bit offsets hold (every count below 2^31 - 1024 is promised, the padding to whole waves
    ends at 2^31 - 512): the last fill tile ends past 2^31 - 1.  Copied ids, padding, and the aggregation over them, whose
    sums are whole numbers below 2^24."""
    n, per_row = 4096, 1 << 19
    ptr = torch.arange(n + 1, device="cuda").mul_(per_row).clamp_(max=num_slots).int()
    col = torch.arange(num_slots, dtype=torch.int32, device="cuda").remainder_(4099).remainder_(n)
    rows = torch.arange(n, dtype=torch.int32, device="cuda")
    plan = api.build_plan(ptr, col, n, num_slots, n, 4, part2node=rows, block_shift=8)
    got = plan.stream_view()
    at, row, _, ids = plan.view(raw_col=True)
    assert got["header"][0] == 1 and int(got["header"][4]) == 0 and int(at[n]) == num_slots
    for q, (a, b, r) in enumerate(zip(at[:-1].tolist(), at[1:].tolist(), row.tolist())):
        want = col[int(ptr[r]):int(ptr[r]) + b - a]
        assert torch.equal(ids[a:b] & 0x7fffffff, want), (q, r)
        assert int(ids[b - 1]) < 0 and not (ids[a:b - 1] < 0).any()
    assert (got["col"][num_slots:] == n).all() and got["col"].numel() == (num_slots + 511) // 512 * 512
    chunk = torch.arange(0, num_slots, 1 << 20, device="cuda") // 32
    ends = torch.searchsorted((at[1:] - 1).long(), chunk * 32)
    assert torch.equal((got["cev"][chunk] & 0x7fffffff).long(), ends)
    x = torch.randint(-4, 5, (n, 4), device="cuda", generator=torch.Generator("cuda").manual_seed(1)).float()
    out = api.spmm_forward(x, col, torch.ones(n, device="cuda"), ptr, rows, part_size=per_row, plan=plan)
    assert api.last_call_used_stream()
    for r in list(range(0, n, 97)) + [n - 2, n - 1]:
        count = torch.bincount(col[int(ptr[r]):int(ptr[r + 1])].long(), minlength=n).double()
        assert torch.equal(out[r].double(), count @ x.double()), r


@pytest.mark.parametrize("n,ps", [(1, 4), (2047, 1), (2048, 3), (2049, 32), (9000, 8)])
def test_split_and_plan_in_one_gives_what_the_two_give(api, n, ps):
    """Around the tiles of the split, an empty row next to a hub: the same group pointers, and in every array the plan that
    the ids of the slots give; a group count or a slot count that is not the path's is refused."""
    rng = np.random.default_rng(n)
    deg = rng.integers(0, 6, n)
    deg[rng.random(n) < 0.4] = 0
    deg[n // 2] = 700                                  # written by a whole wave
    degs = dev(deg, torch.int32)
    slots, e = int(deg.sum()), int(deg.sum()) + 5      # five slots dropped by the marking
    ids, col = dev(np.repeat(np.arange(n), deg), torch.int32), dev(rng.integers(0, n, e), torch.int32)
    pointer, parts, covered = api.split_back_part(degs, e, ps)
    assert (parts, covered) == (int((-(-deg // ps)).sum()), slots)
    for shift in (0, 5, 31):
        a = api.build_plan(pointer, col, parts, covered, n, 16, ids=ids, block_shift=shift)
        one = api.split_and_plan_begin(degs, col, e, ps, parts, slots, 16, shift)
        got = one() if shift else api.finish_all([one])[0]
        assert torch.equal(got[0], pointer) and got[1:3] == (parts, slots)
        b = got[3]
        for x, y in zip(a.view(raw_col=True), b.view(raw_col=True)):
            assert torch.equal(x, y)
        sa, sb = a.stream_view(), b.stream_view()
        assert a.partial_rows == b.partial_rows and sa["header"][:4].tolist() == sb["header"][:4].tolist()
        events, _, fix = sa["header"][1:4].tolist()
        used = {"col": None, "erow": events, "cev": None, "wtail": None, "touched": None, "frow": fix, "fptr": fix + 1}
        for name, count in used.items():
            assert torch.equal(sa[name][:count], sb[name][:count]), name
    wrong = {(max(parts - 1, 1), slots), (parts + 1, slots), (parts, slots - 1), (parts, slots + 1), (parts, e)} - {(parts, slots)}
    for wrong_parts, wrong_slots in wrong:             # edge_list is long enough for all of them
        for shift in (5, 31):
            with pytest.raises(api.EppgcnError, match="other counts|do not fit"):   # the split says so of too few groups
                api.split_and_plan_begin(degs, col, e, ps, wrong_parts, wrong_slots, 16, shift)()


def test_several_results_with_one_wait(api):
    """finish_all gives what the calls give one by one: marking, splits and plans of two streams.  The empty plan among them
    has no record and keeps none of the others from the common wait."""
    indptr, col = csr_of(degrees_of("mixed"), 5)
    n = indptr.size - 1
    pp, p2n = [dev(x) for x in co.build_part(16, indptr)]
    cold, src = dev(col), dev(np.arange(n) % 3 == 0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())

    def issue():
        degs = torch.zeros(n, dtype=torch.int32, device="cuda")
        work = [api.mark_path_begin(p2n, pp, cold, src, None, degs, True, part_size=7), api.split_back_part_begin(degs, col.size, 7),
                api.build_plan_begin(pp, cold, 0, 0, n, 16, part2node=p2n),
                api.build_plan_begin(pp, cold, p2n.numel(), col.size, n, 16, part2node=p2n)]
        with torch.cuda.stream(side):
            sdegs = torch.zeros(n, dtype=torch.int32, device="cuda")
            work += [api.mark_path_begin(p2n, pp, cold, src, None, sdegs, True), api.build_plan_begin(pp, cold, p2n.numel(), col.size, n, 64, part2node=p2n)]
        return work

    together, single = api.finish_all(issue()), [w() for w in issue()]
    assert together[0][2:4] == single[0][2:4] and together[0][5:] == single[0][5:]
    assert together[0][6] == together[1][1] == single[1][1] and together[1][2] == together[0][2]
    for k in (0, 4):
        assert all(torch.equal(x, y) for x, y in zip(together[k][:2], single[k][:2])) and len(together[k]) == 7 - k // 4
    assert torch.equal(together[1][0], single[1][0])
    for k in (2, 3, 5):
        assert together[k].partial_rows == single[k].partial_rows and together[k].num_parts == single[k].num_parts
        assert torch.equal(together[k].view(raw_col=True)[3], single[k].view(raw_col=True)[3])


@pytest.mark.parametrize("count", [1, 31, 32, 33, 65])
def test_more_records_than_one_launch_reads(api, count):
    """32 records fit a launch: every split gets its own counts back, also from the second launch on."""
    degs = [dev(np.arange(k + 1), torch.int32) for k in range(count)]
    got = api.finish_all([api.split_back_part_begin(d, 5000, 3) for d in degs])
    for k, (pointer, parts, covered) in enumerate(got):
        want = -(-np.arange(k + 1) // 3)
        assert (parts, covered) == (int(want.sum()), k * (k + 1) // 2)
        assert pointer[parts] == covered and pointer.numel() == 5001


@pytest.mark.parametrize("capacity", [1, 2, 5, 1 << 20, (1 << 20) + 1, (1 << 20) + 3])
@pytest.mark.parametrize("ps", [1, 3, 4])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_the_entries_behind_the_groups_are_cleared(api, capacity, ps, offset):
    """Either way of clearing (before the split, or behind it for tiny groups in large arrays), any alignment, nothing outside."""
    deg = np.random.default_rng(3).integers(0, 9, 3000).astype(np.int32) if capacity > 5 else np.array([0, min(capacity - 1, 2)], np.int32)
    lib = api.load()
    whole = torch.full((capacity + 64,), 7, dtype=torch.int32, device="cuda")
    out = whole[16 + offset:16 + offset + capacity]
    nbytes = lib.eppgcn_split_workspace_bytes(deg.size)
    ws = torch.empty(nbytes // 8 + 1, dtype=torch.int64, device="cuda")
    rc = lib.eppgcn_split_back_part(dev(deg).data_ptr(), deg.size, ps, out.data_ptr(), capacity, ws.data_ptr(), nbytes, None,
                                    None, None, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    at = np.cumsum(deg) - deg
    starts = np.concatenate([np.arange(a, a + d, ps) for a, d in zip(at, deg)] + [[deg.sum()]])
    want = np.zeros(capacity, np.int64)
    want[:starts.size] = starts
    assert np.array_equal(out.cpu().numpy(), want)
    assert (whole[:16 + offset] == 7).all() and (whole[16 + offset + capacity:] == 7).all()


@pytest.mark.parametrize("order", ["ascending", "descending", "mixed"])
@pytest.mark.parametrize("ps", [1, 7, 32])
def test_rows_in_any_order(api, order, ps):
    """The bitmaps of the rows are put together from runs of neighbouring groups whose rows ascend, and row by row where they
    do not: rows in another order than the groups' give the plan they give in order, for both kernels that run over it."""
    indptr, col = csr_of(degrees_of("mixed"), 9)
    n = indptr.size - 1
    name = np.arange(n, dtype=np.int32)
    if order == "descending":
        name = name[::-1].copy()
    elif order == "mixed":                             # blocks of 96 rows in a random order: ascending and not inside a wave
        blocks = np.random.default_rng(2).permutation((n + 95) // 96)
        name = np.concatenate([np.arange(b * 96, min(n, b * 96 + 96), dtype=np.int32) for b in blocks])
    pp, p2n = co.build_part(ps, indptr)
    rows = dev(name[p2n])
    plan = api.build_plan(dev(pp), dev(col), p2n.size, col.size, n, 16, part2node=rows)
    touched = plan.stream_view()["touched"].cpu().numpy().view(np.uint8)
    want = np.zeros(touched.size * 8, np.uint8)
    want[name[np.diff(indptr) > 0]] = 1
    assert np.array_equal(np.unpackbits(touched, bitorder="little"), want)
    x = np.random.default_rng(1).integers(-4, 5, (n, 16)).astype(np.float32)
    sums = np.zeros((n, 16), np.float32)
    sums[name] = co.spmm_f64(x, indptr, col, np.ones(n, np.float32)).astype(np.float32)
    try:
        for stream in (True, False):                   # the group kernel reads the rows of a single group (stored, not cleared)
            api.set_stream_mode(stream)
            out = torch.full((n, 16), float("nan"), device="cuda")
            api.spmm_forward(dev(x), dev(col), torch.ones(n, device="cuda"), dev(pp), rows, part_size=ps, plan=plan, out=out)
            assert api.last_call_used_stream() == stream and np.array_equal(out.cpu().numpy(), sums)
    finally:
        api.set_stream_mode(True)


@pytest.mark.parametrize("ps", [1, 3, 32])
@pytest.mark.parametrize("shift", [3, 6])
def test_sort_keys_of_rows_that_cross_a_tile(api, ps, shift):
    """Rows of up to 64 slots share a key.  Rows of 60 to 68 slots in groups of one slot reach 64 groups into the next tile of
    2048 groups, at many places relative to it; from the rows of the groups and from the ids of the slots."""
    from tests.test_gpu_parity import _check_plan_order_with
    rng = np.random.default_rng(7)
    n = 700
    deg = np.tile([64, 65, 1, 63, 68, 2, 60], n // 7)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    for keep, classes in ((2, False), (8, True)):
        api.set_plan_keep_rows(keep)
        api.set_plan_length_classes(classes)
        try:
            _check_plan_order_with(api, indptr, col, ps, ((16, shift),), 32 * keep, classes)
            pp, p2n = co.build_part(ps, indptr)
            args = (dev(pp), dev(col), p2n.size, col.size, n, 16)
            a = api.build_plan(*args, part2node=dev(p2n), block_shift=shift)
            b = api.build_plan(*args, ids=dev(np.repeat(np.arange(n, dtype=np.int32), deg)), block_shift=shift)
            assert all(torch.equal(x, y) for x, y in zip(a.view(raw_col=True), b.view(raw_col=True)))
        finally:
            api.set_plan_keep_rows(None)
            api.set_plan_length_classes(None)
