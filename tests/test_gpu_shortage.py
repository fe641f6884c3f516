"""Inserts and reservations that do not get a device buffer: the row-major copy
of the primary codes is optional to an insert, a failed reservation leaves the
lists whole, and merged batches' workspaces make room for anything else."""
import contextlib

import numpy as np
import pytest

import jhq_gpu_amd as jg

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def refused(lo, hi, skip=0, count=1 << 40):
    """Buffers of lo <= bytes < hi fail; yields a list that then holds how many."""
    n = []
    jg.lib().jhq_debug_fail_alloc(lo, hi, skip, count)
    try:
        yield n
    finally:
        n.append(int(jg.lib().jhq_debug_fail_alloc(0, 0, 0, 0)))


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def _make(x, d=512, M=64, **kw):
    p = dict(M=M, B=8, Br=4, alpha=4.0, nlist=8, nprobe=4, ivf_iters=2, batch_size=16, seed=42)
    p.update(kw)
    ix = jg.JHQGpuIndex(d, jg.Params(**p))
    ix.train(x[:1000])
    return ix


def _same(a, b, q, k=10):
    la, lb = a.lists(), b.lists()
    assert all(np.array_equal(la[n], lb[n]) for n in la)
    for kind in (0, 1, 2):  # 2: the pre-scan, whose re-check reads the copy
        a.set_scan_kind(kind)
        b.set_scan_kind(kind)
        (da, ia), (db, ib) = a.search(q, k), b.search(q, k)
        assert np.array_equal(ia, ib) and np.array_equal(_bits(da), _bits(db))
    a.set_scan_kind(0)
    b.set_scan_kind(0)


@pytest.fixture(scope="module")
def data():
    g = np.random.default_rng(3)
    return (g.standard_normal((4000, 512)).astype(np.float32),
            g.standard_normal((40, 512)).astype(np.float32))


def _copy_bytes(ix):
    """The row-major copy of an index's pool (the codes' own buffer has 16
    bytes more)."""
    return (ix.pool()[1] + 15) // 16 * 16 * 64


def test_add_without_row_copy(gpu, data):
    x, q = data
    want, got = _make(x), _make(x)
    want.add(x)
    n = _copy_bytes(want)
    with refused(n, n + 1, count=1) as hit:
        got.add(x)
    assert hit == [1]
    _same(got, want, q)


def test_append_without_row_copy(gpu, data):
    """An append that re-packs the pool while its copy's new buffer is refused,
    then appends in place."""
    x, q = data
    want, got = _make(x), _make(x)
    want.add(x[:2000])
    got.add(x[:2000])
    want.append(x[2000:3900])
    n = _copy_bytes(want)
    with refused(n, n + 1, count=1) as hit:
        got.append(x[2000:3900])
    assert hit == [1]
    _same(got, want, q)
    for ix in (want, got):
        ix.append(x[3900:])
    _same(got, want, q)


def test_shortage_of_the_reservation_leaves_the_lists(gpu, data):
    """The copy stays refused, also to the reservation behind the insert: the
    call fails, the vectors are in, and the index works again with memory."""
    x, q = data
    want, got = _make(x), _make(x)
    want.add(x[:2000])
    want.append(x[2000:])
    got.add(x[:2000])
    n = _copy_bytes(want)
    with refused(n, n + 1) as hit:
        with pytest.raises(jg.JHQDeviceError):
            got.append(x[2000:])
    assert hit[0] >= 2
    assert got.ntotal == want.ntotal
    _same(got, want, q)


# ---- merged batches: one list, long short lists, whose dump of 512 queries is
# 92 MB a lane (3 MB in batches of 16) -----------------------------------------
MB = 1 << 20


@pytest.fixture(scope="module")
def flat():
    g = np.random.default_rng(4)
    return (g.standard_normal((20000, 128)).astype(np.float32),
            g.standard_normal((700, 128)).astype(np.float32))


def _flat(x, n=None):
    ix = _make(x, d=128, M=32, nlist=1, nprobe=1)
    ix.add(x if n is None else x[:n])
    return ix


def _used():
    import torch
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def _device(ix, q, k, gpu):
    import torch
    qt = torch.from_numpy(q).to(gpu)
    d = torch.full((len(q), k), -1.0, device=gpu)
    i = torch.full((len(q), k), -2, dtype=torch.int32, device=gpu)
    ix.search_device(qt, k, d, i, stream=torch.cuda.current_stream())
    torch.cuda.synchronize()
    return d.cpu().numpy(), i.cpu().numpy()


def _equal(a, b):
    assert np.array_equal(a[1], b[1]) and np.array_equal(_bits(a[0]), _bits(b[0]))


def test_merged_shortage_gives_its_buffers_back(gpu, flat):
    x, q = flat
    want = _flat(x)
    want.reserve(100)
    res = want.search(q, 100)
    got = _flat(x)
    before = _used()
    with refused(50 * MB, 1 << 50, skip=2) as hit:  # two lanes get theirs
        got.reserve(100)
    assert hit == [1]
    assert _used() - before < 80 * MB
    _equal(got.search(q, 100), res)
    _equal(_device(got, q, 100, gpu), res)
    # an insert does not try again, jhq_reserve() does
    with refused(50 * MB, 1 << 50) as hit:
        got.append(x[:10])
    assert hit == [0]
    want.append(x[:10])
    _equal(_device(got, q, 100, gpu), want.search(q, 100))
    got.reserve(100)
    assert _used() - before > 80 * MB
    _equal(_device(got, q, 100, gpu), want.search(q, 100))


def test_host_search_shortage_keeps_the_reservation(gpu, flat):
    """A host search past the reserved k whose merged workspace is refused:
    it runs in batches of batch_size, and device searches keep theirs."""
    x, q = flat
    want, got = _flat(x), _flat(x)
    res = want.search(q, 100)
    with refused(50 * MB, 1 << 50) as hit:
        _equal(got.search(q, 100), res)
    assert hit == [1]
    _equal(_device(got, q, 10, gpu), want.search(q, 10))


def test_failed_setter_keeps_the_old_reservation(gpu, flat):
    x, q = flat
    ix = _flat(x)
    ix.reserve(100)
    res = ix.search(q, 100)
    with refused(2 * 10**6, 1 << 50, count=2) as hit:  # merged, then in batches of 16
        with pytest.raises(jg.JHQDeviceError):
            ix.set_alpha(10.0)
    assert hit == [2]
    _equal(_device(ix, q, 100, gpu), res)


@pytest.mark.parametrize("what", ["pool", "scratch"])
def test_insert_takes_the_room_of_merged_batches(gpu, flat, what):
    """An append whose new pool (or input scratch) is refused once succeeds
    in the room of the merged batches' workspaces."""
    x, q = flat
    want, got = _flat(x, 8000), _flat(x, 8000)
    want.reserve(100)
    got.reserve(100)
    want.append(x[8000:])
    n = want.pool()[1] * 32 + 16 if what == "pool" else 12000 * 128 * 4
    with refused(n, n + 1, count=1) as hit:
        got.append(x[8000:])
    assert hit == [1]
    la, lb = got.lists(), want.lists()
    assert all(np.array_equal(la[n], lb[n]) for n in la)
    _equal(_device(got, q, 100, gpu), want.search(q, 100))
