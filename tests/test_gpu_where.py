"""Bit#where / where2 / mask: compaction of bit positions on the device against
the oracle's where / mask on the same bits (integer work: bit-exact), over contiguous
arrays, views that start inside a word, strided and reversed views, and through
the reference's launcher symbols with a device index array and a cursor carried
across calls (narray/gen/tmpl_bit/where_kernel.cu:91-107, mask_kernel.cu:36-54)."""
import ctypes as C
import time

import numpy as np
import pytest

import kat_adjacent as K
from test_gpu_index import hip_runtime, queue_work, side_stream  # noqa: F401  (a fixture among them)

oracle = K.OracleEngine().o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 1000, 8191, 8192, 100003, (1 << 20) + 5, 1 << 25])
def test_where_matches_nonzero(n):
    import cumo_amd
    rng = np.random.default_rng(900 + n % 1000)
    density = rng.choice([0.02, 0.5, 0.97])
    h = (rng.random(n) < density).astype(np.uint8)
    b = cumo_amd.Bit.cast(h)
    got = b.where()
    assert isinstance(got, cumo_amd.Int32)
    assert (got.to_numpy() == oracle.where(h)).all()
    t, f = b.where2()
    assert (t.to_numpy() == oracle.where(h)).all() and (f.to_numpy() == oracle.where(h, invert=True)).all()
    if n > 40:
        for sl in (slice(3, None), slice(5, n - 7), slice(None, None, 2), slice(1, None, 3), slice(None, None, -1)):
            assert (b[sl].where().to_numpy() == oracle.where(h[sl])).all(), sl


def test_where_on_matrices_and_empty_results():
    import cumo_amd
    rng = np.random.default_rng(91)
    h = (rng.random((300, 777)) < 0.3).astype(np.uint8)
    b = cumo_amd.Bit.cast(h)
    assert (b.where().to_numpy() == oracle.where(h)).all()
    # views that do not contract to one run: one launch sequence per row, the cursor carried on the device
    for key in ((slice(5, 200), slice(7, 600)), (slice(None), slice(None, None, 3)), (slice(None, None, -1), slice(None))):
        assert (b[key].where().to_numpy() == oracle.where(h[key])).all(), key
    assert (b.transpose().where().to_numpy() == oracle.where(h.T)).all()
    z = cumo_amd.Bit.cast(np.zeros(5000, dtype=np.uint8))
    assert z.where().to_numpy().shape == (0,)
    assert (z.where2()[1].to_numpy() == np.arange(5000)).all()


@pytest.mark.parametrize("tname,dt", [("SFloat", np.float32), ("DFloat", np.float64), ("Int32", np.int32)])
def test_mask_gathers_in_row_major_order(tname, dt):
    import cumo_amd
    cls = getattr(cumo_amd, tname)
    rng = np.random.default_rng(92)
    for shape in [(7,), (100003,), (300, 777), (5, 6, 130)]:
        hx = rng.integers(-1000, 1000, size=shape).astype(dt)
        hm = (rng.random(shape) < 0.4)
        x, m = cls.cast(hx), cumo_amd.Bit.cast(hm.astype(np.uint8))
        got = m.mask(x)
        assert isinstance(got, cls) and (got.to_numpy() == oracle.mask(hm, hx)).all(), shape
        assert (x[m].to_numpy() == oracle.mask(hm, hx)).all()
        if len(shape) == 2:
            # the masked array as a view: transposed, strided; the mask made from a comparison
            assert (m.transpose().mask(x.transpose()).to_numpy() == hx.T[hm.T]).all()
            assert (m[::2, 1::3].mask(x[::2, 1::3]).to_numpy() == hx[::2, 1::3][hm[::2, 1::3]]).all()
            gt = x > 0
            assert (x[gt].to_numpy() == hx[hx > 0]).all()
    with pytest.raises(cumo_amd.ShapeError):
        cumo_amd.Bit.cast(np.ones(4, dtype=np.uint8)).mask(cls.cast(np.zeros(5, dtype=dt)))


def test_where_and_mask_launchers_with_index_arrays_and_a_carried_cursor():
    from cumo_amd import _lib
    from test_gpu_raw_abi import dev, fetch, free
    rng = np.random.default_rng(93)
    nbits = 50000
    h = (rng.random(nbits) < 0.35).astype(np.uint8)
    words = np.packbits(h, bitorder="little").view(np.uint32) if nbits % 32 == 0 else np.frombuffer(
        np.packbits(np.concatenate([h, np.zeros(32 - nbits % 32, np.uint8)]), bitorder="little").tobytes(), dtype=np.uint32)
    pw = dev(words)
    new = _lib.fn("cumo_bit_where_scratch_new", C.c_void_p, [])
    where = _lib.fn("cumo_bit_where_kernel_launch", None,
                    [C.c_void_p, C.c_size_t, C.c_ssize_t, C.c_void_p, C.c_uint64, C.c_int, C.c_void_p, C.c_size_t, C.c_uint64, C.c_void_p])
    scratch = _lib.call(new)
    # two runs, the second through a device index array, both appended to one output
    n1, p1 = 20000, 13
    idx = rng.permutation(nbits - 100)[:15000].astype(np.uint64)
    pidx = dev(idx)
    want = np.concatenate([oracle.where(h[p1:p1 + n1]), n1 + oracle.where(h[7 + idx.astype(np.int64)])])
    pout = dev(np.full(want.size + 4, -1, dtype=np.int64))
    _lib.call(where, pw, p1, 1, None, n1, 0, pout, 8, 0, scratch)
    _lib.call(where, pw, 7, 0, pidx, idx.size, 0, pout, 8, n1, scratch)
    got = fetch(pout, (want.size + 4,), np.int64)
    assert (got[:want.size] == want).all() and (got[want.size:] == -1).all()
    # the zeros keep their own cursor (scratch word 1): a strided run, every third bit
    n3 = 9000
    wantz = oracle.where(h[5:5 + 3 * n3:3] == 0)
    pz = dev(np.full(wantz.size + 2, -1, dtype=np.int32))
    _lib.call(where, pw, 5, 3, None, n3, 1, pz, 4, 0, scratch)
    gz = fetch(pz, (wantz.size + 2,), np.int32)
    assert (gz[:wantz.size] == wantz).all() and (gz[wantz.size:] == -1).all()
    # mask: positions of the masked array's elements, base 40 bytes and 8 bytes apart
    _lib.lib.cumo_cuda_runtime_free(scratch)
    scratch = _lib.call(new)
    mask = _lib.fn("cumo_bit_mask_kernel_launch", None,
                   [C.c_void_p, C.c_size_t, C.c_ssize_t, C.c_void_p, C.c_uint64, C.c_void_p, C.c_size_t, C.c_ssize_t, C.c_void_p, C.c_void_p])
    wantm = 40 + 8 * oracle.where(h[p1:p1 + n1])
    pm = dev(np.zeros(wantm.size + 1, dtype=np.uint64))
    _lib.call(mask, pw, p1, 1, None, n1, pm, 40, 8, None, scratch)
    gm = fetch(pm, (wantm.size + 1,), np.uint64)
    assert (gm[:wantm.size] == wantm.astype(np.uint64)).all() and gm[wantm.size] == 0
    _lib.lib.cumo_cuda_runtime_free(scratch)
    free(pw, pidx, pout, pz, pm)


@pytest.mark.parametrize("nbits", [1, 31, 8193, 1 << 20, (1 << 25) + 77])
def test_count_then_place_launchers(nbits):
    """The two-launch form for a caller that sizes the result in between: block counts, read back and
    added up, then the placement of positions (set or clear bits, 4- or 8-byte) or of elements."""
    from cumo_amd import _lib
    from test_gpu_raw_abi import dev, fetch, free
    rng = np.random.default_rng(nbits)
    lead = 37                                       # the run starts inside a word
    h = (rng.random(lead + 3 * nbits if nbits < 10000 else lead + nbits) < 0.4).astype(np.uint8)
    pad = (-h.size) % 32
    words = np.frombuffer(np.packbits(np.concatenate([h, np.zeros(pad, np.uint8)]), bitorder="little").tobytes(), dtype=np.uint32)
    pw = dev(words)
    blocks = _lib.fn("cumo_hip_bit_where_blocks", C.c_size_t, [C.c_uint64])
    count = _lib.fn("cumo_hip_bit_where_count_kernel_launch", None, [C.c_void_p, C.c_size_t, C.c_ssize_t, C.c_uint64, C.c_int, C.c_void_p])
    place = _lib.fn("cumo_hip_bit_where_place_kernel_launch", None,
                    [C.c_void_p, C.c_size_t, C.c_ssize_t, C.c_uint64, C.c_int, C.c_void_p, C.c_void_p, C.c_ssize_t, C.c_size_t, C.c_void_p])
    nb = blocks(nbits)
    assert 1 <= nb <= 1024 and blocks(0) == 0
    x = rng.standard_normal(nbits).astype(np.float32)
    xd = rng.standard_normal(2 * nbits)             # every second double
    px, pxd = dev(x), dev(xd)
    cases = [(1, 0, 8), (1, 1, 4)] + ([(3, 0, 4)] if nbits < 10000 else [])
    for step, invert, elmsz in cases:
        run = h[lead:lead + step * nbits:step]
        hits = np.flatnonzero(run == (0 if invert else 1))
        pc = dev(np.full(nb + 1, 12345, dtype=np.uint64))
        _lib.call(count, pw, lead, step, nbits, invert, pc)
        counts = fetch(pc, (nb + 1,), np.uint64)
        assert int(counts[:nb].sum()) == hits.size and counts[nb] == 12345
        it = np.int64 if elmsz == 8 else np.int32
        po = dev(np.full(hits.size + 3, -1, dtype=it))
        _lib.call(place, pw, lead, step, nbits, invert, pc, None, 0, elmsz, po)
        got = fetch(po, (hits.size + 3,), it)
        assert (got[:hits.size] == hits).all() and (got[hits.size:] == -1).all()
        if step == 1 and not invert:
            pv = dev(np.full(hits.size + 1, 7.0, dtype=np.float32))
            _lib.call(place, pw, lead, 1, nbits, 0, pc, px, 4, 4, pv)
            gv = fetch(pv, (hits.size + 1,), np.float32)
            assert (gv[:hits.size] == x[hits]).all() and gv[hits.size] == 7.0
            pv8 = dev(np.full(hits.size + 1, 7.0, dtype=np.float64))
            _lib.call(place, pw, lead, 1, nbits, 0, pc, pxd, 16, 8, pv8)
            gv8 = fetch(pv8, (hits.size + 1,), np.float64)
            assert (gv8[:hits.size] == xd[::2][hits]).all() and gv8[hits.size] == 7.0
            free(pv, pv8)
        free(pc, po)
    free(pw, px, pxd)


@pytest.mark.parametrize("lead", [64, 37])   # a run that starts on a word, and inside one
@pytest.mark.parametrize("nbits", [1, 33, 8192, 8193, 1 << 15, (1 << 15) + 1, (1 << 20) - 5, (1 << 25) + 32 * 1024 + 77])
def test_counts_of_shares_on_device_and_host(nbits, lead):
    """The blocks of the count take four placing blocks' shares each: every share's count, on the device and on
    the host, at sizes that end inside a share, a block and a word; and their sum, which sizes the
    positions, of the set and of the clear bits, of the run and of every third bit of it."""
    from cumo_amd import Bit, _lib
    from test_gpu_raw_abi import dev, fetch, free
    rng = np.random.default_rng(nbits)
    h = (rng.random(lead + nbits) < 0.4).astype(np.uint8)
    words = np.frombuffer(np.packbits(np.concatenate([h, np.ones((-h.size) % 32, np.uint8)]), bitorder="little").tobytes(), dtype=np.uint32)
    pw = dev(words)
    nb = _lib.fn("cumo_hip_bit_where_blocks", C.c_size_t, [C.c_uint64])(nbits)
    to_host = _lib.fn("cumo_hip_bit_where_count_to_host", C.c_int, [C.c_void_p, C.c_size_t, C.c_ssize_t, C.c_uint64, C.c_int, C.c_void_p, C.c_void_p])
    chunks = -(-nbits // 32)
    share = -(-chunks // nb) * 32
    for invert in (0, 1):
        run = h[lead:] ^ invert
        want = np.array([run[k * share:(k + 1) * share].sum(dtype=np.uint64) for k in range(nb)], dtype=np.uint64)
        pc, on_host = dev(np.full(nb + 1, 12345, dtype=np.uint64)), np.full(nb + 1, 777, dtype=np.uint64)
        _lib.call(to_host, pw, lead, 1, nbits, invert, pc, on_host.ctypes.data)
        counts = fetch(pc, (nb + 1,), np.uint64)
        assert (counts[:nb] == want).all() and counts[nb] == 12345 and (on_host[:nb] == want).all() and on_host[nb] == 777
        free(pc)
    free(pw)
    for b, run in ((Bit.cast(h)[lead:], h[lead:]), (Bit.cast(h)[lead::3], h[lead::3])):
        for got, want in zip(b.where2(), (np.flatnonzero(run), np.flatnonzero(run == 0))):
            assert got.shape == want.shape and (got.to_numpy() == want).all()


def test_where_and_mask_into_a_given_result():
    """A result array of exactly the count's length is written in place; any other length is a shape error."""
    import ctypes as C
    import cumo_amd
    from cumo_amd import _lib
    rng = np.random.default_rng(21)
    x = rng.standard_normal((50, 70)).astype(np.float32)
    d = cumo_amd.SFloat.cast(x)
    m = d > 0.25
    want_pos = oracle.where(x > np.float32(0.25)).astype(np.int32)
    pos = cumo_amd.Int32.zeros(len(want_pos))
    md, zd = m._desc(), pos._desc()
    _lib.call(_lib.lib.cumo_hip_na_where, C.byref(md), 0, C.byref(zd))
    assert (pos.to_numpy() == want_pos).all()
    vals = cumo_amd.SFloat.zeros(len(want_pos))
    xd, vd = d._desc(), vals._desc()
    _lib.call(_lib.lib.cumo_hip_na_mask, C.byref(md), C.byref(xd), C.byref(vd))
    assert (vals.to_numpy() == x.ravel()[want_pos]).all()
    short = cumo_amd.Int32.zeros(len(want_pos) - 1)
    sd = short._desc()
    with pytest.raises(cumo_amd.ShapeError):
        _lib.call(_lib.lib.cumo_hip_na_where, C.byref(md), 0, C.byref(sd))


@pytest.mark.parametrize("tname,dt", [("SFloat", np.float32), ("DFloat", np.float64), ("Int32", np.int32)])
def test_mask_of_single_runs_with_offsets_steps_and_reversal(tname, dt):
    """Mask and masked array that each walk as one run (sliced alike) are compacted in place of
    positions: starts inside a word, steps other than 1, a reversed run, different steps on the two sides."""
    import cumo_amd
    cls = getattr(cumo_amd, tname)
    rng = np.random.default_rng(93)
    n = 100003
    hx = rng.integers(-1000, 1000, size=n).astype(dt)
    hm = rng.random(n) < 0.35
    x, m = cls.cast(hx), cumo_amd.Bit.cast(hm.astype(np.uint8))
    for sl in (slice(7, None), slice(33, n - 9), slice(None, None, 2), slice(5, None, 3), slice(None, None, -1), slice(n - 4, 2, -5)):
        got = m[sl].mask(x[sl]).to_numpy()
        assert (got == oracle.mask(hm[sl], hx[sl])).all(), sl
    # the mask contiguous, the masked array every other element of a longer one
    hy = rng.integers(-1000, 1000, size=2 * n).astype(dt)
    y = cls.cast(hy)
    assert (m.mask(y[::2]).to_numpy() == oracle.mask(hm, hy[::2])).all()
    assert (m[::-1].mask(y[1::2]).to_numpy() == oracle.mask(hm[::-1], hy[1::2])).all()
    # nothing set, everything set
    none, every = cumo_amd.Bit.cast(np.zeros(n, dtype=np.uint8)), cumo_amd.Bit.cast(np.ones(n, dtype=np.uint8))
    assert none.mask(x).to_numpy().shape == (0,)
    assert (every.mask(x).to_numpy() == hx).all()


def test_where_beyond_two_to_the_32_elements_answers_int64():
    """More than 2^32 - 1 elements: positions no longer fit Int32 (gen/tmpl_bit/where.c:104-110
    picks Int64 then). The bits are set on the device buffer word by word; no host array of
    that length is made."""
    import ctypes as C
    import cumo_amd
    from cumo_amd import _lib
    n = (1 << 32) + 70
    b = cumo_amd.Bit.zeros(n)
    want = [5, (1 << 31) + 3, (1 << 32) - 1, 1 << 32, (1 << 32) + 69]
    for pos in want:
        word = np.array([1 << (pos % 32)], dtype=np.uint32)
        assert _lib.call(_lib.lib.cumo_hip_copy_from_host, b._buf.ptr + (pos // 32) * 4, word.ctypes.data, 4) == 0
    assert int(b.count_true()) == len(want)
    got = b.where()
    assert isinstance(got, cumo_amd.Int64) and got.to_numpy().tolist() == want
    # a view that starts beyond 2^32 bits
    tail = b[(1 << 32) - 2:]
    assert tail.where().to_numpy().tolist() == [1, 2, 71]
    assert int(tail.count_false()) == 72 - 3
    del b, tail, got
    cumo_amd.MemoryPool.free_all_blocks()


@pytest.mark.parametrize("tname,dt", [("SFloat", np.float32), ("DFloat", np.float64), ("Int32", np.int32)])
def test_mask_around_whole_vectors_chunks_and_tiles(tname, dt):
    """A contiguous run is read in vectors (4 or 2 elements), chunks (32), a wave's 1024 and a block's 4096
    elements, over 1024 blocks' stretches at most; masks and runs that start off their boundaries."""
    import cumo_amd
    cls = getattr(cumo_amd, tname)
    rng = np.random.default_rng(94)
    for n in (1, 2, 3, 5, 31, 33, 1023, 1025, 4095, 4097, 8191, 8193, (1 << 23) + 4099):
        hx = rng.integers(-1000, 1000, size=n + 7).astype(dt)
        x = cls.cast(hx)
        for density in (0.0, 0.003, 0.4, 1.0):
            hm = rng.random(n + 7) < density
            m = cumo_amd.Bit.cast(hm.astype(np.uint8))
            for a, b in ((0, 0), (3, 1), (1, 5)) if n < 100000 else ((0, 0), (3, 1)):
                got = m[a:a + n].mask(x[b:b + n]).to_numpy()
                want = hx[b:b + n][hm[a:a + n]]
                assert got.shape == want.shape and (got == want).all(), (n, density, a, b)


@pytest.mark.parametrize("tname,dt", [("SFloat", np.float32), ("DFloat", np.float64)])
def test_masks_on_either_side_of_one_hit_in_forty(tname, dt):
    """Where elements are placed one by one and where they are packed as vectors; hits spread out and all at one end."""
    import cumo_amd
    rng = np.random.default_rng(95)
    for n in (39, 40, 80, 4000, 400040):
        x = rng.integers(-1000, 1000, size=n).astype(dt)
        dx = getattr(cumo_amd, tname).cast(x)
        for hits in (max(n // 40 - 1, 0), n // 40, n // 40 + 1):
            for spread in (True, False):
                h = np.zeros(n, np.uint8)
                h[rng.permutation(n)[:hits] if spread else np.arange(n - hits, n)] = 1
                assert (dx[cumo_amd.Bit.cast(h)].to_numpy() == x[h != 0]).all(), (n, hits, spread)


def masks(k):
    import cumo_amd
    rng = np.random.default_rng(700 + k)
    h = (rng.random(100000) < rng.random()).astype(np.uint8)
    return h, cumo_amd.Bit.cast(h)


def test_an_error_left_by_an_earlier_call_is_reported_and_leaves_no_kernel_behind():
    import cumo_amd
    hip = hip_runtime()
    long = cumo_amd.DFloat.cast(np.linspace(0.1, 2, 1 << 24))
    many = [masks(k) for k in range(12)]
    many[0][1].where()
    cumo_amd.synchronize()
    queue_work(hip, long)
    hip.hipSetDevice(1 << 20)          # no such device: refused by the runtime, which keeps the error for the thread
    with pytest.raises(RuntimeError):
        many[0][1].where()
    # (a count still to come from the refused call's kernel would be taken for one of these)
    for h, b in many[1:]:
        assert (b.where().to_numpy() == oracle.where(h)).all()


def test_a_stream_under_capture_is_refused_at_once():
    from cumo_amd import _lib
    hip = hip_runtime()
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    h, b = masks(0)
    took = []
    for _ in range(3):
        # (left alone afterwards: the runtime goes on to take a stream whose capture has failed for one under capture)
        stream = _lib.lib.cumo_hip_stream_create()
        _lib.lib.cumo_hip_set_stream(stream)
        assert (b.where().to_numpy() == oracle.where(h)).all()
        assert hip.hipStreamBeginCapture(stream, 2) == 0           # (relaxed: only the wait is refused)
        begin = time.perf_counter()
        with pytest.raises(RuntimeError):
            b.where()
        took.append(time.perf_counter() - begin)
        graph = C.c_void_p()
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) != 0 and not graph.value
        hip.hipGetLastError()
        _lib.lib.cumo_hip_set_stream(None)
    assert min(took) < 1.5e-3          # without the 2 ms that a running stream is looked at
    assert (b.where().to_numpy() == oracle.where(h)).all()


@pytest.mark.parametrize("side", [False, True])
def test_masks_behind_more_work_than_the_host_looks_for(side, side_stream):
    import cumo_amd
    from cumo_amd import _lib
    hip = hip_runtime()
    if side:
        _lib.lib.cumo_hip_set_stream(side_stream)
    long = cumo_amd.DFloat.cast(np.linspace(0.1, 2, 1 << 24))
    x = np.arange(100000, dtype=np.float32)
    dx = cumo_amd.SFloat.cast(x)
    for k in range(3):
        h, b = masks(k)
        begin = time.perf_counter()
        queue_work(hip, long)
        got = dx[b]
        assert time.perf_counter() - begin > 2e-3                  # (it was the runtime's wait that ended)
        queue_work(hip, long)
        at = b.where()
        assert (got.to_numpy() == x[h != 0]).all() and (at.to_numpy() == oracle.where(h)).all()
