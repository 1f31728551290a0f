"""The native object layer (cumo_amd/native/arrays.cpp): the same arrays, bit for bit, as the general Python methods give, for every
form it takes, and what it leaves to them."""
import copy
import gc
import threading

import numpy as np
import pytest

import cumo_amd
from cumo_amd import Bit, DFloat, Int32, MemoryPool, NMath, SFloat, _lib, _native
from cumo_amd.narray import NArray

pytestmark = pytest.mark.gpu
TYPES = {"sfloat": SFloat, "dfloat": DFloat, "int32": Int32}


def same(a, b):
    if isinstance(a, (tuple, list)):
        return len(a) == len(b) and all(same(p, q) for p, q in zip(a, b))
    if not isinstance(a, NArray):
        return type(a) is type(b) and a == b
    return (type(a) is type(b) and a.shape == b.shape and a._strides == b._strides and a._offset == b._offset == 0
            and a._buf.nbytes == b._buf.nbytes and a.to_numpy().tobytes() == b.to_numpy().tobytes())


def arrays(tname, shape):
    rng = np.random.default_rng(3)
    cls = TYPES[tname]
    x, y = [cls.cast(rng.integers(1, 50, size=shape).astype(cls.np_dtype)) for _ in range(2)]
    return x, y


@pytest.mark.parametrize("tname", sorted(TYPES))
@pytest.mark.parametrize("shape", [(7,), (1, 1), (5, 9), (3, 4, 6), (0, 4)])
def test_native_calls_answer_like_the_general_methods(tname, shape):
    x, y = arrays(tname, shape)
    views = [(x, y), (x.transpose(), y.transpose()), (x.reverse(0), y)]
    for v, w in views:
        for other in (w, 3, 2.0, True, np.float32(2), DFloat.cast(w) if v.size else w):
            for left in (False, True):
                assert same(_native.binary(v, other, "add", left), v._binary(other, "add", left))
            if not isinstance(other, float) or tname != "int32":
                assert same(_native.binary(v, other, "copysign" if v.is_float else "mod", False),
                            v._binary(other, "copysign" if v.is_float else "mod", False))
            assert same(_native.compare(v, other, "gt"), v._compare(other, "gt"))
        assert same(_native.unary(v, "abs"), v._unary("abs"))
        assert same(NMath.sqrt(v), NMath._call1("sqrt", v))
        if not v.size:
            with pytest.raises(cumo_amd.ShapeError):
                v.sum(axis=0) if v.shape[0] else v.sum()
            continue
        for axis in (None, 0, -1, (0,), np.int64(0), [0]):
            for name in ("sum", "max", "minmax", "argmin"):
                for keep in (False, True):
                    assert same(_native.reduce(v, name, axis, keep, False), v._reduce(name, axis, keep, False))
            assert same(_native.mulsum(v, w, axis, False, False), v._mulsum(w, axis, False, False))
            assert same(_native.cum(v, "cumsum", axis, False), v._cum("cumsum", axis, False))
        a, b = v > 20, w > 20
        assert same(a & b, a._bit_op2(b, "and"))
        for axis in (None, 0, -1):
            assert same(a.count_true(axis=axis), a._count(False, axis, False))
            assert same(a.count_false(axis=axis, keepdims=True), a._count(True, axis, True))
    empty = Bit(0, 4)
    assert empty.count_true() == 0 and empty.count_true(axis=0) == 0


@pytest.mark.parametrize("tname", sorted(TYPES) + ["int64"])
def test_rows_by_position_answer_like_the_general_form(tname):
    rng = np.random.default_rng(5)
    x = TYPES[tname].cast(rng.integers(-99, 99, size=(7, 6, 5)).astype(TYPES[tname].np_dtype)) if tname in TYPES else \
        DFloat.cast(rng.standard_normal((7, 6, 5))).argmax(axis=2)
    for v in (x, x.transpose(), x.reverse(0), x.reverse(1), x[::2], x[1], x[:, 1:4], x[3:4], x.reshape(x.size), x.reverse(0)[1::3]):
        n = v.shape[0]
        for k in (np.arange(n), np.array([0]), np.array([-1, 0, n - 1, -n, 0]), rng.integers(-n, n, 300), rng.integers(0, n, 9000)):
            got, want = _native.take(v, k), v._gather(v._expand_key(k))
            assert same(got, want) and same(v[k], want)
        one = np.zeros(4, np.int64)
        # what it leaves to the general form, and what that refuses
        for k in (one.astype(np.int32), one.astype(np.uint64), one.astype(float), one[::2], one[:0], one.reshape(2, 2), one.astype(">i8"),
                  np.array(0), np.array([0, n]), np.array([-n - 1])):
            assert _native.take(v, k) is None
        for k in (np.array([0, n]), np.array([-n - 1]), one.reshape(2, 2), np.array([0.5])):
            with pytest.raises(IndexError):
                v[k]
        assert same(v[one.astype(np.int32)], v._gather(v._expand_key(one)))
        assert v[one[:0]].size == 0
    with pytest.raises(TypeError):
        Bit(8)[np.array([0])]
    assert _native.take(SFloat(0, 3), np.array([0])) is None and _native.take(SFloat(3, 0), np.array([0])) is None
    with _lib.record() as calls:
        x[np.array([1, 0])]
    assert len(calls) > 0


@pytest.mark.parametrize("tname", sorted(TYPES))
def test_selections_of_a_derived_class_are_of_that_class(tname):
    class Derived(TYPES[tname]):
        pass
    h = np.arange(24).reshape(4, 6).astype(TYPES[tname].np_dtype)
    w = Derived.cast(h)
    for key in (slice(1, 3), [0, 2], np.array([0, 2]), np.array([0, 2], dtype=np.int32), np.array([-1, 0, 3]), (np.array([1]), slice(None))):
        got = w[key]
        assert type(got) is Derived
        assert (got.to_numpy() == h[key]).all()
    assert type(w.reshape(24)[np.array([5])]) is Derived
    assert type(TYPES[tname].cast(h)[np.array([0, 2])]) is TYPES[tname]


def test_what_is_refused_stays_refused_and_leaks_nothing():
    x = SFloat.cast(np.ones((4, 5), np.float32))
    i = Int32.cast(np.zeros(6, np.int32))
    one = Int32.cast(np.ones(6, np.int32))
    MemoryPool.free_all_blocks()
    gc.collect()
    before = MemoryPool.used_bytes()
    for f, error in ((lambda: x + SFloat(3, 3), cumo_amd.ShapeError), (lambda: x.sum(axis=2), _lib.DimensionError),
                     (lambda: x.sum(axis=(0, -3)), _lib.DimensionError), (lambda: one / i, ZeroDivisionError),
                     (lambda: one / 0, ZeroDivisionError), (lambda: x + "a", TypeError), (lambda: x + 10 ** 400, OverflowError),
                     (lambda: NMath.exp(1.0), TypeError), (lambda: x & 1, TypeError), (lambda: (x > 0) & x, TypeError),
                     (lambda: setattr(x, "shape", 3), TypeError), (lambda: setattr(x, "_buf", 3), TypeError)):
        for _ in range(3):
            with pytest.raises(error):
                f()
    gc.collect()
    assert MemoryPool.used_bytes() == before
    c = copy.copy(x)
    assert c.shape == x.shape and c._ptr() == x._ptr()
    del x
    assert c.to_numpy().sum() == 20


def test_recorded_calls_come_from_the_general_methods():
    x = DFloat.cast(np.arange(6.0))
    with _lib.record() as calls:
        y = x + 1.0
        t = (y * y).sum()
    assert len(calls) == 3 and len(calls.keep) == 1     # y * y died inside the block
    x.fill(2.0)
    _lib.replay(calls)
    assert float(t) == 54.0 and (x + 1.0).to_numpy().tolist() == [3.0] * 6


def test_threads_call_and_release_at_once():
    bad = []

    def work(k):
        x = DFloat.cast(np.full(1000 + k, float(k)))
        for j in range(200):
            y = (x + float(j)) * 2.0
            if j % 50 == 0 and float(y.sum()) != 2.0 * (k + j) * (1000 + k):
                bad.append((k, j))
            try:
                x + DFloat(3)
                bad.append("no error")
            except cumo_amd.ShapeError:
                pass

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad


@pytest.mark.parametrize("cls", [SFloat, DFloat, Int32, cumo_amd.Int64, cumo_amd.UInt64, Bit])
def test_a_deep_copy_has_memory_of_its_own(cls):
    h = (np.arange(60).reshape(5, 12) % 2).astype(cls.np_dtype or np.uint8)
    x = cls.cast(h)
    for v, want in ((x, h), (x.transpose(), h.T), (x[1:, 3:9], h[1:, 3:9])):
        y = copy.deepcopy({"a": [v, v]})["a"]
        assert y[0] is y[1] and type(y[0]) is cls and y[0]._ptr() != v._ptr()
        assert (y[0].to_numpy() == want).all()
        _lib.call(_lib.lib.cumo_hip_memset, y[0]._buf.ptr, 0xff, y[0]._buf.nbytes)
        assert (v.to_numpy() == want).all()
        del y
    assert (x.to_numpy() == h).all()
