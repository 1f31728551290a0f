"""softmax and layernorm along the last dimension: the one-launch form against the
chain of array operations it stands for (run on the device) and against the same
chain on the CPU oracle. Elementwise steps are identical in both; the two row
sums associate differently, so the bar is the float-reduction bar of the parity
contract carried through the division: rel 1e-5*log2(n) SFloat, 1e-12*log2(n)
DFloat."""
import numpy as np
import pytest

import kat_adjacent as K

pytestmark = pytest.mark.gpu
oracle = K.OracleEngine().o


def chain_softmax(m, x):
    mx = x.max(axis=-1, keepdims=True)
    e = m.NMath.exp(x - mx)
    return e / e.sum(axis=-1, keepdims=True)


def chain_layernorm(m, x, eps):
    return (x - x.mean(axis=-1, keepdims=True)) / m.NMath.sqrt(x.var(axis=-1, keepdims=True) + eps)


def oracle_softmax(h):
    mx = oracle.reduce("max", h, axis=h.ndim - 1, keepdims=True)
    e = oracle.unary("exp", oracle.binary("sub", h, np.ascontiguousarray(np.broadcast_to(mx, h.shape))))
    s = oracle.reduce("sum", e, axis=h.ndim - 1, keepdims=True)
    return oracle.binary("div", e, np.ascontiguousarray(np.broadcast_to(s, h.shape)))


def close(got, want, n, dt, what):
    tol = (1e-5 if dt == np.float32 else 1e-12) * max(1.0, np.log2(max(n, 2)))
    g, w = got.astype(np.float64), want.astype(np.float64)
    nan = np.isnan(w)
    assert (np.isnan(g) == nan).all(), what
    err = np.abs(g - w)[~nan]
    bound = tol * np.maximum(np.abs(w[~nan]), 1e-30) + tol * 1e-3
    assert (err <= bound).all(), (what, float(err.max()))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_softmax_matches_the_chain(dt):
    import cumo_amd as m
    cls = m.SFloat if dt == np.float32 else m.DFloat
    rng = np.random.default_rng(61)
    # (rows that end in part of a 128-bit vector, and so start off a 16-byte boundary: 1001, 4095, 13, 131, 7)
    for shape in [(1, 4), (5, 8), (33, 64), (100, 512), (7, 1000), (3, 4, 2048), (9, 4096), (2, 16384), (4, 20000), (6, 7), (2, 3, 5, 128),
                  (7, 1001), (37, 4095), (50, 13), (19, 131), (3, 16383), (5, 4094)]:
        h = (rng.standard_normal(shape) * 2).astype(dt)
        x = cls.cast(h)
        got = m.Fused.softmax(x).to_numpy()
        n = shape[-1]
        close(got, chain_softmax(m, x).to_numpy(), n, dt, (shape, "device chain"))
        if np.prod(shape) <= 200000:
            close(got, oracle_softmax(h), n, dt, (shape, "oracle chain"))
        assert np.allclose(got.astype(np.float64).sum(axis=-1), 1.0, rtol=0, atol=1e-5 if dt == np.float32 else 1e-12)
    # rows that are views: every other row, and a column window that stays 16-byte aligned
    h = (rng.standard_normal((40, 256)) * 2).astype(dt)
    x = cls.cast(h)
    for key in ((slice(None, None, 2), slice(None)), (slice(3, 30), slice(64, 192)), (slice(None), slice(1, 200)), (slice(None), slice(None, None, 2))):
        close(m.Fused.softmax(x[key]).to_numpy(), chain_softmax(m, x[key]).to_numpy(), h[key].shape[-1], dt, key)
    # special values: a NaN poisons its row, -inf entries get weight 0, a row of equal values is uniform
    h = np.zeros((4, 64), dtype=dt)
    h[0, 5] = np.nan
    h[1, :] = -np.inf
    h[1, 7] = 3.0
    h[2, :] = 7.5
    h[3, :] = rng.standard_normal(64)
    got = m.Fused.softmax(cls.cast(h)).to_numpy()
    want = chain_softmax(m, cls.cast(h)).to_numpy()
    assert np.isnan(got[0]).all() and np.isnan(want[0]).all()
    assert got[1, 7] == 1.0 and (np.delete(got[1], 7) == 0).all()
    assert (got[2] == dt(1.0) / dt(64.0)).all()
    close(got[3:], want[3:], 64, dt, "ordinary row")


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_layernorm_matches_the_chain(dt):
    import cumo_amd as m
    cls = m.SFloat if dt == np.float32 else m.DFloat
    rng = np.random.default_rng(62)
    for shape in [(3, 4), (5, 8), (33, 64), (100, 512), (7, 1000), (64, 4096), (3, 16384), (4, 20000), (6, 7), (2, 3, 128),
                  (7, 1001), (37, 4095), (50, 13), (19, 131), (3, 16383), (5, 4094)]:
        h = (rng.standard_normal(shape) * 3 + 1).astype(dt)
        x = cls.cast(h)
        got = m.Fused.layernorm(x, 1e-5).to_numpy()
        want = chain_layernorm(m, x, 1e-5).to_numpy()
        n = shape[-1]
        # the chain's own var is one-pass (Chan); both lie within the bar of the exact statistics
        hd = h.astype(np.float64)
        exact = (hd - hd.mean(axis=-1, keepdims=True)) / np.sqrt(hd.var(axis=-1, ddof=1, keepdims=True) + dt(1e-5))
        tol = (1e-5 if dt == np.float32 else 1e-12) * max(1.0, np.log2(n))
        assert np.abs(got - exact).max() <= tol * 8, (shape, float(np.abs(got - exact).max()))
        assert np.abs(want - exact).max() <= tol * 8, (shape, "chain")
    # a row of one element has no variance: NaN from both
    one = cls.cast(np.array([[2.0], [3.0]], dtype=dt))
    assert np.isnan(m.Fused.layernorm(one).to_numpy()).all() and np.isnan(chain_layernorm(m, one, 1e-5).to_numpy()).all()


# Rows beyond the registers of 256 lanes, which hold 16384 SFloat / 4096 DFloat: a block of 512 lanes up to
# 32768 / 16384 elements, of 1024 lanes up to 65536 / 32768 where there are more than 64 rows, and pieces of 8192 / 4096 elements in
# two launches beyond and for fewer rows. Lengths at those edges, a last piece of one element, a last vector that is partly there.
LONG_ROWS = [(3, 4097), (3, 8193), (3, 16385), (5, 32768), (3, 32769), (2, 65533), (3, 65536), (300, 16390), (3, 65537), (7, 70001), (2, 3, 131073), (1, 1 << 20),
             (64, 16385), (65, 16385), (65, 32768), (64, 32769), (65, 32769), (65, 65533), (65, 65536)]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("shape", LONG_ROWS)
def test_long_rows_match_64_bit_arithmetic(dt, shape):
    import cumo_amd as m
    cls = m.SFloat if dt == np.float32 else m.DFloat
    n = shape[-1]
    h = (np.random.default_rng(n).standard_normal(shape) * 2 + 0.5).astype(dt)
    x = cls.cast(h)
    w = h.astype(np.longdouble)
    e = np.exp(w - w.max(axis=-1, keepdims=True))
    # per element: the difference's rounding (up to half an ulp of ~12), exp, the sum (pairwise, some 2^-23) and the division
    tol = 16 * np.finfo(dt).eps
    want = e / e.sum(axis=-1, keepdims=True)
    assert (np.abs(m.Fused.softmax(x).to_numpy() - want) <= tol * want + np.finfo(dt).tiny).all()
    c = w - w.mean(axis=-1, keepdims=True)
    want = c / np.sqrt((c * c).sum(axis=-1, keepdims=True) / (n - 1) + dt(1e-5))
    assert np.abs(m.Fused.layernorm(x, 1e-5).to_numpy() - want).max() <= tol


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("rows,n", [(6, 20001), (6, 70001), (140, 20001), (140, 40001)])   # (140: a block of 1024 lanes each, DFloat / SFloat)
def test_long_rows_special_values_views_and_overlap(dt, rows, n):
    import cumo_amd as m
    cls = m.SFloat if dt == np.float32 else m.DFloat
    h = (np.random.default_rng(n).standard_normal((rows, n)) * 2).astype(dt)
    h[0, n - 1] = np.nan
    h[1, :] = -np.inf      # whole pieces of -inf, one of them with a number
    h[1, 17] = 3.0
    h[2, 11] = np.inf
    h[3, :] = -np.inf
    h[4, :] = 7.5
    x = cls.cast(h)
    for key in (slice(None), slice(1, None, 2), slice(None, None, -1)):
        got = m.Fused.softmax(x[key]).to_numpy()
        want = chain_softmax(m, x[key]).to_numpy()
        close(got, want, n, dt, ("softmax", key))
        got = m.Fused.layernorm(x[key], 1e-5).to_numpy()
        assert (np.isnan(got) == np.isnan(chain_layernorm(m, x[key], 1e-5).to_numpy())).all()
    want = m.Fused.softmax(x).to_numpy()
    assert want[1, 17] == 1.0 and np.count_nonzero(want[1]) == 1 and np.isnan(want[[0, 2, 3]]).all()


@pytest.mark.parametrize("rows,n", [(4, 20001), (4, 70001), (65, 40001)])
def test_long_rows_into_their_operand_and_into_memory_that_overlaps_it(rows, n):
    import ctypes as C
    import cumo_amd as m
    from cumo_amd import _lib
    h = (np.random.default_rng(n).standard_normal((rows + 1, n)) * 2).astype(np.float32)
    want = m.Fused.softmax(m.SFloat.cast(h[:rows])).to_numpy()
    for down in (0, 1):
        x = m.SFloat.cast(h)
        operand, result = x[:rows], x[down:rows + down]
        d, z = operand._desc(), result._desc()
        assert _lib.lib.cumo_hip_na_softmax(C.byref(d), C.byref(z)) == 0
        close(x.to_numpy()[down:rows + down], want, n, np.float32, ("rows further down", down))
