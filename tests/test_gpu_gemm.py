"""Prefill GEMM (M > 16) through the device-pointer API.

The kernel copies its tiles straight from global memory into a two-stage LDS
ring and writes C through an LDS-staged epilogue; these cases cover both tile
heights (64 rows, and 128 rows once the grid gives two workgroups per CU),
ragged M / N edges (the scalar store tail when rows are not 16-byte
multiples), short and long k-loops, and three-term (f32) activations with
int8 weights. The reference is float64 over the same bf16 / int8 operands:
every product is exact in f32, only the summation order differs, so the
bound is the 1e-4 x RMS contract of gemm_nt_bf16 / gemm_nt_int8
(ops/src/kernels.rs:1199-1287).
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-4


def bf16_bits(x):
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def bf16_value(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32)


def assert_close_rms(got, ref, tol=TOL):
    ref = np.asarray(ref, np.float64)
    err = float(np.abs(np.asarray(got, np.float64) - ref).max())
    rms = float(np.sqrt(np.mean(ref * ref)))
    assert err <= tol * max(rms, 1e-30), f"max|d|={err:.3e} rms={rms:.3e}"


class Device:
    def __init__(self, lib):
        self.lib, self.ptrs = lib, []

    def check(self, rc):
        assert rc == 0, self.lib.vmlm_hip_last_error().decode()

    def up(self, a):
        a = np.ascontiguousarray(a)
        p = C.c_void_p()
        self.check(self.lib.vmlm_hip_malloc(C.byref(p), a.nbytes))
        self.check(self.lib.vmlm_hip_memcpy_h2d(p, a.ctypes.data, a.nbytes))
        self.ptrs.append(p)
        return p

    def empty(self, nbytes):
        p = C.c_void_p()
        self.check(self.lib.vmlm_hip_malloc(C.byref(p), nbytes))
        self.ptrs.append(p)
        return p

    def down(self, p, shape, dtype):
        out = np.empty(shape, dtype)
        self.check(self.lib.vmlm_hip_sync())
        self.check(self.lib.vmlm_hip_memcpy_d2h(out.ctypes.data, p, out.nbytes))
        return out

    def free(self):
        for p in self.ptrs:
            self.lib.vmlm_hip_free(p)


@pytest.fixture
def dev(hip):
    d = Device(hip)
    yield d
    d.free()


@pytest.mark.parametrize("m,n,k", [(1024, 2048, 512),   # config 1
                                   (1, 2048, 512),      # config 1, M = 1 (GEMV path)
                                   (16, 2048, 512),     # GEMV path, 16 rows
                                   (5, 300, 192),       # GEMV path, ragged N
                                   (2048, 4096, 128),   # 128-row tiles
                                   (130, 201, 192),     # ragged, odd row stride
                                   (17, 128, 64)])      # one k-step, one spare row
def test_gemm_bf16_bf16(dev, m, n, k):
    rng = np.random.default_rng(m * 3 + n + k)
    a = bf16_bits(rng.standard_normal((m, k), dtype=np.float32))
    b = bf16_bits(rng.standard_normal((n, k), dtype=np.float32) / np.float32(np.sqrt(k)))
    da, db, dc = dev.up(a), dev.up(b), dev.empty(m * n * 4)
    dev.check(dev.lib.vmlm_hip_gemm_nt_bf16bf16(da, db, dc, m, n, k, None))
    got = dev.down(dc, (m, n), np.float32)
    ref = bf16_value(a).astype(np.float64) @ bf16_value(b).astype(np.float64).T
    assert_close_rms(got, ref)


@pytest.mark.parametrize("m,n,k", [(200, 2304, 5760),   # down projection, 90 k-steps
                                   (2048, 384, 256)])   # many row tiles
def test_gemm_int8_three_terms(dev, oracle, m, n, k):
    rng = np.random.default_rng(m + n * 5 + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    q = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    s = (np.abs(rng.normal(0, 0.02, n)) / 127 + 1e-6).astype(np.float32)
    da, dq, ds, dc = dev.up(a), dev.up(q), dev.up(s), dev.empty(m * n * 4)
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(da, dq, ds, dc, m, n, k, None))
    got = dev.down(dc, (m, n), np.float32)
    ref = (a.astype(np.float64) @ q.astype(np.float64).T) * s.astype(np.float64)
    assert_close_rms(got, ref)
    assert_close_rms(got, oracle.gemm_nt_int8(a, q, s))


def test_gemm_int8_row_split_paths_agree(dev):
    """Up to 256 rows are split into int8 terms by one launch (stats and terms
    per row), more rows by a stats launch and a blocked terms launch. Both
    form the same sums in the same order, so rows 0..255 of a 256-row and a
    257-row call give the same bits (N = 8192: neither call is k-sliced).
    Rows of mixed magnitude, a zero row and a NaN row are among them."""
    m, n, k = 257, 8192, 512
    rng = np.random.default_rng(257)
    a = rng.standard_normal((m, k), dtype=np.float32)
    a *= np.float32(10.0) ** rng.integers(-6, 7, size=(m, 1)).astype(np.float32)
    a[5] = 0.0
    a[17, 3] = np.nan
    q = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    s = (np.abs(rng.normal(0, 0.02, n)) / 127 + 1e-6).astype(np.float32)
    da, dq, ds = dev.up(a), dev.up(q), dev.up(s)
    c256, c257 = dev.empty(256 * n * 4), dev.empty(m * n * 4)
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(da, dq, ds, c256, 256, n, k, None))
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(da, dq, ds, c257, m, n, k, None))
    g256 = dev.down(c256, (256, n), np.float32)
    g257 = dev.down(c257, (m, n), np.float32)
    assert np.isnan(g256[17]).all() and (g256[5] == 0).all()
    np.testing.assert_array_equal(g256.view(np.uint32), g257[:256].view(np.uint32))
    ref = (a.astype(np.float64) @ q.astype(np.float64).T) * s.astype(np.float64)
    ok = np.isfinite(ref).all(axis=1)
    for r in np.flatnonzero(ok)[:40]:
        assert_close_rms(g257[r], ref[r])


def test_gemm_int8_row_split_wave_path_agrees(dev):
    """From 2048 rows one launch splits every row with one wave (eight rows
    per workgroup, the row's maximum across the wave); below, the stats and
    terms launches do. Without a norm the split depends only on each row's
    maximum, so rows 0..2046 of a 2047-row and a 2048-row call give the same
    bits. Rows of mixed magnitude, a zero row and a NaN row are among them."""
    m, n, k = 2048, 8192, 512
    rng = np.random.default_rng(2048)
    a = rng.standard_normal((m, k), dtype=np.float32)
    a *= np.float32(10.0) ** rng.integers(-6, 7, size=(m, 1)).astype(np.float32)
    a[5] = 0.0
    a[1700, 3] = np.nan
    q = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    s = (np.abs(rng.normal(0, 0.02, n)) / 127 + 1e-6).astype(np.float32)
    da, dq, ds = dev.up(a), dev.up(q), dev.up(s)
    c_lo, c_hi = dev.empty((m - 1) * n * 4), dev.empty(m * n * 4)
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(da, dq, ds, c_lo, m - 1, n, k, None))
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(da, dq, ds, c_hi, m, n, k, None))
    g_lo = dev.down(c_lo, (m - 1, n), np.float32)
    g_hi = dev.down(c_hi, (m, n), np.float32)
    assert np.isnan(g_hi[1700]).all() and (g_hi[5] == 0).all()
    np.testing.assert_array_equal(g_lo.view(np.uint32), g_hi[:m - 1].view(np.uint32))
    ref = (a[:64].astype(np.float64) @ q.astype(np.float64).T) * s.astype(np.float64)
    for r in range(0, 64, 7):
        if r != 5:
            assert_close_rms(g_hi[r], ref[r])


@pytest.mark.parametrize("m,n", [(2048, 4096),    # 32 x 32 tiles of 64 x 128
                                 (2100, 4112)])   # ragged last tile row and column
def test_gemm_int8_many_tiles_exact(dev, m, n):
    """A large grid (two LDS stages; the weights as they are, where the pass that
    swizzles them does not pay). Integer activations
    give exact int8 terms and exact f32 sums, so the result is the float64
    product bit for bit; the ragged case clamps the copies of column tiles
    past the weights and stores only rows < M and columns < N. A NaN row goes
    through the f32 recomputation."""
    k = 256
    rng = np.random.default_rng(m + n)
    a = rng.integers(-8, 9, size=(m, k)).astype(np.float32)
    a[m - 1, 7] = np.nan
    q = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    s = np.ones(n, np.float32)
    da, dq, ds, dc = dev.up(a), dev.up(q), dev.up(s), dev.empty(m * n * 4)
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(da, dq, ds, dc, m, n, k, None))
    got = dev.down(dc, (m, n), np.float32)
    ref = a[:m - 1].astype(np.float64) @ q.astype(np.float64).T
    np.testing.assert_array_equal(got[:m - 1].astype(np.float64), ref)
    assert np.isnan(got[m - 1]).all()


@pytest.mark.parametrize("n", [4096, 4112])
def test_gemm_int8_swizzled_exact(dev, n):
    """Enough tiles for the call to swizzle the weights (ragged last tile row and,
    at 4112, column): exact on integers, rows with a NaN or an infinity recomputed
    from the row-major weights."""
    m, k = 4100, 256
    rng = np.random.default_rng(n)
    a = rng.integers(-8, 9, size=(m, k)).astype(np.float32)
    q = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    q[:, 9] = np.where(q[:, 9] == 0, 1, q[:, 9])
    q[0, 9] = 0
    a[m - 1, 7] = np.nan
    a[63, 9] = np.inf
    da, dq, ds, dc = dev.up(a), dev.up(q), dev.up(np.ones(n, np.float32)), dev.empty(m * n * 4)
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(da, dq, ds, dc, m, n, k, None))
    got = dev.down(dc, (m, n), np.float32)
    rows = np.delete(np.arange(m), [63, m - 1])
    ref = a[rows].astype(np.float64) @ q.astype(np.float64).T
    np.testing.assert_array_equal(got[rows].astype(np.float64), ref)
    assert np.isnan(got[m - 1]).all() and np.isnan(got[63, 0])
    np.testing.assert_array_equal(got[63, 1:], np.where(q[1:, 9] > 0, np.inf, -np.inf))


def direct_case(rng, m, n, k, int8):
    a = rng.standard_normal((m, k), dtype=np.float32)
    if int8:
        w = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
        return a, w, w.astype(np.float64), rng.uniform(1e-4, 1e-3, n).astype(np.float32)
    u = rng.standard_normal((n, k), dtype=np.float32).view(np.uint32) & np.uint32(0xffff0000)
    return a, (u >> np.uint32(16)).astype(np.uint16), u.view(np.float32).astype(np.float64), None


# One launch over the rows as they are: K below, at and past the 64-wide blocks
# and the eight runs, rows and columns at the edges of each tile (16 x 16, 16 x
# 32, 16 x 64, 32 x 32, 32 x 64) and operands at any byte or float alignment.
@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (2, 17, 63), (16, 33, 65), (17, 40, 577),
                                   (33, 2050, 513), (77, 1537, 1001), (100, 2304, 5760),
                                   (300, 1000, 1000), (1000, 1500, 100), (12, 9000, 1536)])
def test_gemm_direct_edges(dev, m, n, k, int8):
    """Against float64. A result is at most ceil(K / 64 / 4) blocks of two
    MFMAs and three terms in one chain, each MFMA adding 32 products in f32,
    then at most eight waves: the error is within (32 * 6 * ceil(K / 256) + 10)
    roundings of 2^-24 of sum |a w|. Roundings of both signs leave far less, 1.8e-7
    of the result's norm at most; two of the three terms would leave 2.2e-6 or
    more at each of these sizes (2^-18 of an element), so 5e-7 tells them apart."""
    rng = np.random.default_rng(m + n + k)
    a, w, w64, s = direct_case(rng, m, n, k, int8)
    ref = a.astype(np.float64) @ w64.T
    bound = (192 * -(-k // 256) + 10) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(w64).T)
    if int8:
        ref, bound = ref * s, bound * s
    c = dev.empty(m * n * 4)
    for skew in (0, 1):  # rows as allocated, then off by one element (f32 4 bytes, weights 1 or 2)
        off = skew * w.itemsize
        da = dev.up(np.concatenate([np.zeros(4 * skew, np.uint8), a.view(np.uint8).ravel()]))
        dw = dev.up(np.concatenate([np.zeros(off, np.uint8), w.view(np.uint8).ravel()]))
        pa, pw = C.c_void_p(da.value + 4 * skew), C.c_void_p(dw.value + off)
        if int8:
            dev.check(dev.lib.vmlm_hip_gemm_nt_int8(pa, pw, dev.up(s), c, m, n, k, None))
        else:
            dev.check(dev.lib.vmlm_hip_gemm_nt_bf16(pa, pw, c, m, n, k, None))
        got = dev.down(c, (m, n), np.float32).astype(np.float64)
        assert (np.abs(got - ref) <= bound).all()
        assert np.linalg.norm(got - ref) <= 5e-7 * np.linalg.norm(ref)


@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize("m,n,k", [(2, 17, 63), (17, 40, 577), (33, 2050, 513), (77, 1537, 1001),
                                   (100, 2304, 5760), (300, 1000, 1000), (12, 9000, 1537)])
def test_gemm_direct_all_24_bits(dev, m, n, k, int8):
    """One power of two in each weight row: the product is one row element times
    it, so all 24 bits of the element come back, each from its term."""
    rng = np.random.default_rng(m * n + k)
    a = rng.integers(2 ** 23, 2 ** 24, (m, k)).astype(np.float32) * rng.choice([-1, 1], (m, k))
    a = (a * 2.0 ** rng.integers(-30, -20, (m, k))).astype(np.float32)
    at, v = rng.integers(0, k, n), rng.choice([-64, -1, 1, 2, 32], n)
    w = np.zeros((n, k), np.float32)
    w[np.arange(n), at] = v
    c = dev.empty(m * n * 4)
    if int8:
        ds = dev.up(np.ones(n, np.float32))
        dev.check(dev.lib.vmlm_hip_gemm_nt_int8(dev.up(a), dev.up(w.astype(np.int8)), ds, c, m, n,
                                                k, None))
    else:
        dev.check(dev.lib.vmlm_hip_gemm_nt_bf16(dev.up(a), dev.up(bf16_bits(w)), c, m, n, k, None))
    np.testing.assert_array_equal(dev.down(c, (m, n), np.float32), a[:, at] * v.astype(np.float32))


def test_gemm_direct_infinite_and_nan_rows(dev):
    """A row with an infinity or a NaN takes the split that keeps them in the
    first term: +-inf by the weight's sign, NaN at a zero weight or a NaN."""
    rng = np.random.default_rng(2)
    m, n, k = 20, 70, 130
    a, w, w64, s = direct_case(rng, m, n, k, True)
    a[3, 129] = np.inf
    a[4, 5] = np.nan
    a[19, 0] = -np.inf
    with np.errstate(invalid="ignore"):
        ref = (a.astype(np.float64) @ w64.T) * s
    c = dev.empty(m * n * 4)
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(dev.up(a), dev.up(w), dev.up(s), c, m, n, k, None))
    got = dev.down(c, (m, n), np.float32)
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(got), f(ref))
    ok = np.isfinite(ref)
    assert np.abs(got[ok] - ref[ok]).max() <= 1e-5 * np.sqrt(np.mean(ref[ok] ** 2))


# int8 rows: rows with a NaN or an infinity written by the GEMM's epilogue (odd N;
# 96 columns a tile) and by the slice reduction; the rows' split in one launch and
# in two (rows x K past 3.6e6), fewer and more k-slices.
@pytest.mark.parametrize("m,n,k", [(129, 131, 256), (300, 2304, 128), (630, 64, 5760),
                                   (150, 256, 2304), (200, 2048, 4096)])
def test_gemm_int8_rows_infinite_and_nan_rows(dev, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, w, w64, s = direct_case(rng, m, n, k, True)
    w[:20, 9] = 0
    w64[:20, 9] = 0
    rows = [0, 1, 62, 63, 64, 100, m - 2, m - 1]
    a[rows[::2], 9] = np.inf
    a[rows[1::2], k - 1] = -np.inf
    a[64, 3] = np.nan
    with np.errstate(invalid="ignore"):
        ref = (a.astype(np.float64) @ w64.T) * s
    c = dev.empty(m * n * 4)
    dev.check(dev.lib.vmlm_hip_gemm_nt_int8(dev.up(a), dev.up(w), dev.up(s), c, m, n, k, None))
    got = dev.down(c, (m, n), np.float32)
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(got), f(ref))
    ok = np.isfinite(ref)
    # three int8 terms leave at most 2^-21 of the row's maximum per element
    bound = (np.abs(np.where(np.isfinite(a), a, 0)).max(1)[:, None] * 2.0 ** -21 *
             np.abs(w64).sum(1) * s + 1e-5 * np.sqrt(np.mean(ref[ok] ** 2)))
    assert (np.abs(got[ok].astype(np.float64) - ref[ok]) <= bound[ok]).all()


# f32 GEMM: each tile (32 x 32, 32 x 64, 64 x 64, 128 x 128), rows and columns at
# their edges, k at the 32-deep steps' edges, rows on and off 16 bytes (k % 4, n %
# 4, operands a float off), with k-slices and without, NT and NN.
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (31, 33, 31), (33, 2305, 96), (40, 100, 1030),
                                   (513, 1028, 64), (1030, 1020, 36), (2049, 2052, 33)])
def test_gemm_f32_edges(dev, m, n, k):
    """Against float64: at most k products in one accumulator, then eight of them
    and up to 16 slices: (k + 20) roundings of 2^-24 of sum |a b|."""
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((n, k), dtype=np.float32)
    c0 = rng.standard_normal((m, n), dtype=np.float32)
    ref = a.astype(np.float64) @ b.astype(np.float64).T
    bound = (k + 20) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T +
                                     np.abs(c0))
    zero = np.zeros(1, np.float32)
    for off in (0, 1):
        pad = zero[:off]
        da = C.c_void_p(dev.up(np.concatenate([pad, a.ravel()])).value + 4 * off)
        for f, bb in ((dev.lib.vmlm_hip_gemm_nt, b), (dev.lib.vmlm_hip_gemm, b.T)):
            db = C.c_void_p(dev.up(np.concatenate([pad, bb.ravel()])).value + 4 * off)
            for acc in (False, True):
                dc = dev.up(c0)
                dev.check(f(da, db, dc, m, n, k, acc, None))
                got = dev.down(dc, (m, n), np.float32).astype(np.float64)
                assert (np.abs(got - (ref + c0 if acc else ref)) <= bound).all()


@pytest.mark.parametrize("m,k,int8", [(77, 1001, True), (17, 256, True), (9, 384, False)])
def test_gemm_over_its_own_rows(dev, m, k, int8):
    """The result written over the activation rows (n = k), against float64."""
    rng = np.random.default_rng(m * 3 + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    s = np.full(k, 0.01, np.float32)
    if int8:
        w = rng.integers(-127, 128, (k, k), dtype=np.int8)
        ref = (a.astype(np.float64) @ w.astype(np.float64).T) * s
    else:
        w = bf16_bits(rng.standard_normal((k, k), dtype=np.float32))
        ref = a.astype(np.float64) @ bf16_value(w).astype(np.float64).T
    c = dev.up(a)
    if int8:
        dev.check(dev.lib.vmlm_hip_gemm_nt_int8(c, dev.up(w), dev.up(s), c, m, k, k, None))
    else:
        dev.check(dev.lib.vmlm_hip_gemm_nt_bf16(c, dev.up(w), c, m, k, k, None))
    assert_close_rms(dev.down(c, (m, k), np.float32), ref)


# every path of the int8 / bf16 GEMM: full-K and k-split GEMV, one slice and more;
# one launch; int8 rows without and with k-slices, weights in rows and swizzled;
# term planes over weights as they are and over a padded copy
@pytest.mark.parametrize("m,k,int8,over", [
    (m, k, int8, over)
    for m, k, int8 in [(3, 2304, True), (16, 384, True), (9, 2304, True), (77, 1001, True),
                       (300, 512, True), (150, 256, True), (1600, 2304, True), (4100, 130, True),
                       (300, 640, False), (3, 1024, False), (1000, 770, False)]
    for over in ("rows", "weights", "scales")[:3 if int8 else 2]])
def test_gemm_over_any_operand(dev, m, k, int8, over):
    """The result written over an operand (n = k) has the bits of the result in a
    buffer of its own, rows with an infinity or a NaN included."""
    rng = np.random.default_rng(m * 5 + k)
    a, w, _, s = direct_case(rng, m, k, k, int8)
    a[m - 1, 5] = np.inf
    a[m // 2, k - 1] = np.nan
    size = max(m * k * 4, k * k * 2)

    def put(x):
        p = dev.empty(size)
        dev.check(dev.lib.vmlm_hip_memcpy_h2d(p, np.ascontiguousarray(x).ctypes.data, x.nbytes))
        return p

    out = []
    for own in (True, False):
        da, dw, ds = put(a), put(w), put(s) if int8 else None
        c = dev.empty(size) if own else dict(rows=da, weights=dw, scales=ds)[over]
        if int8:
            dev.check(dev.lib.vmlm_hip_gemm_nt_int8(da, dw, ds, c, m, k, k, None))
        else:
            dev.check(dev.lib.vmlm_hip_gemm_nt_bf16(da, dw, c, m, k, k, None))
        out.append(dev.down(c, (m, k), np.uint32))
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("m,k", [(40, 512), (3, 2304), (77, 1001),
                                 (1500, 2304),   # C beside the int8 rows: more than the scratch
                                 (1000, 1500)])  # C beside the terms and the padded copy alike
def test_gemm_noalloc_over_its_own_rows(dev, m, k):
    rng = np.random.default_rng(m + k)
    a, w, _, s = direct_case(rng, m, k, k, True)
    dw, ds, c, da = dev.up(w), dev.up(s), dev.empty(m * k * 4), dev.up(a)
    f = dev.lib.vmlm_hip_gemm_nt_int8_noalloc
    dev.check(f(da, dw, ds, c, m, k, k, None))
    want = dev.down(c, (m, k), np.float32)
    dev.check(f(da, dw, ds, da, m, k, k, None))
    got = dev.down(da, (m, k), np.float32)
    ref = (a.astype(np.float64) @ w.astype(np.float64).T) * s
    assert_close_rms(want, ref)
    assert_close_rms(got, ref)


# f32: no slice at any k, one and more slices otherwise; each tile
@pytest.mark.parametrize("m,k", [(20, 64), (100, 256), (256, 448), (64, 1030), (1000, 300),
                                 (1500, 1028), (2100, 96)])
@pytest.mark.parametrize("over", ["a", "b"])
def test_gemm_f32_over_its_operands(dev, m, k, over):
    """n = k, NT and NN, overwriting and accumulating: as in a buffer of its own
    that held the operand's values."""
    rng = np.random.default_rng(m + 3 * k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, k), dtype=np.float32)
    size = max(m, k) * k * 4
    under = a if over == "a" else b  # what C holds before, where it accumulates

    def put(x):
        p = dev.empty(size)
        dev.check(dev.lib.vmlm_hip_memset(p, 0, size))
        dev.check(dev.lib.vmlm_hip_memcpy_h2d(p, x.ctypes.data, x.nbytes))
        return p

    for f in (dev.lib.vmlm_hip_gemm_nt, dev.lib.vmlm_hip_gemm):
        for acc in (False, True):
            out = []
            for own in (True, False):
                da, db = put(a), put(b)
                c = put(under) if own else da if over == "a" else db
                dev.check(f(da, db, c, m, k, k, acc, None))
                out.append(dev.down(c, (m, k), np.uint32))
            assert np.array_equal(out[0], out[1])


def test_memset_after_queued_work(dev):
    """memset comes after the calls that the library stream was given before it
    (a millisecond of products that write the buffer) and before the next one."""
    n = 2048
    rng = np.random.default_rng(4)
    a = rng.standard_normal((n, n), dtype=np.float32)
    da, c = dev.up(a), dev.empty(n * n * 4)
    for _ in range(3):
        for _ in range(8):
            dev.check(dev.lib.vmlm_hip_gemm_nt(da, da, c, n, n, n, False, None))
        dev.check(dev.lib.vmlm_hip_memset(c, 0, n * n * 4))
        assert not dev.down(c, (n, n), np.uint32).any()
        dev.check(dev.lib.vmlm_hip_memset(c, 0x3f, n * n * 4))
        dev.check(dev.lib.vmlm_hip_scale(c, c, n * n, 2.0, None))
        got = dev.down(c, (n, n), np.float32)
        assert (got == 2 * np.uint32(0x3f3f3f3f).view(np.float32)).all()


@pytest.mark.parametrize("m,n,k", [(m, n, k) for m, n in [(1, 40), (33, 64), (100, 256)]
                                   for k in (130, 448, 2304, 16384, 65536) if m * k < 6e6])
def test_gemm_f32_sums_in_short_runs(dev, m, n, k):
    """Outputs of few tiles: 1 + (k - 1) 2^-25. A product that meets a sum with the
    1 in it is lost, so the error counts the products of that sum's run (at most
    64, or 128 past k = 2304), and half an ulp of 1 for each sum of runs (eight
    accumulators, in three steps) and of slices (64 at most)."""
    a = np.full((m, k), 2.0 ** -25, np.float32)
    a[:, 0] = 1
    c = dev.empty(m * n * 4)
    da, db = dev.up(a), dev.up(np.ones((n, k), np.float32))
    run, slices = 64 if k <= 2304 else 128, 1 if k < 449 else 64
    for f in (dev.lib.vmlm_hip_gemm_nt, dev.lib.vmlm_hip_gemm):  # ones either way
        dev.check(f(da, db, c, m, n, k, False, None))
        got = dev.down(c, (m, n), np.float32).astype(np.float64)
        assert np.abs(got - (1 + (k - 1) * 2.0 ** -25)).max() <= (run + 2 * (3 + slices)) * 2.0 ** -25


def test_upload_after_queued_work(dev):
    """memcpy_h2d comes after the calls that still read what it writes over."""
    n = 2048
    rng = np.random.default_rng(5)
    a, b = (rng.standard_normal((n, n), dtype=np.float32) for _ in range(2))
    da, one = dev.up(a), dev.up(np.eye(n, dtype=np.float32))
    cs = [dev.empty(n * n * 4) for _ in range(8)]
    for c in cs:
        dev.check(dev.lib.vmlm_hip_gemm_nt(da, one, c, n, n, n, False, None))
    dev.check(dev.lib.vmlm_hip_memcpy_h2d(da, b.ctypes.data, b.nbytes))
    for c in cs:
        assert np.array_equal(dev.down(c, (n, n), np.float32), a)
    assert np.array_equal(dev.down(da, (n, n), np.float32), b)
