"""Edges of the fp32-activation reader's tile kernels (uq_frontier.hip) against the
CPU oracle: ragged tiles of 16 rows, columns that fill no whole step (128 or 256
values), fewer steps than a workgroup has waves, many tiles per workgroup, groups
of 256 values whose range exceeds the integer digits, infinite block scales, and
both launch forms of a job table.

Outputs are the exact double sum rounded to f32 once, so the bound is 1 ulp (a
double sum a few 2^-53 off may round the other way)."""
import ctypes

import numpy as np
import pytest

import oracle as O
import uq
from test_gpu_linear import ulps

pytestmark = pytest.mark.gpu

TILE_KINDS = [k for k in uq.LINEAR_KINDS if k not in (uq.KIND_F32, uq.KIND_BF16)]
BLOCK32 = (uq.KIND_Q8_0, uq.KIND_IQ4_NL)


def check(kind, n, m, x, seed):
    raw = uq.synth_quant(kind, seed, m, n)
    y = uq.linear(uq.Weight(kind, n, m, raw), x)
    ref = O.linear(kind, raw, n, m, x)
    assert ulps(y, ref).max() <= 1, (kind, n, m)
    return y


@pytest.mark.parametrize("kind", TILE_KINDS)
@pytest.mark.parametrize("m", [1, 15, 16, 17, 4097])
def test_ragged_rows(gpu, kind, m):
    check(kind, 512, m, uq.synth_normal(m, 512), 0x711 + kind)


@pytest.mark.parametrize("kind,n", [(k, n) for k in BLOCK32 for n in (32, 96, 160, 288, 1056, 2528)] +
                         [(k, n) for k in TILE_KINDS for n in (256, 768, 2304, 16384)])
def test_columns(gpu, kind, n):
    check(kind, n, 50, uq.synth_normal(n, n), 0xC01 + kind)


@pytest.mark.parametrize("kind", TILE_KINDS)
@pytest.mark.parametrize("n", [256, 1280])
def test_many_tiles_per_workgroup(gpu, kind, n):
    # 20011 rows = 1251 tiles: several tiles for every workgroup of 256 CUs
    check(kind, n, 20011, uq.synth_normal(n + 1, n), 0x3A9 + kind)


@pytest.mark.parametrize("kind", TILE_KINDS)
@pytest.mark.parametrize("groups", [(0,), (1, 4), (0, 1, 2, 3, 4)])
def test_wide_groups(gpu, kind, groups):
    """Groups of 256 values whose smallest value lies more than 2^38 below the
    largest run in double, the others beside them on the digits."""
    n = 1280
    x = uq.synth_normal(kind, n)
    for g in groups:
        x[256 * g + 7] = np.float32(1e-20)
        x[256 * g + 200] = np.float32(-3e-39)  # denormal
    check(kind, n, 100, x, 0x51D + kind)
    x[3] = np.float32(2e30)  # and a value that swamps its own group
    check(kind, n, 100, x, 0x51E + kind)


@pytest.mark.parametrize("kind,offset", [(uq.KIND_Q8_0, 0), (uq.KIND_IQ4_NL, 0), (uq.KIND_IQ4_XS, 0),
                                         (uq.KIND_IQ3_XXS, 0), (uq.KIND_Q6_K, 208)])
def test_infinite_scale(gpu, kind, offset):
    """A row with an infinite block scale is not finite; the rows of its tile and
    the other tiles keep their values."""
    n, m = 1024, 40
    raw = uq.synth_quant(kind, 0x1F + kind, m, n)
    rb = uq.row_bytes(kind, n)
    raw[20 * rb + offset], raw[20 * rb + offset + 1] = 0x00, 0x7C
    x = uq.synth_normal(kind + 9, n)
    w = uq.Weight(kind, n, m, raw)
    L = uq.lib()
    dx, dy = ctypes.c_void_p(), ctypes.c_void_p()
    assert L.uq_dev_alloc(4 * n, ctypes.byref(dx)) == 0 and L.uq_dev_alloc(4 * m, ctypes.byref(dy)) == 0
    try:
        assert L.uq_memcpy_h2d(dx, x.ctypes.data, 4 * n) == 0
        assert L.uq_linear_dev(w.handle, dx, dy, None) == 0
        y = np.empty(m, np.float32)
        assert L.uq_memcpy_d2h(y.ctypes.data, dy, 4 * m) == 0
    finally:
        L.uq_dev_free(dx)
        L.uq_dev_free(dy)
    ref = O.linear(kind, raw, n, m, x)
    assert not np.isfinite(y[20]) and not np.isfinite(ref[20])
    assert (np.isnan(y[20]) and np.isnan(ref[20])) or y[20] == ref[20]
    rest = np.arange(m) != 20
    assert ulps(y[rest], ref[rest]).max() <= 1


@pytest.mark.parametrize("sizes", [[40] * 12, [5000] + [3] * 30, [1, 16, 17, 700]])
def test_job_table_forms_equal_single_calls(gpu, sizes):
    """Tables of similar jobs (a grid row per job) and of very unequal ones (starts
    searched) give the bits of the single calls."""
    pairs = []
    for i, m in enumerate(sizes):
        kind = uq.LINEAR_KINDS[i % len(uq.LINEAR_KINDS)]
        n = (512, 1024)[i % 2]
        pairs.append((uq.Weight(kind, n, m, uq.synth_quant(kind, i, m, n)), uq.synth_normal(i, n)))
    for (w, x), y in zip(pairs, uq.linear_batch(pairs)):
        assert np.array_equal(y.view(np.uint32), uq.linear(w, x).view(np.uint32))


@pytest.mark.parametrize("kind", [uq.KIND_Q8_0, uq.KIND_Q6_K])
def test_negative_values_far_below_their_group(gpu, kind):
    """Values that lie more than 2^62 below the largest of their 256 are no whole
    number of the group's unit, whatever their sign. The largest meets a zero code,
    so that only the small ones are in the sum."""
    n, m = 512, 33
    raw = uq.synth_quant(kind, 0x2E6 + kind, m, n).reshape(m, -1)
    if kind == uq.KIND_Q8_0:
        raw[:, 2] = 0
    else:  # code 32: low bits 0, high bits 2
        raw[:, 0] &= 0xF0
        raw[:, 128] = (raw[:, 128] & 0xFC) | 2
    raw = raw.reshape(-1)
    rng = np.random.default_rng(kind)
    for lo, hi in ((-36, -30), (-24, -21), (-19, -17), (-15, -12)):
        x = np.zeros(n, np.float32)
        x[1:256] = -(10.0 ** rng.uniform(lo, hi, 255))
        x[0] = 1.0
        y = uq.linear(uq.Weight(kind, n, m, raw), x)
        assert ulps(y, O.linear(kind, raw, n, m, x)).max() <= 1, (lo, hi)


SCALE_AT = {uq.KIND_Q8_0: 0, uq.KIND_IQ4_NL: 0, uq.KIND_IQ4_XS: 0, uq.KIND_IQ3_XXS: 0, uq.KIND_Q6_K: 208}


def linear_dev(kind, n, m, raw, x):
    """uq_linear_dev, which gives non-finite outputs where uq_linear refuses."""
    w = uq.Weight(kind, n, m, raw)
    L = uq.lib()
    dx, dy = ctypes.c_void_p(), ctypes.c_void_p()
    assert L.uq_dev_alloc(4 * n, ctypes.byref(dx)) == 0 and L.uq_dev_alloc(4 * m, ctypes.byref(dy)) == 0
    try:
        assert L.uq_memcpy_h2d(dx, x.ctypes.data, 4 * n) == 0
        assert L.uq_linear_dev(w.handle, dx, dy, None) == 0
        y = np.empty(m, np.float32)
        assert L.uq_memcpy_d2h(y.ctypes.data, dy, 4 * m) == 0
    finally:
        L.uq_dev_free(dx)
        L.uq_dev_free(dy)
    return y


def test_rows_beside_an_infinite_scale_keep_their_bits(gpu):
    """A row that is not finite is summed again, in another order; the other rows of
    its tile stay as they are. They hold pairs that cancel and a rest some 2^-44 of
    them, so that a sum of products in double differs in the leading bits, while
    the integer digits give the rest exactly."""
    n, m = 544, 40
    rng = np.random.default_rng(3)
    codes = np.zeros((m, n), np.int8)
    codes[:, :256] = rng.integers(-127, 128, (m, 256))
    codes[:, 256:512] = -codes[:, :256]
    codes[:, 512:] = rng.integers(-127, 128, (m, 32))
    raw = np.zeros((m, n // 32, 34), np.uint8)
    raw[:, :, 1] = 0x3C  # every scale 1.0
    raw[:, :, 2:] = codes.view(np.uint8).reshape(m, n // 32, 32)
    x = np.zeros(n, np.float32)
    x[:256] = rng.normal(0, 1, 256) * 2.0 ** rng.integers(-24, 1, 256)
    x[256:512] = x[:256]
    x[512:] = rng.normal(0, 1, 32) * 2.0 ** -44
    exact = (codes[:, 512:].astype(np.float64) * x[512:].astype(np.float64)).sum(1).astype(np.float32)
    clean = linear_dev(uq.KIND_Q8_0, n, m, raw.reshape(-1), x)
    assert ulps(clean, exact).max() <= 1
    raw[20, 3, 1] = 0x7C
    y = linear_dev(uq.KIND_Q8_0, n, m, raw.reshape(-1), x)
    assert not np.isfinite(y[20])
    rest = np.arange(m) != 20
    assert np.array_equal(y[rest].view(np.uint32), clean[rest].view(np.uint32))


@pytest.mark.parametrize("kind", TILE_KINDS)
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("signs", ["one", "both"])
def test_infinite_scale_gives_what_the_products_give(gpu, kind, wide, signs):
    """A row with an infinite scale is an infinity where its products have one sign
    and NaN where they have both (or a zero code), with and without groups of x that
    run in double."""
    n, m, row = 1024, 40, 20
    raw = uq.synth_quant(kind, 0x41F + kind, m, n)
    rb = uq.row_bytes(kind, n)
    if kind == uq.KIND_Q8_0:
        codes = raw[row * rb:(row + 1) * rb].reshape(-1, 34)[:, 2:]
        codes[codes == 0] = 1
    weights = O.dequantize(kind, raw[row * rb:(row + 1) * rb], n)
    x = np.abs(uq.synth_normal(kind + 9, n)) * np.where(weights < 0, np.float32(-1), np.float32(1))
    if signs == "both":
        x[1] = -x[1]
    if wide:
        x[[2, 600]] = 1e-20 * np.sign(x[[2, 600]])
    raw[row * rb + SCALE_AT[kind]], raw[row * rb + SCALE_AT[kind] + 1] = 0x00, 0x7C
    y = linear_dev(kind, n, m, raw, x)
    ref = O.linear(kind, raw, n, m, x)
    rest = np.arange(m) != row
    assert ulps(y[rest], ref[rest]).max() <= 1
    assert (np.isnan(y[row]) and np.isnan(ref[row])) or y[row] == ref[row]
    if signs == "one" and kind in (uq.KIND_Q8_0, uq.KIND_IQ4_NL, uq.KIND_IQ3_XXS):
        assert y[row] == np.inf  # (no zero code or sub-scale in these)


def far_x(n, seed, share):
    """Ordinary values, `share` of each group of 256 more than 2^38 below its largest
    (some denormal, some zero)."""
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1, n).astype(np.float32)
    far = rng.random(n) < share
    far[5::256] = True
    x[far] *= np.float32(2.0) ** rng.integers(-140, -40, far.sum())
    return x


def repeated_rows(kind, n, m, seed, rows=997):
    """Rows 0 .. 996 over and over: a weight of m rows and the raw bytes of the 997."""
    raw = uq.synth_quant(kind, seed, rows, n)
    return raw, np.resize(raw.reshape(rows, -1), (m, raw.size // rows)).reshape(-1)


def check_repeated(y, ref, m):
    assert ulps(y[:ref.size], ref).max() <= 1
    assert np.array_equal(y.view(np.uint32), np.resize(y[:ref.size], m).view(np.uint32))


# n 2048: more than eight tiles a workgroup, four of them summed at once, and the
# buffers used again; 512: fewer steps than waves; 8192: x leaves room for one
# tile's sums at once
@pytest.mark.parametrize("kind", TILE_KINDS)
@pytest.mark.parametrize("n,m", [(2048, 150001), (512, 150001), (8192, 30011)])
@pytest.mark.parametrize("share", [None, 0.004, 0.5])
def test_sums_of_many_tiles(gpu, kind, n, m, share):
    x = uq.synth_normal(n, n) if share is None else far_x(n, n, share)
    raw, big = repeated_rows(kind, n, m, 0x6B1 + kind)
    y = uq.linear(uq.Weight(kind, n, m, big), x)
    check_repeated(y, O.linear(kind, raw, n, 997, x), m)


@pytest.mark.parametrize("kind", TILE_KINDS)
@pytest.mark.parametrize("wide", [False, True])
def test_infinite_scales_in_late_tiles(gpu, kind, wide):
    """Every wave finds its own rows again: infinite scales in tiles all over a
    workgroup's."""
    n, m = 1024, 60011
    raw, big = repeated_rows(kind, n, m, 0x6C1 + kind)
    rb = uq.row_bytes(kind, n)
    bad = np.arange(7, m, 1999)
    at = bad * rb + SCALE_AT[kind]
    big[at], big[at + 1] = 0x00, 0x7C
    x = far_x(n, n, 0.01) if wide else uq.synth_normal(n, n)
    y = linear_dev(kind, n, m, big, x)
    assert not np.isfinite(y[bad]).any()
    for r in bad[:: max(1, len(bad) // 8)]:
        ref = O.linear(kind, big[r * rb:(r + 1) * rb], n, 1, x)[0]
        assert (np.isnan(y[r]) and np.isnan(ref)) or y[r] == ref
    ref = O.linear(kind, raw, n, 997, x)
    good = np.setdiff1d(np.arange(m), bad)
    assert ulps(y[good], np.resize(ref, m)[good]).max() <= 1


def test_far_values_in_a_job_table(gpu):
    """A table in which some jobs' x have such values gives the bits of the single
    calls."""
    pairs = []
    for i, m in enumerate([700, 33, 5000, 16, 1, 900, 64]):
        kind = TILE_KINDS[i % len(TILE_KINDS)]
        n = (512, 2560)[i % 2]
        x = far_x(n, i, 0.02) if i % 3 else uq.synth_normal(i, n)
        pairs.append((uq.Weight(kind, n, m, uq.synth_quant(kind, i, m, n)), x))
    for (w, x), y in zip(pairs, uq.linear_batch(pairs)):
        assert np.array_equal(y.view(np.uint32), uq.linear(w, x).view(np.uint32))


# either side of one and two workgroups a CU, of whole shares of the tiles and a
# workgroup on every CU, and of the longest x that leaves LDS for two (256 CUs)
@pytest.mark.parametrize("kind", TILE_KINDS)
@pytest.mark.parametrize("n,m", [(512, 32768), (512, 32769), (1024, 16384), (1024, 16385), (2560, 28672), (2560, 28673),
                                 (4096, 12288), (4096, 12289), (4096, 28673), (5376, 28673), (5632, 28673)])
def test_workgroups_of_one_weight(gpu, kind, n, m):
    x = uq.synth_normal(n + m, n)
    raw, big = repeated_rows(kind, n, m, 0x6D1 + kind)
    y = uq.linear(uq.Weight(kind, n, m, big), x)
    check_repeated(y, O.linear(kind, raw, n, 997, x), m)
