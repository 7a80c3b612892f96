"""GPU parity: dense row-major GEMM on the matrix cores (fp32 and bf16-in / fp32-accumulate).

Tolerance (written once, used everywhere): normwise ||C - C64||_F / ||C64||_F <= 1e-4 and, per
entry, |C - C64| <= 1e-4 * (|A|·|B|)_ij, against a float64 GEMM of the same inputs (for bf16, of
the bf16-rounded inputs). Element-relative error is ill-posed where C_ij ~ 0, hence the |A||B|
scaling. Large sizes are checked on sampled full rows plus a Freivalds product over all of C.
The reference's own case is CudaRealWorldAlgorithmTests.cs:56-96 (m=512, n=768, k=384, seeds 42/43,
abs 1e-3 vs a CPU fp32 triple loop), reproduced below against the oracle's fp32 loop.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

REL = 1e-4


def make_inputs(m, n, k, seed_a=42, seed_b=43):
    a = oracle.gen_uniform_f32(m * k, seed_a, 0).reshape(m, k)
    b = oracle.gen_uniform_f32(k * n, seed_b, 0).reshape(k, n)
    return a, b


def run_gemm(ctx, a, b, kind="f32"):
    m, k = a.shape
    _, n = b.shape
    c = ctx.empty((m, n), np.float32)
    if kind == "f32":
        da, db = ctx.to_device(a), ctx.to_device(b)
        ctx.gemm_f32(da, db, c, m, n, k)
    else:
        da, db = ctx.to_device(oracle.f32_to_bf16(a)), ctx.to_device(oracle.f32_to_bf16(b))
        ctx.gemm_bf16(da, db, c, m, n, k)
    ctx.synchronize()
    out = c.to_host()
    for x in (da, db, c):
        ctx.free(x)
    return out


def check_rows(c, a, b, rows):
    ref, absref = oracle.gemm_f64_rows(np.ascontiguousarray(a), np.ascontiguousarray(b), rows)
    got = c[rows].astype(np.float64)
    err = np.abs(got - ref)
    assert np.all(err <= REL * absref + 1e-30), f"max per-entry ratio {np.max(err / np.maximum(absref, 1e-30)):.3e}"
    normwise = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert normwise <= REL, normwise
    return normwise


def freivalds(c, a, b, seed=0):
    """C·r vs A·(B·r) in float64 with r in {-1,+1}^n; bound 1e-4 * (|A|·(|B|·1))."""
    rng = np.random.default_rng(seed)
    n = b.shape[1]
    r = rng.choice([-1.0, 1.0], size=n)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    lhs = c.astype(np.float64) @ r
    rhs = a64 @ (b64 @ r)
    bound = np.abs(a64) @ (np.abs(b64) @ np.ones(n))
    assert np.all(np.abs(lhs - rhs) <= REL * bound)


@pytest.mark.parametrize("shape", [(128, 128, 128), (256, 384, 640), (512, 768, 384), (1024, 1024, 1024)])
def test_gemm_f32_full_tiles(ctx, shape):
    m, n, k = shape
    a, b = make_inputs(m, n, k)
    c = run_gemm(ctx, a, b)
    check_rows(c, a, b, np.arange(m))


# Full 64-tiles on the fp32 instructions (direct-to-LDS loads): one, two and an odd number of 32-wide k
# tiles, few and many tiles.
@pytest.mark.parametrize("shape", [(128, 128, 32), (192, 320, 96), (256, 64, 64), (4096, 2048, 32),
                                   (2048, 4096, 64), (4096, 2048, 96)])
def test_gemm_f32_k_tile_counts(ctx, shape):
    m, n, k = shape
    a, b = make_inputs(m, n, k)
    c = run_gemm(ctx, a, b)
    check_rows(c, a, b, np.arange(m))


def test_gemm_f32_reference_case_vs_fp32_loop(ctx):
    """CudaRealWorldAlgorithmTests.cs:56-96: m=512, n=768, k=384, abs tol 1e-3 vs the fp32 triple loop."""
    m, n, k = 512, 768, 384
    a, b = make_inputs(m, n, k)
    c = run_gemm(ctx, a, b)
    expected = oracle.gemm_f32_naive(a, b, threads=8)
    assert np.max(np.abs(c - expected)) <= 1e-3


# The bounds-checked 64x64 tiles (fewer than 64 columns, k of 16 or less), and ragged split tiles: 64 with
# one and two k groups, 128 for (4000, 2100, 37).
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 7), (100, 37, 53), (129, 130, 131), (257, 64, 1000),
                                   (4000, 2100, 37)])
def test_gemm_f32_ragged(ctx, shape):
    m, n, k = shape
    a, b = make_inputs(m, n, k, 7, 8)
    c = run_gemm(ctx, a, b)
    check_rows(c, a, b, np.arange(m))


def test_gemm_f32_k_zero_gives_zeros(ctx):
    c = ctx.empty((4, 5), np.float32)
    a = ctx.empty(1, np.float32)
    ctx.gemm_f32(a, a, c, 4, 5, 0)
    ctx.synchronize()
    assert np.all(c.to_host() == 0)
    ctx.free(c)
    ctx.free(a)


def test_gemm_identity_and_permutation_exact(ctx):
    n = 256
    a, _ = make_inputs(n, n, n)
    eye = np.eye(n, dtype=np.float32)
    assert np.array_equal(run_gemm(ctx, a, eye), a)  # one nonzero term per entry: exact
    perm = np.eye(n, dtype=np.float32)[np.random.default_rng(1).permutation(n)]
    assert np.array_equal(run_gemm(ctx, perm, a), perm @ a)


@pytest.mark.slow
@pytest.mark.parametrize("n", [4096, 8192])
def test_gemm_f32_large_sampled(ctx, n):
    a, b = make_inputs(n, n, n)
    c = run_gemm(ctx, a, b)
    rows = np.unique(np.concatenate([[0, n - 1], np.random.default_rng(n).integers(0, n, 30)]))
    check_rows(c, a, b, rows)
    freivalds(c, a, b)


# (64-tiles with one and two k groups, over 1, 2, 3, 6 and more 64-wide k tiles; B through transposing LDS
# reads. (100, 37, 53): loads through registers. The others: test_gemm_bf16_ragged_tiles.)
@pytest.mark.parametrize("shape", [(128, 128, 64), (512, 768, 384), (100, 37, 53), (256, 256, 64),
                                   (1024, 512, 1024), (768, 1280, 192), (256, 512, 4096), (384, 256, 64),
                                   (512, 256, 128)])
def test_gemm_bf16(ctx, shape):
    m, n, k = shape
    a, b = make_inputs(m, n, k)
    c = run_gemm(ctx, a, b, kind="bf16")
    ar = oracle.bf16_to_f32(oracle.f32_to_bf16(a)).reshape(m, k)
    br = oracle.bf16_to_f32(oracle.f32_to_bf16(b)).reshape(k, n)
    check_rows(c, ar, br, np.arange(m))


@pytest.mark.slow
def test_gemm_bf16_8192_sampled(ctx):
    n = 8192
    a, b = make_inputs(n, n, n)
    c = run_gemm(ctx, a, b, kind="bf16")
    ar = oracle.bf16_to_f32(oracle.f32_to_bf16(a)).reshape(n, n)
    br = oracle.bf16_to_f32(oracle.f32_to_bf16(b)).reshape(n, n)
    rows = np.unique(np.concatenate([[0, n - 1], np.random.default_rng(5).integers(0, n, 16)]))
    check_rows(c, ar, br, rows)
    freivalds(c, ar, br)  # every entry, through C·r against A·(B·r) on the bf16-rounded inputs


def test_convert_f32_to_bf16_bit_exact(ctx):
    x = np.concatenate([oracle.gen_uniform_f32(100_000, 3, 0) * 1000,
                        np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-40, 3.3895314e38, 1.0039062], np.float32)])
    d = ctx.to_device(x)
    o = ctx.empty(x.size, np.uint16)
    ctx.convert_f32_to_bf16(d, o)
    ctx.synchronize()
    got = o.to_host()
    ref = oracle.f32_to_bf16(x)
    assert np.array_equal(got, ref)
    ctx.free(d)
    ctx.free(o)


# One shape or more per tile choice of the bf16 dispatch (on 256 CUs), with ragged rows, columns and a
# last k tile that is not whole. 16-byte rows: 256-tiles of one to four k tiles, 128-tiles (two), 128-tiles with two k
# groups, 64-tiles with one, two and four; other rows: 128-tiles, 64-tiles with one and four k groups,
# fewer columns than a tile. (host_tests.cpp checks that each shape takes the kernel it is here for.)
@pytest.mark.parametrize("shape", [(4096, 4096, 64), (2824, 3080, 72), (2816, 3072, 192), (2824, 3080, 200), (4104, 4360, 136),
                                   (2200, 2056, 200), (1800, 1912, 136), (200, 264, 200), (8, 8, 8),
                                   (456, 520, 520), (72, 136, 2120), (1799, 1911, 137), (63, 65, 129), (300, 50, 70),
                                   (129, 131, 1001), (70, 9, 64)])
def test_gemm_bf16_ragged_tiles(ctx, shape):
    m, n, k = shape
    a, b = make_inputs(m, n, k)
    a = oracle.bf16_to_f32(oracle.f32_to_bf16(a)).reshape(m, k)
    b = oracle.bf16_to_f32(oracle.f32_to_bf16(b)).reshape(k, n)
    c = run_gemm(ctx, a, b, kind="bf16")
    ref = a.astype(np.float64) @ b.astype(np.float64)
    absref = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    # products of bf16 values are exact in float32; k additions, each within one float32 ulp
    assert np.all(np.abs(c - ref) <= k * 2.0 ** -23 * absref)
    # what lies past a row's end (the next row, here of infinities) reaches no result
    a[1:] = np.inf
    c0 = run_gemm(ctx, a, b, kind="bf16")[0]
    assert np.array_equal(c0, c[0])


# One shape per kernel of the fp32 dispatch (on 256 CUs): split 256x128, 128, 128 with two k groups, 64,
# 64 with two and four, each with ragged rows, columns and last k tile; the fp32 instructions on full and
# on ragged tiles. (host_tests.cpp checks that each shape takes the kernel it is here for.)
F32_KERNELS = [(2570, 2571, 515), (2824, 3083, 67), (1799, 1911, 771), (300, 333, 61), (300, 333, 257),
               (129, 131, 1537), (128, 192, 64), (65, 60, 40)]


# (and the smallest k that the split kernels take, one less, and two shapes of few columns or rows)
@pytest.mark.parametrize("shape", F32_KERNELS + [(65, 64, 17), (65, 64, 16), (200, 64, 49), (64, 1000, 49)])
def test_gemm_f32_split_tiles(ctx, shape):
    m, n, k = shape
    a, b = make_inputs(m, n, k)

    def check(a, b):
        c = run_gemm(ctx, a, b)
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        # each product within 2^-24 of itself, k additions each within one float32 ulp
        assert np.all(np.abs(c - a64 @ b64) <= (k + 1) * 2.0 ** -23 * (np.abs(a64) @ np.abs(b64)))
        return c

    c = check(a, b)
    # values whose bf16 pieces would not hold them: everywhere, and in one row
    check(a * np.float32(2.0 ** -110), b)
    tiny = a.copy()
    tiny[m // 2] *= np.float32(2.0 ** -120)
    c2 = check(tiny, b)
    far = np.abs(np.arange(m) - m // 2) > 256  # rows of other tiles: the very same sums
    assert np.array_equal(c2[far], c[far])
    check(np.where(np.arange(m * k).reshape(m, k) % 3 == 0, a * np.float32(2.0 ** -115), a), b)
    # infinities, NaN and values that round to infinity in bf16 stay in their rows
    odd = a.copy()
    odd[0, 0], odd[1, 1], odd[2, k - 1], odd[3, 0] = np.inf, np.nan, -np.inf, 3.4e38
    bz = b.copy()
    bz[0, 0] = 0.0
    got = run_gemm(ctx, odd, bz)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = (odd.astype(np.float64) @ bz.astype(np.float64)).astype(np.float32)
    assert np.array_equal(np.isnan(got[:3]), np.isnan(ref[:3])) and np.array_equal(np.isinf(got[:3]), np.isinf(ref[:3]))
    # (row 3 by the bound above: its column 0 is an ordinary sum that cancels, no relative bound holds)
    bound3 = (k + 1) * 2.0 ** -23 * (np.abs(odd[3]).astype(np.float64) @ np.abs(bz).astype(np.float64))
    assert np.isfinite(got[3:]).all() and np.all(np.abs(got[3] - ref[3].astype(np.float64)) <= bound3)


def test_gemm_f32_split_permutation_exact(ctx):
    n = 2100  # one nonzero term per entry: the three pieces add up to the value itself
    a, _ = make_inputs(n, n, n)
    perm = np.eye(n, dtype=np.float32)[np.random.default_rng(1).permutation(n)]
    assert np.array_equal(run_gemm(ctx, perm, a), perm @ a)
    assert np.array_equal(run_gemm(ctx, a, perm), a @ perm)


@pytest.mark.parametrize("shape", F32_KERNELS)
def test_gemm_f32_single_terms(ctx, shape):
    """Scaled rows and columns: one product per entry, which the sum must hold as its roundings allow.

    The sum of the large products is one product and exact. The seven small products are below 2^-6.9
    |ab| in all; each addition of theirs is off by an ulp (2^-23 of the sum) at most, so with the product
    left out (2^-34) they are off by less than 2^-27 |ab|, an eighth of an ulp; the two sums are added with
    one rounding, half an ulp."""
    m, n, k = shape
    rng = np.random.default_rng(m)

    def values(*size):  # every mantissa bit, four binades, and 1.0038986 (pieces 1, 2^-8 and -2^-17) among them
        x = rng.uniform(1.0, 2.0, size) * 2.0 ** rng.integers(-2, 2, size) * rng.choice([-1.0, 1.0], size)
        x[rng.uniform(size=size) < 0.1] = 1.0038986
        return x.astype(np.float32)

    def check(got, exact):
        ulp = np.spacing(np.abs(exact).astype(np.float32)).astype(np.float64)
        assert np.max(np.abs(got - exact) / ulp) <= 0.5 + 2.0 ** -3

    place, factor = rng.integers(0, k, m), values(m)
    a, b = np.zeros((m, k), np.float32), values(k, n)
    a[np.arange(m), place] = factor
    check(run_gemm(ctx, a, b), factor[:, None].astype(np.float64) * b[place])
    place, factor = rng.integers(0, k, n), values(n)
    a, b = values(m, k), np.zeros((k, n), np.float32)
    b[place, np.arange(n)] = factor
    check(run_gemm(ctx, a, b), factor.astype(np.float64) * a[:, place])


@pytest.mark.parametrize("shape", F32_KERNELS)
def test_gemm_f32_integers_exact(ctx, shape):
    """9-bit integers, 60 at most per row: every partial sum is below 2^24, so any order is exact, and
    every value but the multiples of two has a second piece."""
    m, n, k = shape
    rng = np.random.default_rng(n)
    a = rng.integers(-511, 512, (m, k)) * (rng.uniform(size=(m, k)) < 50 / max(k, 50))
    for row in a:
        row[np.flatnonzero(row)[60:]] = 0
    b = rng.integers(-511, 512, (k, n))
    assert np.array_equal(run_gemm(ctx, a.astype(np.float32), b.astype(np.float32)), (a @ b).astype(np.float32))


@pytest.mark.parametrize("shape", F32_KERNELS + [(1537, 2049, 1023)])
def test_gemm_f32_error_of_a_float32_sum(ctx, shape):
    """Normal inputs: k roundings of partial sums, each of rms 2^-24 / sqrt(3) of a sum whose mean square
    is half of the last one's, make 2^-24 sqrt(k / 6) in the 2-norm; every second-order product of
    pieces (rms 2^-19 of a product) would show."""
    m, n, k = shape
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((k, n), np.float32)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.linalg.norm(run_gemm(ctx, a, b) - ref) <= 2.0 ** -24 * (k / 6) ** 0.5 * np.linalg.norm(ref)


@pytest.mark.parametrize("shape", F32_KERNELS)
def test_gemm_f32_exceptional_values_stay_in_their_rows_and_columns(ctx, shape):
    """A sum's arithmetic depends on its row of A and its column of B alone: rows and columns with an
    infinity, NaN, a value that rounds to infinity in bf16 or values whose pieces are lost leave every
    other entry's bits as they are."""
    m, n, k = shape
    a, b = make_inputs(m, n, k)
    c = run_gemm(ctx, a, b)
    odd_a, odd_b = a.copy(), b.copy()
    rows, cols = [0, 1, 2, 3, m // 2, m - 1], [5, n // 2, n - 1]
    odd_a[0, 0], odd_a[1, k - 1], odd_a[2, k // 2], odd_a[3, 1] = np.inf, np.nan, -np.inf, 3.4e38
    odd_a[m // 2] *= np.float32(2.0 ** -126)
    odd_a[m - 1, 1::2] *= np.float32(2.0 ** -130)
    odd_b[k - 1, 5], odd_b[:, n // 2], odd_b[0, n - 1] = np.nan, 0.0, -3.4e38
    got = run_gemm(ctx, odd_a, odd_b)
    same = np.ones((m, n), bool)
    same[rows], same[:, cols] = False, False
    assert np.array_equal(got[same], c[same])
    with np.errstate(invalid="ignore", over="ignore"):
        ref = odd_a.astype(np.float64) @ odd_b.astype(np.float64)
        bound = (k + 1) * 2.0 ** -23 * (np.abs(odd_a).astype(np.float64) @ np.abs(odd_b).astype(np.float64)) + 2.0 ** -149 * k
        fin = np.isfinite(ref) & (np.abs(ref) < 3.4e38)
        assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.all(np.abs(got[fin] - ref[fin]) <= bound[fin])


@pytest.mark.parametrize("shape", F32_KERNELS)
def test_gemm_f32_values_whose_pieces_are_lost(ctx, shape):
    """Values near 2^-130 times ones near 2^100: their bf16 pieces would be off by up to 2^-134, a
    sixteenth of the value. All of A, all of B, one row among ordinary ones (with a NaN in a column of B
    too), and the values at every fourth place of a row of A or a column of B, the rest of it zero."""
    m, n, k = shape
    a, b = make_inputs(m, n, k)
    small, large = np.float32(2.0 ** -130), np.float32(2.0 ** 100)
    cases = [(a * small, b * large), (a * large, b * small)]
    row, nan = a * np.float32(2.0 ** -60), b * large
    row[m // 2] = a[m // 2] * small
    nan[k - 1, 4] = np.nan
    cases += [(row, b * large), (row, nan)]
    for place in range(4):
        row, col = a * np.float32(2.0 ** -60), b * np.float32(2.0 ** -60)
        row[m // 2] = 0
        row[m // 2, place::4] = a[m // 2, place::4] * small
        # (four k of A are one load, and four columns of B)
        col[:, n // 8 * 4 + place] = b[:, n // 8 * 4 + place] * small
        cases += [(row, b * large), (a * large, col)]
    for x, y in cases:
        got = run_gemm(ctx, x, y)
        x64, y64 = x.astype(np.float64), y.astype(np.float64)
        # (the float32 product's error, as in the other tests: each of k additions within one ulp)
        err, bound = np.abs(got - x64 @ y64), (k + 1) * 2.0 ** -23 * (np.abs(x64) @ np.abs(y64))
        assert np.all((err <= bound) | np.isnan(bound))


@pytest.mark.slow
@pytest.mark.parametrize("shape", [(8, 128256, 8192), (8, 130048, 8200), (8, 130056, 8200)])
def test_gemm_bf16_b_of_almost_two_gib(ctx, shape):
    """B's byte offsets up to the end of the direct-to-LDS loads' buffer range, and just past it."""
    m, n, k = shape
    rng = np.random.default_rng(n)
    a = oracle.f32_to_bf16(rng.uniform(-1, 1, m * k).astype(np.float32)).reshape(m, k)
    part = oracle.f32_to_bf16(rng.uniform(-1, 1, 1000003).astype(np.float32))  # (a prime: no two rows alike)
    b = np.resize(part, n * k).reshape(k, n)
    da, db, c = ctx.to_device(a), ctx.to_device(b), ctx.empty((m, n), np.float32)
    ctx.gemm_bf16(da, db, c, m, n, k)
    ctx.synchronize()
    got = c.to_host()
    for x in (da, db, c):
        ctx.free(x)
    cols = np.unique(np.concatenate([rng.integers(0, n, 150), np.arange(n - 10, n), np.arange(10)]))
    a64 = oracle.bf16_to_f32(a).reshape(m, k).astype(np.float64)
    b64 = oracle.bf16_to_f32(np.ascontiguousarray(b[:, cols])).reshape(k, -1).astype(np.float64)
    # products of bf16 values are exact in float32; k additions, each within one float32 ulp
    assert np.all(np.abs(got[:, cols] - a64 @ b64) <= k * 2.0 ** -23 * (np.abs(a64) @ np.abs(b64)))


@pytest.mark.slow
@pytest.mark.parametrize("kind,m,n", [("f32", 2 ** 30 - 1, 1), ("f32", 1, 2 ** 30 - 1), ("bf16", 2 ** 30 - 1, 1)])
def test_gemm_longest_vectors(ctx, kind, m, n):
    """The largest m and n that the entries take: 2^24 tiles of 64, more work items than one row of a grid."""
    part = np.random.default_rng(1).integers(-100, 100, 1000003).astype(np.float32)  # exact in bf16
    long = np.resize(part if kind == "f32" else oracle.f32_to_bf16(part), max(m, n))
    other = np.full(1, 2.0, np.float32)
    dl, do = ctx.to_device(long), ctx.to_device(other if kind == "f32" else oracle.f32_to_bf16(other))
    c = ctx.empty(m * n, np.float32)
    (ctx.gemm_f32 if kind == "f32" else ctx.gemm_bf16)(*((dl, do) if m > n else (do, dl)), c, m, n, 1)
    ctx.synchronize()
    got = c.to_host()
    for x in (dl, do, c):
        ctx.free(x)
    whole = got[: got.size // part.size * part.size].reshape(-1, part.size)
    assert np.array_equal(whole[0], 2 * part) and (whole == whole[0]).all()
    assert np.array_equal(got[whole.size:], 2 * part[:got.size - whole.size])
