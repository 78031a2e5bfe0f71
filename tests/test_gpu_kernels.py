"""Single kernels of the device path at the sizes where their tiles, remainders and scans can go wrong."""
import ctypes as C

import numpy as np
import pytest

from pcaone_amd import _lib, api

pytestmark = pytest.mark.gpu

CODE_VALUE = np.array([1.0, 0.0, 0.5, 0.0])  # BED2GENO (code 01 missing)


def say(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(0)
    yield c
    c.close()


def pack(codes):
    m, n = codes.shape
    out = np.zeros((m, (n + 3) // 4), dtype=np.uint8)
    for e in range(4):
        sub = codes[:, e::4].astype(np.uint8)
        out[:, : sub.shape[1]] |= sub << (2 * e)
    return out


def random_codes(rng, m, n, miss):
    codes = rng.choice([0, 2, 3], (m, n))
    codes[rng.random((m, n)) < miss] = 1
    return codes


def standardized(codes):
    """The matrix of the products (rows = SNPs) in FP64, centered, scaled, missing entries 0, and the scales."""
    seen = codes != 1
    x = CODE_VALUE[codes]
    cnt = seen.sum(1)
    F = np.divide(x.sum(1), cnt, out=np.zeros(len(x)), where=cnt > 0)
    sd = np.sqrt(F * (1 - F))
    sc = np.where(sd > 1e-9, np.sqrt(2.0) / np.where(sd > 1e-9, sd, 1.0), 1.0)
    return np.where(seen, (x - F[:, None]) * sc[:, None], 0.0), sc


@pytest.mark.parametrize("n,m,miss", [(17, 33, 0.5), (63, 1025, 0.1), (64, 1024, 0.02), (1025, 65, 0.3),
                                      (2049, 1023, 0.01), (4100, 40, 1.0)])
def test_missing_lists(ctx, n, m, miss):
    """Products with missing genotypes in FP64 against the dense matrix: every entry of both lists counts.
    Rows without a missing entry and rows with nothing else are among them."""
    say(f"missing lists n={n} m={m} miss={miss}")
    rng = np.random.default_rng(n + m)
    codes = random_codes(rng, m, n, miss)
    codes[0] = rng.choice([0, 2, 3], n)
    codes[m // 2] = 1
    codes[:, n // 3] = 1
    codes[m - 1, n - 1] = 1
    L = 16
    omega = rng.standard_normal((n, L))
    ctx.upload_packed(pack(codes), n)
    assert ctx.dims() == (n, m, int((codes == 1).sum()))
    ctx.standardize()
    ctx.configure("fp64", L)
    ctx.set_omega(omega)
    ctx.sketch(0, m, 0)
    A, sc = standardized(codes)
    G = A @ omega
    H = A.T @ G
    # The device sums sc (v / 4) w, sc (1/2 - F) w and, per missing entry, the latter taken back: each entry
    # counts at most sc (1/2 + 1/2 + 1/2) |w|, also where the row has nothing but missing entries.  n (m) FP64
    # sums of such terms, a handful of operations each.
    u = 8 * 2.0**-53
    g_terms = 1.5 * sc[:, None] * np.abs(omega).sum(0)
    g_bound = u * n * g_terms
    assert (np.abs(ctx.get_g(0, m, L) - G) / g_bound).max() <= 1.0
    h_bound = u * m * 1.5 * (sc @ np.abs(G)) + 1.5 * (sc @ g_bound)
    assert (np.abs(ctx.get_h(0, L) - H) / h_bound).max() <= 1.0


@pytest.mark.parametrize("form", ["fp32", "bf16", "fp16", "fp8", "int8"])
@pytest.mark.parametrize("miss", [0.0, 0.1])
def test_cut_windows_match_whole_ones(ctx, form, miss):
    """H of a window that starts and ends between the pieces' aligned stores (every offset of 8 bytes, one and two
    64-row tiles, one row) after a longer window has filled the same buffer: the same operand pieces, hence the same
    G, and zeros around them, hence H as from that window's matrix alone."""
    say(f"cut windows {form} miss={miss}")
    rng = np.random.default_rng(7)
    n, m, L = 130, 700, 20
    codes = random_codes(rng, m, n, miss)
    ctx.upload_packed(pack(codes), n)
    ctx.standardize()
    ctx.configure(form, L)
    ctx.set_omega(rng.standard_normal((n, L)))
    A, sc = standardized(codes)
    for j0, j1 in ((1, 64), (2, 130), (3, 68), (4, 5), (261, 389), (262, 330), (263, 520), (519, 700), (5, 690)):
        ctx.sketch(0, m, 0)
        ctx.sketch(j0, j1, 0)
        G, H = ctx.get_g(j0, j1, L), ctx.get_h(0, L)
        # H = A^T G in 32-bit sums over j1 - j0 rows: each step rounds sums of at most sc (1/2 + 1/2) |G|, and one
        # product more for the centering; FP8 and INT8 give G as the sum of its pieces, so that H's operand is G
        bound = (j1 - j0 + 2) * 2.0**-23 * (1.5 * sc[j0:j1] @ np.abs(G))
        assert (np.abs(H - A[j0:j1].T @ G) / bound).max() <= 1.0, (j0, j1)


@pytest.mark.parametrize("miss", [0.0, 0.1])
def test_zeroed_h1_and_h2(ctx, miss):
    """H1 and H2 after zero_h: read back as zeros, the first window written, the second added, also when the zeroed
    one is summed into H untouched."""
    say(f"zeroed H1, H2 miss={miss}")
    rng = np.random.default_rng(3)
    n, m, L = 70, 300, 12
    ctx.upload_packed(pack(random_codes(rng, m, n, miss)), n)
    ctx.standardize()
    ctx.configure("fp64", L)
    ctx.set_omega(rng.standard_normal((n, L)))
    ctx.sketch(0, 130, 0)
    a = ctx.get_h(0, L)
    ctx.sketch(130, m, 0)
    b = ctx.get_h(0, L)
    for which in (1, 2):
        ctx.sketch(0, m, which)  # what zeroing has to undo
        ctx.zero_h(which)
        assert not ctx.get_h(which, L).any()
        ctx.zero_h(which)
        ctx.sketch(0, 130, which)
        np.testing.assert_array_equal(ctx.get_h(which, L), a)
        ctx.sketch(130, m, which)
        if not miss:  # a window's correction is a sum of its own: (a + dense part) + correction
            np.testing.assert_array_equal(ctx.get_h(which, L), a + b)
        ctx.zero_h(which)
    ctx.sketch(0, 130, 1)
    ctx.update_omega(1)  # H = H1 + H2
    np.testing.assert_array_equal(ctx.get_h(0, L), a)


@pytest.mark.parametrize("n,m,L", [(18, 200, 16), (65, 300, 20), (1023, 1200, 40), (1030, 700, 64), (4097, 500, 80),
                                   (20011, 300, 33), (130, 400, 100)])
def test_omega_update(ctx, n, m, L):
    """Two Omega updates (thin-Q with Householder's column signs, then flipOmg) against LAPACK's Q, seen through
    the next G = A Omega: L below, at and past the 16-column blocks, N below and past the row blocks."""
    say(f"omega update n={n} m={m} L={L}")
    rng = np.random.default_rng(n + L)
    codes = random_codes(rng, m, n, 0.0)
    # a planted structure: the columns of successive Q then agree up to their signs
    for g in range(5):
        codes[g * m // 6:(g + 1) * m // 6, g * n // 6:(g + 1) * n // 6] = rng.choice([0, 2], (m // 6 + 1, n // 6 + 1))[
            :(g + 1) * m // 6 - g * m // 6, :(g + 1) * n // 6 - g * n // 6]
    A, _ = standardized(codes)
    omega = rng.standard_normal((n, L))
    ctx.upload_packed(pack(codes), n)
    ctx.standardize()
    ctx.configure("fp64", L)
    ctx.set_omega(omega)
    ref, amplify = omega, 1.0
    for _ in range(2):
        ctx.sketch(0, m, 0)
        ctx.update_omega(0)
        H = A.T @ (A @ ref)
        Q = np.linalg.qr(H)[0]
        flip = np.abs(ref - Q).sum(0) > 2 * np.abs(ref + Q).sum(0)
        ref = np.where(flip, -Q, Q)
        amplify *= 1.0 + np.linalg.cond(H)
    ctx.sketch(0, m, 0)
    G = A @ ref
    # each thin-Q is within a moderate multiple of u cond(H) of the exact one, and the next starts from it
    err = np.abs(ctx.get_g(0, m, L) - G).max() / np.abs(G).max()
    assert err <= 1e4 * 2.0**-53 * amplify


@pytest.mark.parametrize("m,k", [(60, 3), (65, 1), (1000, 10), (16385, 2), (40001, 16)])
def test_emu_flip_uv(ctx, m, k):
    """flip_UV with V as the base after every EM iteration: V's entry of largest magnitude is positive in every
    column, and U went with it (A V points along U)."""
    say(f"flip_UV m={m} k={k}")
    n = 90
    rng = np.random.default_rng(m + k)
    codes = random_codes(rng, m, n, 0.05)
    for g in range(k):
        codes[g::k + 1, g * n // (k + 1):(g + 1) * n // (k + 1)] = rng.choice([0, 2])
    ctx.upload_packed(pack(codes), n)
    r = ctx.run(svd=1, k=k, oversamples=10, emu=1, maxiter=2, printv=1, precision="fp64", want_v=True)
    V, U = r.V, r.U
    assert np.all(V[np.abs(V).argmax(0), np.arange(k)] > 0)
    A, _ = standardized(codes)
    assert np.all(((A.T @ V) * U).sum(0) > 0)


@pytest.mark.parametrize("n,m,L", [(150, 33, 1), (150, 300, 17), (150, 1025, 128), (150, 20001, 128)])
def test_read_back(ctx, n, m, L):
    """G and H read back column-major: whole and in windows, below and past the 32-row tiles and the 8 MB slots."""
    say(f"read back n={n} m={m} L={L}")
    rng = np.random.default_rng(m + L)
    codes = random_codes(rng, m, n, 0.0)
    omega = rng.standard_normal((n, L))
    ctx.upload_packed(pack(codes), n)
    ctx.standardize()
    ctx.configure("fp64", L)
    ctx.set_omega(omega)
    ctx.sketch(0, m, 0)
    A, _ = standardized(codes)
    G = ctx.get_g(0, m, L)
    ref = A @ omega
    assert np.abs(G - ref).max() <= 1e-12 * np.abs(ref).max()  # a placement test: FP64 sums of 150 terms
    for j0, j1 in [(0, 1), (1, 33), (m // 3, m), (m - 1, m)]:
        np.testing.assert_array_equal(ctx.get_g(j0, j1, L), G[j0:j1])
    H = A.T @ ref
    assert np.abs(ctx.get_h(0, L) - H).max() <= 1e-12 * np.abs(H).max()


@pytest.mark.parametrize("svd,m", [(1, 40), (2, 2049)])
def test_loadings_order(ctx, svd, m):
    """Loadings come back in the original SNP order, with and without winSVD's shuffle: V S = A U."""
    say(f"loadings svd={svd} m={m}")
    n, k = 120, 3
    rng = np.random.default_rng(m)
    codes = random_codes(rng, m, n, 0.0)
    for g in range(3):
        codes[g::4, g * 30:g * 30 + 30] = 2 * (g % 2)
    ctx.upload_packed(pack(codes), n)
    r = ctx.run(svd=svd, k=k, oversamples=10, maxp=30, tol=1e-12, bands=8, precision="fp64", want_v=True)
    A, _ = standardized(codes)
    proj = A @ r.U
    # V is G~'s own left factor: it agrees with A U up to the convergence of the subspace
    for c in range(k):
        assert np.dot(r.V[:, c], proj[:, c]) / np.linalg.norm(proj[:, c]) >= 0.999


@pytest.mark.parametrize("form,tol", [("fp64", 1e-10), ("fp8", 1e-4)])
def test_batch_row_slices(ctx, form, tol):
    """Cohorts whose rows fall on and beside the batched kernels' slices (128), items (1,024) and sums of 128
    items, against the single-matrix FP64 runs."""
    dims = [(20, 127), (127, 128), (128, 129), (129, 1023), (1024, 1024), (1025, 16385), (2049, 40), (4100, 300)]
    say(f"batch row slices {form}")
    rng = np.random.default_rng(5)
    cohorts = []
    for n, m in dims:
        codes = random_codes(rng, m, n, 0.0)
        codes[: m // 3, : n // 3] = 0
        codes[m // 2:, n // 2:] = 3
        cohorts.append((pack(codes), n))
    k = 3
    kw = dict(svd=1, k=k, oversamples=10, maxp=5, tol=0.0)
    ctx.batch_upload(cohorts)
    r = ctx.batch_run(precision=form, kchunk_g=4096, kchunk_h=8192, **kw)
    assert np.all(r["status"] == 0)
    for c, (rows, n) in enumerate(cohorts):
        ctx.upload_packed(rows, n)
        one = ctx.run(precision="fp64", **kw)
        np.testing.assert_allclose(r["S"][c], one.S, rtol=tol)
        U = ctx.batch_get_u(c)
        # the two structured components, which the passes have converged
        assert np.all(np.abs((U * one.U).sum(0))[:2] >= 1 - tol)


@pytest.mark.parametrize("k,os", [(1, 10), (5, 10), (5, 11), (6, 11), (10, 11), (10, 21), (16, 16)])
def test_batch_small_steps(ctx, k, os):
    """The batched L x L steps at L = 11 .. 32, odd and even, beside and past the 16-pivot panels: all singular
    values, U and V of a cohort against the single-matrix FP64 run (host eigen-solver, other L x L kernels)."""
    L = k + max(k, os)
    say(f"batch small steps L={L}")
    rng = np.random.default_rng(L)
    n, m = 300, 900
    codes = random_codes(rng, m, n, 0.0)
    for g in range(5):
        codes[g::6, g * 50:g * 50 + 50 - 7 * g] = 2 * (g % 2)
    kw = dict(svd=1, k=k, oversamples=os, maxp=4, tol=0.0, precision="fp64")
    ctx.batch_upload([(pack(codes), n)])
    r = ctx.batch_run(want_v=True, **kw)
    assert r["status"][0] == 0 and r["epochs"][0] == 5
    ctx.upload_packed(pack(codes), n)
    one = ctx.run(want_v=True, **kw)
    # both solve the same L x L problems in FP64; neighbouring noise components are a percent apart
    np.testing.assert_allclose(r["S"][0], one.S, rtol=1e-11)
    for x, y in ((ctx.batch_get_u(0), one.U), (ctx.batch_get_v(0), one.V)):
        np.testing.assert_allclose(np.abs((x * y).sum(0)), 1.0, rtol=1e-9)
    np.testing.assert_allclose(ctx.batch_trace(0), one.trace, atol=1e-11)


@pytest.mark.parametrize("form,L", [(f, L) for f in ("fp32", "fp64") for L in (17, 20, 21, 28, 29, 33, 36, 40, 41)] +
                         [("fp64", L) for L in (44, 45, 49, 60, 61)])
@pytest.mark.parametrize("nrows,ncodes", [(1, 255), (511, 257), (513, 1000)])
def test_short_column_blocks(ctx, form, L, nrows, ncodes):
    """The FP32 and FP64 products with their last columns in groups of 4 (L = 17..28, 33..40; FP64 also 41..44 and
    49..60) and beside those ranges, exact on values whose products and sums FP32 holds."""
    say(f"{form} columns L={L} nrows={nrows} ncodes={ncodes}")
    rng = np.random.default_rng(nrows + ncodes + L)
    codes = rng.integers(0, 4, (nrows, ncodes)).astype(np.uint8)
    W = rng.integers(-64, 64, (ncodes, L)) / 8.0
    Y = ctx.packed_gemm(form, pack(codes), ncodes, W)
    np.testing.assert_array_equal(Y, np.array([2.0, 0.0, 0.0, -2.0])[codes] @ W)


@pytest.mark.parametrize("k", [10, 20])
def test_fp32_column_groups_same_bits(ctx, k):
    """The 4-column groups add the same products in the same order as the 16-column blocks: whole runs agree to the
    bit with workgroup shapes that take the blocks alone (32-row waves), missing genotypes and windows included."""
    say(f"fp32 column groups k={k}")
    rng = np.random.default_rng(k)
    n, m = 700, 3001
    codes = random_codes(rng, m, n, 0.01)
    for g in range(3):
        codes[g::5, g * 200:g * 200 + 150] = 2 * (g % 2)
    ctx.upload_packed(pack(codes), n)
    for svd in (1, 2):
        runs = [ctx.run(svd=svd, k=k, oversamples=10, maxp=3, tol=0.0, bands=4, precision="fp32", want_v=True, wm_g=wm,
                        wm_h=wm, waves_g=wv, waves_h=wv, kchunk_g=512, kchunk_h=1024)
                for wm, wv in ((2, 4), (4, 4), (4, 8))]
        for r in runs[1:]:
            np.testing.assert_array_equal(r.S, runs[0].S)
            np.testing.assert_array_equal(r.U, runs[0].U)
            np.testing.assert_array_equal(r.V, runs[0].V)


@pytest.mark.parametrize("form,L,wide", [("fp64", 17, 32), ("fp64", 20, 32), ("fp64", 28, 32), ("fp64", 36, 48),
                                         ("fp64", 44, 48), ("fp64", 52, 64), ("fp64", 60, 64), ("fp32", 20, 32),
                                         ("fp32", 25, 32), ("fp32", 40, 48)])
def test_column_groups_same_bits_as_whole_blocks(ctx, form, L, wide):
    """A product of L columns (the last ones in groups of 4) and the same W with more columns (16-column blocks
    alone): the first L columns are the same bits, on values whose sums round at every step."""
    say(f"{form} columns {L} of {wide}")
    rng = np.random.default_rng(L)
    nrows, ncodes = 513, 1000
    rows = pack(rng.integers(0, 4, (nrows, ncodes)).astype(np.uint8))
    W = rng.standard_normal((ncodes, wide)) * np.exp(3 * rng.standard_normal((ncodes, 1)))
    whole = ctx.packed_gemm(form, rows, ncodes, W)
    np.testing.assert_array_equal(ctx.packed_gemm(form, rows, ncodes, np.ascontiguousarray(W[:, :L])), whole[:, :L])


@pytest.mark.parametrize("miss", [0.0, 0.05])
def test_overflowing_pieces_stay_infinite(ctx, miss):
    """FP16 pieces of diag(sc) G beyond 65,504 are infinite, and so is G, with its sign, as the piece divided by sc."""
    say(f"overflowing pieces miss={miss}")
    rng = np.random.default_rng(9)
    n, m, L = 130, 300, 20
    codes = random_codes(rng, m, n, miss)
    ctx.upload_packed(pack(codes), n)
    ctx.standardize()
    ctx.configure("fp16", L)
    omega = 1500 * rng.standard_normal((n, L))
    ctx.set_omega(omega)
    ctx.sketch(0, m, 0)
    A, sc = standardized(codes)
    exact = A @ omega
    G = ctx.get_g(0, m, L)
    # Omega's FP16 rounding moves sc G by at most 2^-11 sc |A| |Omega| <= a few units of 1,000: 10,000 apart
    size = np.abs(sc[:, None] * exact)
    over, under = size > 75000, size < 55000
    assert over.any() and under.any()
    np.testing.assert_array_equal(G[over], np.copysign(np.inf, exact[over]))
    bound = 2.0**-10 * (np.abs(A) @ np.abs(omega))
    assert (np.abs(G - exact) / bound)[under].max() <= 1.0


@pytest.mark.parametrize("form", ["fp8", "int8"])
def test_tiny_columns_keep_their_digits(ctx, form):
    """Column scales whose reciprocal overflows: a column of Omega near the smallest FP64 numbers gives the G of the
    same column at an ordinary size, scaled."""
    say(f"tiny columns {form}")
    rng = np.random.default_rng(10)
    n, m, L = 130, 300, 20
    codes = random_codes(rng, m, n, 0.0)
    ctx.upload_packed(pack(codes), n)
    ctx.standardize()
    ctx.configure(form, L)
    omega = rng.standard_normal((n, L))
    ctx.set_omega(omega)
    ctx.sketch(0, m, 0)
    G = ctx.get_g(0, m, L)
    small = omega.copy()
    small[:, 3] *= 2.0**-1020
    ctx.set_omega(small)
    ctx.sketch(0, m, 0)
    T = ctx.get_g(0, m, L)
    np.testing.assert_array_equal(np.delete(T, 3, 1), np.delete(G, 3, 1))
    # the scale itself has 2^-1074 steps there: 2^-40 of its size at the least, and G's a few dozen more
    A, _ = standardized(codes)
    bound = 2.0**-12 * (np.abs(A) @ np.abs(omega[:, 3]))
    assert (np.abs(np.ldexp(T[:, 3], 1020) - G[:, 3]) / bound).max() <= 1.0


def free_memory():
    free, total = C.c_size_t(), C.c_size_t()
    assert _lib.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # of the runtime that the library has loaded
    return free.value


def test_batch_read_back_takes_no_device_memory(ctx):
    """U and V of every cohort, twice, in any order, in the memory that the run left: the device's free memory stays,
    and so do the results and those of the next run."""
    say("batch read back in place")
    rng = np.random.default_rng(12)
    k = 16
    kw = dict(svd=1, k=k, oversamples=10, maxp=2, tol=0.0, precision="fp32", kchunk_g=4096, kchunk_h=8192)
    ctx.batch_upload([(pack(random_codes(rng, m, n, 0.0)), n) for n, m in [(60, 100000), (40000, 50), (300, 700)]])
    first = ctx.batch_run(want_v=True, **kw)
    assert np.all(first["status"] == 0)
    before = free_memory()
    got = [(ctx.batch_get_u(c), ctx.batch_get_v(c)) for c in range(3)]
    assert free_memory() >= before
    for c in (2, 0, 1):
        np.testing.assert_array_equal(ctx.batch_get_v(c), got[c][1])
        np.testing.assert_array_equal(ctx.batch_get_u(c), got[c][0])
    again = ctx.batch_run(want_v=True, **kw)
    np.testing.assert_array_equal(again["S"], first["S"])
    for c in range(3):
        np.testing.assert_array_equal(ctx.batch_get_u(c), got[c][0])
        np.testing.assert_array_equal(ctx.batch_get_v(c), got[c][1])
        assert np.abs(got[c][1].T @ got[c][1] - np.eye(k)).max() < 1e-4  # whole columns of whole matrices


def test_permuted_loadings_take_no_device_memory():
    """Loadings of a shuffled run of more SNPs than one part of the positions holds (2 (2,048 256 + 2 128^2)): in
    the memory of the run without them, every SNP in its place."""
    n, m, k = 24, 1150000, 2
    say(f"permuted loadings m={m}")
    rng = np.random.default_rng(13)
    codes = random_codes(rng, m, n, 0.0)
    codes[::2, : n // 2] = 0
    codes[1::3, n // 2:] = 3
    kw = dict(svd=2, k=k, oversamples=10, maxp=6, tol=0.0, bands=4, precision="fp64")
    with api.Context(0) as ctx:
        ctx.upload_packed(pack(codes), n)
        ctx.run(**kw)
        before = free_memory()
        r = ctx.run(want_v=True, **kw)
        assert free_memory() >= before
    A, _ = standardized(codes)
    proj = A @ r.U
    for c in range(k):
        assert np.dot(r.V[:, c], proj[:, c]) / np.linalg.norm(proj[:, c]) >= 0.999
        tail = slice(m - 30000, m)  # past the first part
        assert np.corrcoef(r.V[tail, c], proj[tail, c])[0, 1] >= 0.99


@pytest.mark.parametrize("L,rows", [(1, 6553), (1, 6554), (16, 1638), (16, 1639), (20, 1170), (20, 1171), (100, 256),
                                    (100, 257)])
def test_read_back_on_both_sides_of_the_direct_rows(ctx, L, rows):
    """Reads of as many rows as are still transposed on the host, and of one more (rows (pitch + 4 k) about 131,072):
    the same values as in a read of all."""
    say(f"read back L={L} rows={rows}")
    rng = np.random.default_rng(rows)
    n, m = 150, 8000
    ctx.upload_packed(pack(random_codes(rng, m, n, 0.0)), n)
    ctx.standardize()
    ctx.configure("fp64", L)
    ctx.set_omega(rng.standard_normal((n, L)))
    ctx.sketch(0, m, 0)
    G = ctx.get_g(0, m, L)
    np.testing.assert_array_equal(ctx.get_g(0, rows, L), G[:rows])
    np.testing.assert_array_equal(ctx.get_g(m - rows, m, L), G[m - rows:])


@pytest.mark.parametrize("m", [3640, 3641])
def test_shuffled_loadings_on_both_sides_of_the_direct_rows(ctx, m):
    """Loadings of a shuffled run, placed on the host (m (32 + 4) <= 131,072) and on the device."""
    say(f"shuffled loadings m={m}")
    n, k = 120, 1
    rng = np.random.default_rng(m)
    codes = random_codes(rng, m, n, 0.0)
    codes[::2, : n // 3] = 0
    ctx.upload_packed(pack(codes), n)
    r = ctx.run(svd=2, k=k, oversamples=19, maxp=20, tol=1e-12, bands=8, precision="fp64", want_v=True)
    A, _ = standardized(codes)
    proj = A @ r.U
    assert np.corrcoef(r.V[:, 0], proj[:, 0])[0, 1] >= 0.999
