"""HIP engine vs the CPU oracle on identical seeded inputs, through the C ABI.

Tolerances: FP64 paths agree to rounding (relative 1e-12 or tighter; the
summation order differs between the GPU kernels and the oracle); the FP32
SpMM to 1e-5 relative; split-BF16 Gram/rotation to 5e-5 relative.
"""
import numpy as np
import pytest

import oracle
from ttdft_public_amd import engine as E

pytestmark = pytest.mark.gpu


def dev(ctx, a, dtype=np.float64):
    return E.DeviceArray.from_host(ctx, np.ascontiguousarray(a, dtype=dtype))


def synth(p=5, dims=(8, 8, 8), bands=(2, 2, 3), seed=7):
    s = E.SynthHam(*dims, *bands, p, seed=seed)
    return s, oracle.Ham.from_synth(s)


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


# ---------------------------------------------------------------- H apply
@pytest.mark.parametrize("k", [1, 7, 64, 65, 130, 300])
def test_ham_apply_f64(ctx, k):
    s, H = synth()
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32)
    X = np.random.default_rng(k).standard_normal((s.n, k))
    dX, dY = dev(ctx, X), E.DeviceArray(ctx, (s.n, k))
    ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, E.F64)
    assert rel(dY.to_host(), oracle.ham_apply(H, X)) < 1e-13


@pytest.mark.parametrize("k", [5, 64, 300])
def test_ham_apply_f32(ctx, k):
    s, H = synth()
    ham = ctx.ham_upload(s, E.HAM_F32)
    X = np.random.default_rng(k).standard_normal((s.n, k)).astype(np.float32)
    dX, dY = dev(ctx, X, np.float32), E.DeviceArray(ctx, (s.n, k), np.float32)
    ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, E.F32)
    assert rel(dY.to_host().astype(np.float64), oracle.ham_apply(H, X.astype(np.float64))) < 1e-5


@pytest.mark.parametrize("k", [1, 70, 300])
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_ham_apply_wide_projectors(ctx, k, dtype):
    """Few projectors with ~1300 nonzeros each: the projection is split over blocks."""
    s, H = synth(p=4, dims=(20, 18, 16), bands=(2, 2, 2), seed=1)
    assert s.nnz_c // 4 > 1024
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=True)
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = np.random.default_rng(k).standard_normal((s.n, k)).astype(npdt)
    dX, dY = dev(ctx, X, npdt), E.DeviceArray(ctx, (s.n, k), npdt)
    ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, dtype)
    ref = oracle.ham_apply(H, X.astype(np.float64))
    assert rel(dY.to_host().astype(np.float64), ref) < (1e-13 if dtype == E.F64 else 1e-5)


def test_ham_apply_ragged_and_no_projectors(ctx):
    """Empty rows, a single dense row, p = 0, leading dimension > k."""
    n = 200
    rng = np.random.default_rng(3)
    rows = []
    for i in range(n):
        if i % 7 == 0:
            rows.append([])
        elif i == 5:
            rows.append(list(range(n)))
        else:
            rows.append(sorted(set(rng.integers(0, n, size=rng.integers(1, 90)).tolist())))
    # symmetrise the pattern with random values
    A = np.zeros((n, n))
    for i, cs in enumerate(rows):
        for c in cs:
            A[i, c] = A[c, i] = rng.standard_normal()
    rowptr = np.zeros(n + 1, np.int64)
    cols, vals = [], []
    for i in range(n):
        nz = np.nonzero(A[i])[0]
        cols.extend(nz.tolist())
        vals.extend(A[i, nz].tolist())
        rowptr[i + 1] = len(cols)
    ham = E.Hamiltonian(ctx, n, rowptr, np.array(cols, np.int32), np.array(vals), 0, None, None,
                        None, None)
    k, ld = 70, 80
    X = rng.standard_normal((n, ld))
    dX, dY = dev(ctx, X), dev(ctx, np.full((n, ld), 7.0))
    ctx.ham_apply(ham, dX.ptr, ld, dY.ptr, ld, k, E.F64)
    Y = dY.to_host()
    assert rel(Y[:, :k], A @ X[:, :k]) < 1e-13
    assert np.all(Y[:, k:] == 7.0)  # padding columns untouched


def test_ham_upload_rejects_bad_csr(ctx):
    with pytest.raises(E.TtdftError) as ei:
        E.Hamiltonian(ctx, 3, np.array([0, 1, 2, 3]), np.array([0, 5, 2], np.int32),
                      np.ones(3), 0, None, None, None, None)
    assert ei.value.status == E.EBADARG


# ---------------------------------------------------------------- band format
@pytest.mark.parametrize("dims,bands,k", [((11, 9, 7), (3, 2, 2), 16), ((20, 10, 6), (2, 3, 1), 64),
                                          ((12, 12, 12), (6, 6, 7), 100),
                                          ((50, 6, 5), (6, 2, 2), 300),
                                          ((70, 5, 4), (3, 1, 1), 40),    # two x-chunks
                                          ((6, 7, 5), (1, 2, 2), 33),     # padded narrow chunk
                                          ((17, 9, 8), (7, 3, 2), 81),    # widest x band
                                          ((22, 6, 5), (2, 2, 1), 50),    # two split x-bricks
                                          ((12, 12, 12), (6, 6, 7), 900),  # 900 states: 3 / 12 groups
                                          ((17, 9, 8), (7, 3, 2), 900)])
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_band_spmm_matches_oracle(ctx, dims, bands, k, dtype):
    s = E.SynthHam(*dims, *bands, 4, seed=sum(dims))
    H = oracle.Ham.from_synth(s)
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=True)
    fmt, b = ham.format()
    assert fmt == 1 and b == tuple(bands)
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = np.random.default_rng(k).standard_normal((s.n, k)).astype(npdt)
    dX, dY = dev(ctx, X, npdt), E.DeviceArray(ctx, (s.n, k), npdt)
    ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, dtype)
    ref = oracle.ham_apply(H, X.astype(np.float64))
    assert rel(dY.to_host().astype(np.float64), ref) < (1e-13 if dtype == E.F64 else 1e-5)


@pytest.mark.parametrize("dims,bands", [((20, 18, 16), (6, 6, 7)), ((13, 11, 9), (7, 3, 2)),
                                         ((9, 10, 7), (1, 2, 2))])
@pytest.mark.parametrize("k", [257, 300, 400])
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_band_spmm_state_groups_in_one_workgroup(ctx, monkeypatch, dims, bands, k, dtype):
    """More than 4 state groups' worth of states (FP64 > 256, FP32 > 240) runs
    all state groups of a row block in one workgroup (x-chunks of 3 or 4
    bricks, the last one ragged); it must give the same bits as one workgroup
    per state group, and match the oracle."""
    s = E.SynthHam(*dims, *bands, 4, seed=sum(dims) + k)
    H = oracle.Ham.from_synth(s)
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=True)
    assert ham.format()[0] == 1
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = np.random.default_rng(k).standard_normal((s.n, k)).astype(npdt)
    dX, dY = dev(ctx, X, npdt), E.DeviceArray(ctx, (s.n, k), npdt)
    out = {}
    for co in ("1", "0"):
        monkeypatch.setenv("TTDFT_BRICK_COGROUPS", co)
        ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, dtype)
        out[co] = dY.to_host()
    assert np.array_equal(out["1"], out["0"])
    ref = oracle.ham_apply(H, X.astype(np.float64))
    assert rel(out["1"].astype(np.float64), ref) < (1e-13 if dtype == E.F64 else 1e-5)


@pytest.mark.parametrize("dims,bands,k", [((20, 18, 16), (6, 6, 7), 300),
                                          ((13, 11, 9), (7, 3, 2), 320),
                                          ((9, 10, 7), (1, 2, 2), 257),
                                          ((17, 9, 5), (7, 3, 2), 80),
                                          ((22, 6, 3), (2, 2, 1), 50)])
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_band_spmm_two_planes_per_workgroup(ctx, monkeypatch, dims, bands, k, dtype):
    """Workgroups over two z planes (a staged line serves both planes in its
    z band) give the same bits as one plane per workgroup, odd plane counts
    included (the last workgroup has one plane), and match the oracle."""
    s = E.SynthHam(*dims, *bands, 4, seed=sum(dims) + k)
    H = oracle.Ham.from_synth(s)
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=True)
    assert ham.format()[0] == 1
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = np.random.default_rng(k).standard_normal((s.n, k)).astype(npdt)
    dX, dY = dev(ctx, X, npdt), E.DeviceArray(ctx, (s.n, k), npdt)
    out = {}
    for zb in ("1", "2"):
        monkeypatch.setenv("TTDFT_BRICK_ZB", zb)
        print(f"band two planes dims={dims} k={k} dtype={dtype} zb={zb}", flush=True)
        ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, dtype)
        out[zb] = dY.to_host()
    assert np.array_equal(out["1"], out["2"])
    ref = oracle.ham_apply(H, X.astype(np.float64))
    assert rel(out["2"].astype(np.float64), ref) < (1e-13 if dtype == E.F64 else 1e-5)


def test_band_filter_with_holes_matches_oracle(ctx):
    """Truncation leaves holes inside the band: stored as zeros, same result."""
    s = E.SynthHam(10, 10, 10, 4, 4, 4, 6, truncation=2e-5, seed=3)
    H = oracle.Ham.from_synth(s)
    ham = ctx.ham_upload(s, tucker=True)
    assert ham.format()[0] == 1
    assert s.nnz < 1000 * 9 ** 3  # some entries were truncated
    k, m = 48, 9
    X = np.random.default_rng(2).standard_normal((s.n, k))
    dX = dev(ctx, X)
    ctx.cheb_filter(ham, dX.ptr, k, k, m, -0.5, 30.0, -3.0, 2, E.F64)
    ref = oracle.cheb_filter(H, X, m, -0.5, 30.0, -3.0, 2)
    assert rel(dX.to_host(), ref) < 1e-12


def test_band_rejects_sparse_band_keeps_csr(ctx):
    """A band with too few entries stays in CSR (and stays correct)."""
    n = 6 * 6 * 6
    rows = [[i, (i + 7 * 36) % n] for i in range(n)]  # far coupling -> wide, empty band
    A = np.zeros((n, n))
    for i, cs in enumerate(rows):
        for c in cs:
            A[i, c] = A[c, i] = 1.0 + 0.01 * i
    rowptr = np.zeros(n + 1, np.int64)
    cols, vals = [], []
    for i in range(n):
        nz = np.nonzero(A[i])[0]
        cols += nz.tolist()
        vals += A[i, nz].tolist()
        rowptr[i + 1] = len(cols)
    ham = E.Hamiltonian(ctx, n, rowptr, np.array(cols, np.int32), np.array(vals), 0, None, None,
                        None, None, dims=(6, 6, 6))
    assert ham.format()[0] == 0
    X = np.random.default_rng(1).standard_normal((n, 32))
    dX, dY = dev(ctx, X), E.DeviceArray(ctx, (n, 32))
    ctx.ham_apply(ham, dX.ptr, 32, dY.ptr, 32, 32)
    assert rel(dY.to_host(), A @ X) < 1e-13


# ---------------------------------------------------------------- filter
@pytest.mark.parametrize("convention", [E.DEGREE_REFERENCE, E.DEGREE_EXACT])
@pytest.mark.parametrize("m,nb", [(1, 1), (2, 1), (5, 1), (8, 3)])
def test_cheb_filter_f64(ctx, convention, m, nb):
    s, H = synth()
    ham = ctx.ham_upload(s)
    k = 24
    X = np.random.default_rng(m).standard_normal((s.n, k))
    a, b, a0 = -5.0, 20.0, -30.0
    dX = dev(ctx, X)
    ctx.cheb_filter(ham, dX.ptr, k, k, m, a, b, a0, nb, E.F64, convention)
    ref = oracle.cheb_filter(H, X, m, a, b, a0, nb, convention)
    assert rel(dX.to_host(), ref) < 1e-12


def test_cheb_filter_f32(ctx):
    s, H = synth()
    ham = ctx.ham_upload(s, E.HAM_F32)
    k, m = 40, 10
    X = np.random.default_rng(9).standard_normal((s.n, k)).astype(np.float32)
    dX = dev(ctx, X, np.float32)
    ctx.cheb_filter(ham, dX.ptr, k, k, m, -5.0, 20.0, -30.0, 1, E.F32)
    ref = oracle.cheb_filter(H, X.astype(np.float64), m, -5.0, 20.0, -30.0)
    assert rel(dX.to_host().astype(np.float64), ref) < 5e-5


# ---------------------------------------------------------------- dense
@pytest.mark.parametrize("n,k", [(512, 24), (3000, 65), (5000, 300)])
def test_gram_f64(ctx, n, k):
    rng = np.random.default_rng(n + k)
    X, Y = rng.standard_normal((n, k)), rng.standard_normal((n, k))
    dS = E.DeviceArray(ctx, (k, k))
    dX, dY = dev(ctx, X), dev(ctx, Y)  # keep the buffers alive through the call
    ctx.gram(dX.ptr, k, dY.ptr, k, n, k, dS.ptr)
    S = dS.to_host().T  # column-major on device
    assert rel(S, oracle.gram(X, Y)) < 1e-13


@pytest.mark.parametrize("n,k,ld,same", [(5000, 300, 300, True), (5000, 300, 300, False),
                                          (3001, 161, 163, True), (3001, 161, 163, False),
                                          (777, 333, 333, True), (100, 17, 17, False),
                                          (20000, 900, 900, True), (40, 160, 161, False)])
def test_gram_f64_shapes(ctx, n, k, ld, same):
    """FP64 Gram over its tilings (160-wide blocks, 16-row steps staged in LDS):
    ragged k and n, odd leading dimension (scalar loads), fewer rows than
    one step.  X^T X takes the upper-triangle form and is exactly
    symmetric."""
    rng = np.random.default_rng(n + k + same)
    X = rng.standard_normal((n, ld))
    Y = X if same else rng.standard_normal((n, ld))
    dX = dev(ctx, X)
    dY = dX if same else dev(ctx, Y)
    dS = E.DeviceArray(ctx, (k, k))
    print(f"gram f64 n={n} k={k} ld={ld} same={same}", flush=True)
    ctx.gram(dX.ptr, ld, dY.ptr, ld, n, k, dS.ptr)
    S = dS.to_host().reshape(k, k).T
    assert rel(S, oracle.gram(np.ascontiguousarray(X[:, :k]), np.ascontiguousarray(Y[:, :k]))) \
        < 1e-13
    if same:
        assert np.array_equal(S, S.T)


@pytest.mark.parametrize("n,k,ld", [(1000, 24, 24), (5001, 131, 133), (3000, 300, 301),
                                     (2000, 300, 300), (129, 17, 20), (700, 900, 900)])
def test_rotate_f64_shapes(ctx, n, k, ld):
    """FP64 rotation from pre-arranged Q fragments: several groups of eight
    column tiles, k not a multiple of 16 or 4, odd leading dimension (scalar
    loads), n not a multiple of the 128-row workgroup.  Columns past k are
    left alone."""
    rng = np.random.default_rng(n + k + ld)
    X = rng.standard_normal((n, ld))
    Q = rng.standard_normal((k, k)) / np.sqrt(k)
    dX = dev(ctx, X)
    dQ = dev(ctx, Q.T.copy())  # column-major
    print(f"rotate f64 n={n} k={k} ld={ld}", flush=True)
    ctx.rotate(dX.ptr, ld, n, k, dQ.ptr, E.F64, E.GEMM_F64)
    got = dX.to_host().reshape(n, ld)
    assert rel(got[:, :k], oracle.rotate(np.ascontiguousarray(X[:, :k]), Q)) < 1e-13
    assert np.array_equal(got[:, k:], X[:, k:])


@pytest.mark.parametrize("n,k", [(512, 24), (5000, 300)])
def test_gram_bf16x3(ctx, n, k):
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, k)).astype(np.float32)
    Y = rng.standard_normal((n, k)).astype(np.float32)
    dS = E.DeviceArray(ctx, (k, k))
    dX, dY = dev(ctx, X, np.float32), dev(ctx, Y, np.float32)
    ctx.gram(dX.ptr, k, dY.ptr, k, n, k, dS.ptr, E.F32, E.GEMM_BF16X3)
    ref = X.astype(np.float64).T @ Y.astype(np.float64)
    # error relative to the natural scale sqrt(n) of a Gram entry
    assert np.abs(dS.to_host().T - ref).max() / np.sqrt(n) < 5e-5


@pytest.mark.parametrize("n,k,ld,same", [(5000, 300, 300, True), (5000, 300, 300, False),
                                          (3001, 161, 163, True), (3001, 161, 163, False),
                                          (777, 333, 336, True), (100, 17, 17, False),
                                          (20000, 900, 900, True), (40, 160, 160, False)])
def test_gram_bf16x3_shapes(ctx, n, k, ld, same):
    """Split-BF16 Gram over its tilings: one to six 160-wide blocks per
    dimension, k not a multiple of 16 or of 4, rows not 16-byte aligned (odd
    leading dimension: scalar loads), n below one 16-row step and not a
    multiple of it.  X^T X (same pointer) runs the upper-triangle form and
    must come out exactly symmetric.

    The bar is elementwise against |X|^T |Y|: the three-term split drops
    lo*lo' (up to 2^-18 of each product) and rounds x = hi + lo to ~2^-17,
    which on the diagonal of X^T X is a one-signed bias growing with n (a
    numpy emulation of the split on the 5000 x 300 case gives 3.1e-6 of
    |X|^T |X|, the same 0.0155 maximum error the kernel shows), so the
    sqrt(n) scale of a random-sign sum does not bound it."""
    rng = np.random.default_rng(n + k + same)
    X = rng.standard_normal((n, ld)).astype(np.float32)
    Y = X if same else rng.standard_normal((n, ld)).astype(np.float32)
    dX = dev(ctx, X, np.float32)
    dY = dX if same else dev(ctx, Y, np.float32)
    dS = E.DeviceArray(ctx, (k, k))
    print(f"gram bf16x3 n={n} k={k} ld={ld} same={same}", flush=True)
    ctx.gram(dX.ptr, ld, dY.ptr, ld, n, k, dS.ptr, E.F32, E.GEMM_BF16X3)
    S = dS.to_host().reshape(k, k).T
    X64, Y64 = X[:, :k].astype(np.float64), Y[:, :k].astype(np.float64)
    ref = X64.T @ Y64
    scale = np.abs(X64).T @ np.abs(Y64)
    assert np.all(np.abs(S - ref) <= 1e-5 * scale + 1e-12)
    if same:
        assert np.array_equal(S, S.T)


@pytest.mark.parametrize("n,k,ld", [(1000, 24, 24), (5001, 131, 133), (3000, 300, 301),
                                     (2000, 300, 300), (129, 17, 20)])
def test_rotate_bf16x3_shapes(ctx, n, k, ld):
    """Split-BF16 rotation over its tilings: several groups of eight column
    tiles (k = 300), k not a multiple of 16, rows not 16-byte aligned
    (odd leading dimension: scalar loads), n not a multiple of the 128-row
    workgroup.  Columns past k are left alone."""
    rng = np.random.default_rng(n + k)
    X = rng.standard_normal((n, ld)).astype(np.float32)
    Q = rng.standard_normal((k, k)) / np.sqrt(k)
    dX = dev(ctx, X, np.float32)
    dQ = dev(ctx, Q.T.copy())  # column-major
    print(f"rotate bf16x3 n={n} k={k} ld={ld}", flush=True)
    ctx.rotate(dX.ptr, ld, n, k, dQ.ptr, E.F32, E.GEMM_BF16X3)
    got = dX.to_host().reshape(n, ld).astype(np.float64)
    ref = oracle.rotate(X[:, :k].astype(np.float64), Q)
    assert rel(got[:, :k], ref) < 5e-5
    assert np.array_equal(got[:, k:], X[:, k:].astype(np.float64))


@pytest.mark.parametrize("k", [1, 32, 33, 64, 65, 255, 319, 320, 321])
@pytest.mark.parametrize("n", [1, 31, 33, 128, 129])
def test_rotate_in_place_edges(ctx, n, k):
    """The in-place form (up to 320 columns) at the edges of its 32-row waves,
    128-row workgroups, 32-deep steps and 64-column variants, with aligned and
    odd leading dimensions; columns past k stay as they are.  Split-BF16: a
    value less its hi half is at most 2^-8 of it, so a product leaves out
    lo lo' (2^-16) and the roundings of both lo halves (2^-17 each)."""
    rng = np.random.default_rng(n * 1000 + k)
    Q = rng.standard_normal((k, k))
    for ld in (k, (k + 8) // 4 * 4, k + 1):
        X = rng.standard_normal((n, ld)).astype(np.float32)
        dX, dQ = dev(ctx, X, np.float32), dev(ctx, Q.T.copy())
        print(f"rotate in place n={n} k={k} ld={ld}", flush=True)
        ctx.rotate(dX.ptr, ld, n, k, dQ.ptr, E.F32, E.GEMM_BF16X3)
        Z = dX.to_host().reshape(n, ld)
        assert rel(Z[:, :k].astype(np.float64), X[:, :k].astype(np.float64) @ Q) < 2.0 ** -15
        assert np.array_equal(Z[:, k:], X[:, k:])


@pytest.mark.parametrize("mode", [E.GEMM_F64, E.GEMM_BF16X3])
def test_rotate_and_orth(ctx, mode):
    n, k = 4000, 100
    rng = np.random.default_rng(mode)
    f32 = mode == E.GEMM_BF16X3
    dt, npdt = (E.F32, np.float32) if f32 else (E.F64, np.float64)
    X = rng.standard_normal((n, k)).astype(npdt)
    Q = rng.standard_normal((k, k))
    dX = dev(ctx, X, npdt)
    dQ = dev(ctx, Q.T.copy())  # column-major
    ctx.rotate(dX.ptr, k, n, k, dQ.ptr, dt, mode)
    ref = oracle.rotate(X.astype(np.float64), Q)
    tol = 1e-13 if not f32 else 5e-5
    assert rel(dX.to_host().astype(np.float64), ref) < tol
    ctx.orth(dX.ptr, k, n, k, dt, mode)
    Xo = dX.to_host().astype(np.float64)
    # Cholesky-QR leaves an orthogonality error of order eps * cond(X)^2
    assert np.abs(Xo.T @ Xo - np.eye(k)).max() < (1e-10 if not f32 else 1e-5)
    # same span as the input
    assert np.abs(Xo @ (Xo.T @ ref) - ref).max() / np.abs(ref).max() < (1e-11 if not f32 else 1e-4)


@pytest.mark.parametrize("k", [40, 64, 80])  # k <= 64: one-workgroup Cholesky inverse
def test_orth_matches_oracle_f64(ctx, k):
    n = 2000
    X = np.random.default_rng(1).standard_normal((n, k))
    dX = dev(ctx, X)
    ctx.orth(dX.ptr, k, n, k)
    assert rel(dX.to_host(), oracle.orth(X)) < 1e-11


@pytest.mark.parametrize("k", [1, 31, 32, 33, 63, 65, 96, 97, 300, 513])
def test_orth_block_columns_of_the_factorisation(ctx, k):
    """Cholesky inverse by 32 columns a launch: one block, remainders of 1 and
    31, many blocks, against numpy on a block of condition about 20 (squared
    in the overlap: 400 eps, times the growth of sums over k)."""
    n = k + 700
    rng = np.random.default_rng(k)
    X = rng.standard_normal((n, k)) * np.linspace(1.0, 0.1, k)
    dX = dev(ctx, X)
    ctx.orth(dX.ptr, k, n, k)
    L = np.linalg.cholesky(X.T @ X)
    assert rel(dX.to_host(), np.linalg.solve(L, X.T).T) < 1e-12


@pytest.mark.parametrize("k,col", [(8, 5), (80, 0), (80, 31), (80, 32), (80, 79), (300, 290)])
@pytest.mark.parametrize("f32", [False, True])
def test_orth_not_spd_in_any_block(ctx, k, col, f32):
    """A zero column gives an exactly zero pivot in whichever launch meets it;
    X is left as it was, also where the rotation runs in place (FP32)."""
    npdt = np.float32 if f32 else np.float64
    X = np.random.default_rng(2).standard_normal((600, k)).astype(npdt)
    X[:, col] = 0.0
    dX = dev(ctx, X, npdt)
    with pytest.raises(E.TtdftError) as ei:
        ctx.orth(dX.ptr, k, 600, k, E.F32 if f32 else E.F64,
                 E.GEMM_BF16X3 if f32 else E.GEMM_F64)
    assert ei.value.status == E.ENOTSPD and f"minor {col + 1}" in str(ei.value)
    assert np.array_equal(dX.to_host(), X)


def test_orth_not_spd_reports_error(ctx):
    n, k = 300, 8
    X = np.random.default_rng(2).standard_normal((n, k))
    X[:, 5] = 0.0  # singular overlap: pivot 5 is exactly zero
    dX = dev(ctx, X)
    with pytest.raises(E.TtdftError) as ei:
        ctx.orth(dX.ptr, k, n, k)
    assert ei.value.status in (E.ENOTSPD,)


@pytest.mark.parametrize("k", [1, 7, 24, 64, 65, 300])  # k <= 64: one-workgroup Jacobi
def test_rr_eig(ctx, k):
    A = np.random.default_rng(k).standard_normal((k, k))
    A = A + A.T
    dA = dev(ctx, A.T.copy())
    dE, dQ = E.DeviceArray(ctx, (k,)), E.DeviceArray(ctx, (k, k))
    ctx.rr_eig(dA.ptr, k, dE.ptr, dQ.ptr)
    w = dE.to_host()
    Q = dQ.to_host().T
    wo, Qo = oracle.syev(A)
    assert np.abs(w - wo).max() < 1e-12 * np.abs(wo).max()
    assert np.abs(A @ Q - Q * w).max() < 1e-11
    # same eigenvectors up to sign
    assert np.abs(np.abs(np.sum(Q * Qo, axis=0)) - 1).max() < 1e-9


# ---------------------------------------------------------------- Lanczos
@pytest.mark.parametrize("dims,p", [((8, 8, 8), 5), ((20, 18, 16), 4)])
def test_lanczos_matches_oracle(ctx, dims, p):
    s, H = synth(p=p, dims=dims, bands=(2, 2, 2))
    ham = ctx.ham_upload(s)
    up, lo = ctx.lanczos_bounds(ham, 20, seed=11)
    upo, loo = oracle.lanczos_bounds(H, 20, seed=11)
    assert abs(up - upo) < 1e-9 * abs(upo) and abs(lo - loo) < 1e-9 * abs(loo)


# ---------------------------------------------------------------- density
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_density(ctx, dtype):
    rng = np.random.default_rng(5)
    rx, ry, rz = 6, 5, 7
    px, py, pz = 70, 33, 20
    Bx, By, Bz = (rng.standard_normal((p, r)) for p, r in ((px, rx), (py, ry), (pz, rz)))
    k = 21
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = rng.standard_normal((rx * ry * rz, k)).astype(npdt)
    occ = np.linspace(1.0, 0.0, k)  # last state has zero weight
    dRho = E.DeviceArray(ctx, (pz, py, px))
    dX = dev(ctx, X, npdt)
    dBx, dBy, dBz = dev(ctx, Bx.T.copy()), dev(ctx, By.T.copy()), dev(ctx, Bz.T.copy())
    ctx.density(dX.ptr, k, k, occ, (rx, ry, rz), dBx.ptr, dBy.ptr, dBz.ptr, (px, py, pz),
                dRho.ptr, dtype)
    ref = oracle.density(X.astype(np.float64), occ, (rx, ry, rz), Bx, By, Bz)
    got = dRho.to_host()
    # an FP32 block is contracted in FP32 up to the y-factor density matrices
    tol = 1e-12 if dtype == E.F64 else 1e-5
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < tol


@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_density_chunked_with_sparse_weights(ctx, monkeypatch, dtype):
    """Several qz chunks, zero weights scattered among the states, ry > rx, rz."""
    monkeypatch.setenv("TTDFT_DENSITY_PLANES", "4")
    rng = np.random.default_rng(11)
    rx, ry, rz = 9, 17, 5
    px, py, pz = 40, 31, 23
    Bx, By, Bz = (rng.standard_normal((p, r)) for p, r in ((px, rx), (py, ry), (pz, rz)))
    k = 37
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = rng.standard_normal((rx * ry * rz, k + 3)).astype(npdt)  # ld > k
    occ = rng.uniform(0.0, 1.0, k)
    occ[[0, 5, 6, 20, 36]] = 0.0
    dRho = E.DeviceArray(ctx, (pz, py, px))
    dX = dev(ctx, X, npdt)
    dBx, dBy, dBz = dev(ctx, Bx.T.copy()), dev(ctx, By.T.copy()), dev(ctx, Bz.T.copy())
    ctx.density(dX.ptr, k + 3, k, occ, (rx, ry, rz), dBx.ptr, dBy.ptr, dBz.ptr, (px, py, pz),
                dRho.ptr, dtype)
    ref = oracle.density(X[:, :k].astype(np.float64), occ, (rx, ry, rz), Bx, By, Bz)
    got = dRho.to_host()
    tol = 1e-12 if dtype == E.F64 else 1e-5
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < tol


@pytest.mark.parametrize("dtype", [E.F64, E.F32])
@pytest.mark.parametrize("ry", [33, 50, 70, 97, 128])
def test_density_wide_y(ctx, ry, dtype):
    """y ranks spanning 3..8 MFMA row tiles (the y contraction's tile groups)."""
    rng = np.random.default_rng(ry)
    rx, rz = 3, 2
    px, py, pz = 7, 19, 5
    Bx, By, Bz = (rng.standard_normal((p, r)) for p, r in ((px, rx), (py, ry), (pz, rz)))
    k = 22
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = rng.standard_normal((rx * ry * rz, k)).astype(npdt)
    occ = rng.uniform(0.0, 1.0, k)
    dRho = E.DeviceArray(ctx, (pz, py, px))
    dX = dev(ctx, X, npdt)
    dBx, dBy, dBz = dev(ctx, Bx.T.copy()), dev(ctx, By.T.copy()), dev(ctx, Bz.T.copy())
    ctx.density(dX.ptr, k, k, occ, (rx, ry, rz), dBx.ptr, dBy.ptr, dBz.ptr, (px, py, pz),
                dRho.ptr, dtype)
    ref = oracle.density(X.astype(np.float64), occ, (rx, ry, rz), Bx, By, Bz)
    tol = 1e-12 if dtype == E.F64 else 1e-5
    assert np.linalg.norm(dRho.to_host() - ref) / np.linalg.norm(ref) < tol


@pytest.mark.parametrize("dtype", [E.F64, E.F32])
@pytest.mark.parametrize("rx,ry,k", [(13, 16, 9), (30, 20, 17), (50, 40, 8), (61, 64, 33),
                                     (4, 50, 3), (70, 70, 11), (80, 72, 5)])
def test_density_fused_shapes(ctx, monkeypatch, rx, ry, k, dtype):
    """The fused x + y-factor step over its tile classes (a steps of 4, 8, 13, 16, 20; 1-5
    blocks of 16 b; ranks past 64 are fused in FP32 only), a ragged last qx tile and ragged
    state chunks, against the oracle and against the two-step form (x GEMM to memory, then
    the packed y-factor products)."""
    rng = np.random.default_rng(rx * 100 + ry)
    rz = 2
    px, py, pz = 37, 11, 3
    Bx, By, Bz = (rng.standard_normal((p, r)) for p, r in ((px, rx), (py, ry), (pz, rz)))
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = rng.standard_normal((rx * ry * rz, k)).astype(npdt)
    occ = rng.uniform(0.1, 1.0, k)
    dX = dev(ctx, X, npdt)
    dBx, dBy, dBz = dev(ctx, Bx.T.copy()), dev(ctx, By.T.copy()), dev(ctx, Bz.T.copy())
    got = {}
    for fused in ("1", "0"):
        monkeypatch.setenv("TTDFT_DENSITY_FUSED", fused)
        dRho = E.DeviceArray(ctx, (pz, py, px))
        ctx.density(dX.ptr, k, k, occ, (rx, ry, rz), dBx.ptr, dBy.ptr, dBz.ptr, (px, py, pz),
                    dRho.ptr, dtype)
        got[fused] = dRho.to_host()
    ref = oracle.density(X.astype(np.float64), occ, (rx, ry, rz), Bx, By, Bz)
    tol = 1e-12 if dtype == E.F64 else 1e-5
    for f in ("1", "0"):
        assert np.linalg.norm(got[f] - ref) / np.linalg.norm(ref) < tol, f
    assert np.linalg.norm(got["1"] - got["0"]) / np.linalg.norm(ref) < tol


def test_initial_density_and_integrals(ctx):
    r = np.linspace(0.0, 9.0, 901)
    rho_r = np.exp(-r**2) * (1 + 0.3 * r)
    xyz = np.array([[0.3, -0.2, 0.1], [1.7, 0.4, -0.9], [-1.1, 1.2, 0.6]])
    x, w = np.polynomial.legendre.leggauss(40)
    gx, wx = 7.0 * x, 7.0 * w
    gy = np.linspace(-8, 8, 35)
    wy = np.full(35, 16 / 34)
    gz = gx[::2].copy()
    wz = wx[::2].copy()
    dims = (len(gx), len(gy), len(gz))
    dR = E.DeviceArray(ctx, (dims[2], dims[1], dims[0]))
    dgx, dgy, dgz = dev(ctx, gx), dev(ctx, gy), dev(ctx, gz)
    ctx.initial_density(xyz, r, rho_r, dgx.ptr, dgy.ptr, dgz.ptr, dims, dR.ptr)
    ref = oracle.initial_density(xyz, r, rho_r, gx, gy, gz)
    got = dR.to_host()
    assert np.abs(got - ref).max() < 1e-13 * np.abs(ref).max()
    dwx, dwy, dwz = dev(ctx, wx), dev(ctx, wy), dev(ctx, wz)
    q = ctx.grid_integral(dR.ptr, dims, dwx.ptr, dwy.ptr, dwz.ptr)
    assert abs(q - oracle.grid_integral(ref, wx, wy, wz)) < 1e-11 * abs(q)
    dR2 = dev(ctx, ref * 1.01)
    res = ctx.grid_residual(dR.ptr, dR2.ptr, dims, dwx.ptr, dwy.ptr, dwz.ptr)
    assert abs(res - oracle.grid_integral((0.01 * ref) ** 2, wx, wy, wz)) < 1e-10 * res
    ctx.grid_scale(dR.ptr, int(np.prod(dims)), 2.0)
    assert np.abs(dR.to_host() - 2 * ref).max() < 1e-13 * np.abs(ref).max()


# ---------------------------------------------------------------- driver
def test_chfsi_step_matches_oracle(ctx):
    s, H = synth(p=5, seed=21)
    ham = ctx.ham_upload(s)
    k, nocc = 16, 10
    X0 = oracle.orth(oracle.rng_normal(5, s.n * k).reshape(s.n, k))
    Xo = X0.copy()
    evo = np.zeros(k)
    sto = oracle.new_state()
    dX = dev(ctx, X0)
    ev = np.zeros(k)
    st = E.new_state()
    for scf in range(6):
        rt = 10 if scf == 0 else 3
        oracle.chfsi_step(H, Xo, evo, sto, m=12, scf_iter=scf, occ_index=nocc, restart_times=rt)
        ctx.chfsi_step(ham, dX.ptr, k, k, 12, ev, st, scf, nocc, rt)
        assert st.passes == sto.passes and st.lanczos_runs == sto.lanczos_runs
        # occupied + stop-test states agree to rounding; the unconverged top of
        # the block amplifies the different summation orders through the filter
        assert np.abs(ev[: nocc + 1] - evo[: nocc + 1]).max() < 1e-9, scf
        assert np.abs(ev - evo).max() < 1e-6, scf
        assert abs(st.upper - sto.upper) < 1e-8 * abs(sto.upper)
    assert np.abs(ev - evo).max() < 1e-8
    lam = np.linalg.eigvalsh(H.dense())
    assert np.abs(ev[:nocc] - lam[:nocc]).max() < 1e-8
    # band energy and density from the converged subspace
    ef, occ = E.fermi_occupancy(ev, 2 * nocc - 1)
    efo = oracle.fermi_energy(evo, 2 * nocc - 1)
    assert abs(ef - efo) < 1e-8
    X = dX.to_host()
    # subspaces agree (eigenvector signs are free)
    assert np.abs(np.abs(np.sum(X[:, :nocc] * Xo[:, :nocc], axis=0)) - 1).max() < 1e-6


@pytest.mark.parametrize("tucker", [False, True])
def test_dense_storage_matches_oracle(ctx, tucker):
    """A small, nearly full H_loc (every 1-D factor couples all basis
    functions) is stored dense and applied by one matrix product plus the
    fused epilogue: H X, the filter and both precisions against the oracle."""
    s = E.SynthHam(9, 8, 7, 8, 7, 6, 5, seed=17)
    assert s.nnz > 0.2 * s.n ** 2
    H = oracle.Ham.from_synth(s)
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=tucker)
    assert ham.format()[0] == 2
    for dtype, tol in ((E.F64, 1e-13), (E.F32, 1e-5)):
        npdt = np.float64 if dtype == E.F64 else np.float32
        X = np.random.default_rng(4).standard_normal((s.n, 40)).astype(npdt)
        dX, dY = dev(ctx, X, npdt), E.DeviceArray(ctx, (s.n, 40), npdt)
        ctx.ham_apply(ham, dX.ptr, 40, dY.ptr, 40, 40, dtype)
        assert rel(dY.to_host().astype(np.float64), oracle.ham_apply(H, X.astype(np.float64))) < tol
    X = np.random.default_rng(5).standard_normal((s.n, 24))
    dX = dev(ctx, X)
    ctx.cheb_filter(ham, dX.ptr, 24, 24, 8, -0.5, 30.0, -3.0, 1, E.F64)
    assert rel(dX.to_host(), oracle.cheb_filter(H, X, 8, -0.5, 30.0, -3.0, 1)) < 1e-12
    X32 = X.astype(np.float32)
    dX = dev(ctx, X32, np.float32)
    ctx.cheb_filter(ham, dX.ptr, 24, 24, 8, -0.5, 30.0, -3.0, 1, E.F32)
    ref = oracle.cheb_filter(H, X32.astype(np.float64), 8, -0.5, 30.0, -3.0, 1)
    assert rel(dX.to_host().astype(np.float64), ref) < 5e-5


@pytest.mark.parametrize("form", ["0", "-1", "3"])
@pytest.mark.parametrize("dims", [(4, 3, 5), (9, 8, 7), (11, 10, 13)])
@pytest.mark.parametrize("k", [1, 8, 16, 24, 33, 64, 80, 96, 100, 150, 192])
def test_dense_product_tilings(ctx, monkeypatch, dims, k, form):
    """The dense product over its state tilings (16 to 96 states per
    workgroup, one or two workgroup columns, partial tiles), leading dimension
    of the block above k, and n not a multiple of 32, in one kernel (n = 60: six
    of the eight waves get no l range; n = 1430: the last wave's range is
    shorter) and split into one part of up to 45 stages and into three (n = 60:
    two).  An FP32-only matrix keeps its projectors apart."""
    rx, ry, rz = dims
    s = E.SynthHam(rx, ry, rz, rx - 1, ry - 1, rz - 1, 3, seed=k)
    H = oracle.Ham.from_synth(s)
    monkeypatch.setenv("TTDFT_DENSE_LDS", form)
    print(f"dense product n={s.n} k={k} form={form}", flush=True)
    # an odd and an even leading dimension (96-state multiples with an even
    # one take the six-consecutive-states layout)
    for copies, ld, dtype, npdt, tol in (
            (E.HAM_F64 | E.HAM_F32, k + 3, E.F64, np.float64, 1e-13),
            (E.HAM_F64 | E.HAM_F32, k + 3, E.F32, np.float32, 1e-5),
            (E.HAM_F64, k + 4, E.F64, np.float64, 1e-13),
            (E.HAM_F32, k + 4, E.F32, np.float32, 1e-5)):
        ham = ctx.ham_upload(s, copies, tucker=False)
        assert ham.format()[0] == 2
        X = np.random.default_rng(k).standard_normal((s.n, ld)).astype(npdt)
        dX, dY = dev(ctx, X, npdt), dev(ctx, np.full((s.n, ld), 7.0), npdt)
        ctx.ham_apply(ham, dX.ptr, ld, dY.ptr, ld, k, dtype)
        Y = dY.to_host().reshape(s.n, ld).astype(np.float64)
        ref = oracle.ham_apply(H, X[:, :k].astype(np.float64))
        assert rel(Y[:, :k], ref) < tol
        assert np.all(Y[:, k:] == 7.0)  # columns past k untouched
        ham.free()


@pytest.mark.parametrize("n", [1, 31, 33, 127, 129, 255, 257, 300])
@pytest.mark.parametrize("k", [1, 17, 96, 97])
def test_dense_product_row_blocks_and_parts(ctx, monkeypatch, n, k):
    """Row blocks of 128 (FP64) and 256 (FP32) rows, stages of 32 columns and
    one to three parts of them at their edges, in a filter whose steps hand
    the block on as operand fragments.  FP32 keeps FP32 accuracy: m - 1 steps
    with sums of n products each, an error of 2^-24 per operation that adds
    up like a random walk, times the filter's growth (4 here)."""
    rng = np.random.default_rng(n + k)
    A = rng.standard_normal((n, n)) / np.sqrt(n)
    A = A + A.T
    ham = E.Hamiltonian(ctx, n, np.arange(n + 1, dtype=np.int64) * n,
                        np.tile(np.arange(n, dtype=np.int32), n), A.reshape(-1), 0, None, None,
                        None, None, copies=E.HAM_F64 | E.HAM_F32)
    assert ham.format()[0] == 2
    X = rng.standard_normal((n, k))
    m, a, b, a0 = 4, -1.0, 3.0, -3.0
    e, c = (b - a) / 2, (b + a) / 2
    for dtype, npdt, tol in ((E.F64, np.float64, 1e-13),
                             (E.F32, np.float32, 4 * 2.0 ** -24 * np.sqrt(3.0 * n + 16))):
        Xc = X.astype(npdt)
        A_c = A.astype(npdt).astype(np.float64)
        sigma = e / (a0 - c)
        gamma = 2.0 / sigma
        prev = Xc.astype(np.float64)
        cur = (sigma / e) * (A_c @ prev - c * prev)
        for _ in range(2, m):
            nxt = 1.0 / (gamma - sigma)
            prev, cur = cur, (2 * nxt / e) * (A_c @ cur - c * cur) - sigma * nxt * prev
            sigma = nxt
        for parts in ("-1", "2", "3"):
            monkeypatch.setenv("TTDFT_DENSE_LDS", parts)
            dX = dev(ctx, Xc, npdt)
            print(f"dense row blocks n={n} k={k} dtype={dtype} parts={parts}", flush=True)
            ctx.cheb_filter(ham, dX.ptr, k, k, m, a, b, a0, 1, dtype)
            assert rel(dX.to_host().astype(np.float64), cur) < tol
    ham.free()


@pytest.mark.parametrize("n", [40, 65, 1030, 1500])
@pytest.mark.parametrize("k", [7, 8, 17, 37, 80, 96, 97])
def test_csr_block_storage(ctx, monkeypatch, n, k):
    """CSR matrices whose 32 x 32 blocks are at least a tenth full, by blocks
    from 8 states on: one and two clumps in a matrix of two and three row tiles,
    one of them empty or of one row (n = 40, 65); bands with holes, a row and a
    whole row tile without entries, n past multiples of 16, 32 and 1024, blocks
    cut by the last column (1030); full rows in one tile, 12 parts of partial
    sums (1500); a duplicate entry, a row whose columns descend, projectors; a
    filter with its fused recurrence, leading dimension above k.  FP64 to 1e-13
    (sums of `most` products), FP32 to 8 steps of 2^-24 sqrt(most)."""
    monkeypatch.setenv("TTDFT_CSR_BLOCKS", "1")
    rng = np.random.default_rng(n + k)
    i, j = np.indices((n, n))
    if n < 100:
        on = ((i < 16) & (j < 16)) | ((n > 64) & (i // 16 == 2) & (j // 16 == 2)) | \
            ((n > 64) & (i == 64) & (j == 64))
    else:
        on = (np.abs(i - j) <= (40 if n == 1030 else 9)) & ((i * j) % 7 != 3)
        on &= (i != 5) & (j != 5)
        on &= (i // 32 != 4) & (j // 32 != 4)
        on |= (n == 1500) & (i // 8 == 9)
    A = np.where(on, rng.standard_normal((n, n)), 0.0)
    most = int(on.sum(1).max())
    rowptr, col, val = [0], [], []
    for r in range(n):
        c = np.nonzero(on[r])[0]
        v = A[r, c]
        if r == 3:  # its first entry in two parts
            c, v = np.insert(c, 0, c[0]), np.insert(v, 0, 0.25)
            v[1] -= 0.25
        if r == 9 or r == n - 2:
            c, v = c[::-1], v[::-1]
        col += c.tolist()
        val += v.tolist()
        rowptr.append(len(col))
    col = np.array(col, np.int32)
    tiles = np.repeat(np.arange(n), np.diff(rowptr)) // 32
    blocks = np.unique(tiles * 100 + col // 32)
    assert 0.1 * 1024 * len(blocks) <= len(col) < 0.2 * n * n
    assert n == 65 or len(np.unique(tiles)) < (n + 31) // 32  # an empty tile
    # (a part holds four blocks at least)
    assert n != 1500 or np.bincount(blocks // 100).max() > 44
    C = np.zeros((2, n))
    C[0, :9], C[1, n // 2:n // 2 + 5] = 0.3, -0.2
    cc = [np.nonzero(C[q])[0] for q in range(2)]
    inv = np.array([0.7, -0.4])
    ham = E.Hamiltonian(ctx, n, np.array(rowptr), col, np.array(val), 2,
                        np.array([0, len(cc[0]), len(cc[0]) + len(cc[1])]),
                        np.concatenate(cc).astype(np.int32),
                        np.concatenate([C[0, cc[0]], C[1, cc[1]]]), inv,
                        copies=E.HAM_F64 | E.HAM_F32)
    assert ham.format()[0] == 0
    H = A + C.T @ (inv[:, None] * C)
    ld = k + 3
    X = rng.standard_normal((n, ld))
    a, b, a0 = -2.0, 30.0, -10.0
    e, c0 = (b - a) / 2, (b + a) / 2
    for dtype, npdt, tol in ((E.F64, np.float64, 1e-13),
                             (E.F32, np.float32, 8 * 2.0 ** -24 * np.sqrt(most))):
        Xc = X.astype(npdt)
        sigma = e / (a0 - c0)
        gamma = 2.0 / sigma
        prev = Xc[:, :k].astype(np.float64)
        cur = (sigma / e) * (H @ prev - c0 * prev)
        for _ in range(2, 5):
            nxt = 1.0 / (gamma - sigma)
            prev, cur = cur, (2 * nxt / e) * (H @ cur - c0 * cur) - sigma * nxt * prev
            sigma = nxt
        dX = dev(ctx, Xc, npdt)
        print(f"csr blocks n={n} k={k} dtype={dtype}", flush=True)
        ctx.cheb_filter(ham, dX.ptr, ld, k, 5, a, b, a0, 1, dtype)
        got = dX.to_host().reshape(n, ld)
        assert rel(got[:, :k].astype(np.float64), cur) < tol
        assert np.array_equal(got[:, k:], Xc[:, k:])
    ham.free()


def banded_csr(n, half, seed, rows=()):
    """Symmetric banded CSR with holes; `rows` are full rows (not mirrored)."""
    rng = np.random.default_rng(seed)
    rowptr, col, val = [0], [], []
    for r in range(n):
        c = np.arange(n) if r in rows else np.arange(max(0, r - half), min(n, r + half + 1))
        c = c if r in rows else c[(r * c) % 7 != 3]
        col.append(c)
        val.append(rng.standard_normal(len(c)))
        rowptr.append(rowptr[-1] + len(c))
    return np.array(rowptr, np.int64), np.concatenate(col).astype(np.int32), np.concatenate(val)


def csr_product(n, rowptr, col, val, X):
    """H X in FP64, a row's products added in its order."""
    Y = np.zeros((n, X.shape[1]))
    for r in range(n):
        Y[r] = val[rowptr[r]:rowptr[r + 1]] @ X[col[rowptr[r]:rowptr[r + 1]]]
    return Y


@pytest.mark.parametrize("form", ["blocks", "dense"])
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_split_products_keep_the_rows_infinities(ctx, monkeypatch, form, dtype):
    """Infinities, NaN, the largest numbers and states 2^-115 small through the
    block and the split dense product: every result is what the row's own
    entries give (an infinite state reaches no row without an entry there, and
    stays infinite), and a small state keeps its precision (rounding of sums of
    `most` products in the type, 8 sqrt(most) eps)."""
    npdt, eps = (np.float64, 2.0 ** -53) if dtype == E.F64 else (np.float32, 2.0 ** -24)
    if form == "blocks":
        n, most = 1000, 19
        rowptr, col, val = banded_csr(n, 9, 11)
    else:
        n, most = 300, 300
        rowptr, col = np.arange(n + 1, dtype=np.int64) * n, np.tile(np.arange(n, dtype=np.int32), n)
        val = np.random.default_rng(12).standard_normal(n * n)
        monkeypatch.setenv("TTDFT_DENSE_LDS", "2")
    val = val.astype(npdt).astype(np.float64)
    ham = E.Hamiltonian(ctx, n, rowptr, col, val, 0, None, None, None, None,
                        copies=E.HAM_F64 if dtype == E.F64 else E.HAM_F32)
    k = 40
    X = np.random.default_rng(13).standard_normal((n, k)).astype(npdt)
    X[n // 2, 3] = np.inf
    X[n // 5, 5] = np.nan
    X[n // 3, 7], X[n // 3 + 4, 7] = -np.inf, np.inf
    X[n - 1, 9] = np.finfo(npdt).max
    X[:, 11] *= npdt(2.0 ** -115)
    dX, dY = dev(ctx, X, npdt), dev(ctx, np.full((n, k), 7.0), npdt)
    ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, dtype)
    with np.errstate(all="ignore"):
        ref = csr_product(n, rowptr, col, val, X.astype(np.float64)).astype(npdt)
    got = dY.to_host().reshape(n, k)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    for c in range(k):
        f = np.isfinite(ref[:, c])
        g, r = got[f, c].astype(np.longdouble), ref[f, c].astype(np.longdouble)
        if len(r):
            assert np.abs(g - r).max() <= 8 * eps * np.sqrt(most) * np.abs(r).max(), c
    ham.free()


@pytest.mark.parametrize("copies", [E.HAM_F64, E.HAM_F32, E.HAM_F64 | E.HAM_F32])
def test_csr_without_room_for_blocks(monkeypatch, copies):
    """Block storage (2.3 MB an FP64 copy here, 1.1 MB FP32) that finds no
    memory is left out: the CSR rows (0.7 MB at most an array) apply, with the
    row kernel's bits, as seven columns (always the row kernel) show."""
    n, k = 3000, 20
    rowptr, col, val = banded_csr(n, 15, 5)
    X = np.random.default_rng(6).standard_normal((n, k))
    monkeypatch.setenv("TTDFT_ALLOC_LIMIT", str(1 << 20))
    c = E.Context(0)
    try:
        ham = E.Hamiltonian(c, n, rowptr, col, val, 0, None, None, None, None, copies=copies)
        ref = csr_product(n, rowptr, col, val, X)
        for dtype, npdt, copy, tol in ((E.F64, np.float64, E.HAM_F64, 1e-13),
                                       (E.F32, np.float32, E.HAM_F32, 1e-5)):
            if not copies & copy:
                continue
            got = {}
            for kk in (7, k):
                dX = dev(c, X[:, :kk], npdt)
                dY = E.DeviceArray(c, (n, kk), npdt)
                c.ham_apply(ham, dX.ptr, kk, dY.ptr, kk, kk, dtype)
                got[kk] = dY.to_host()
            assert rel(got[k].astype(np.float64), ref) < tol
            assert np.array_equal(got[k][:, :7], got[7])
        ham.free()
    finally:
        c.close()


@pytest.mark.parametrize("dtype,fewest", [(E.F64, 64), (E.F32, 128)])
def test_csr_product_form_by_states(ctx, monkeypatch, dtype, fewest):
    """Blocks just over a tenth full: few states go by blocks, from `fewest` on
    (one more pass of the row kernel's 64 states or the blocks' 96 aside) by
    rows, each with the bits of the form that the switch takes."""
    n = 4000
    rowptr, col, val = banded_csr(n, 6, 14)
    rows, keep = np.repeat(np.arange(n), np.diff(rowptr)), np.arange(len(col)) % 9 != 0
    rows, col, val = rows[keep], col[keep], val[keep]
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    blocks = len(np.unique(rows // 32 * 125 + col // 32))
    assert 0.1 < len(col) / (1024.0 * blocks) < 0.11
    npdt = np.float64 if dtype == E.F64 else np.float32
    ham = E.Hamiltonian(ctx, n, rowptr, col, val, 0, None, None, None, None,
                        copies=E.HAM_F64 if dtype == E.F64 else E.HAM_F32)
    for k in (8, 16, fewest):
        X = np.random.default_rng(k).standard_normal((n, k)).astype(npdt)
        dX, got = dev(ctx, X, npdt), {}
        for form in (None, "0", "1"):
            if form is not None:
                monkeypatch.setenv("TTDFT_CSR_BLOCKS", form)
            dY = E.DeviceArray(ctx, (n, k), npdt)
            ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, dtype)
            got[form] = dY.to_host()
            monkeypatch.delenv("TTDFT_CSR_BLOCKS", raising=False)
        assert not np.array_equal(got["0"], got["1"])
        assert np.array_equal(got[None], got["0" if k == fewest else "1"]), k
    ham.free()


def test_csr_block_parts_are_bounded(monkeypatch):
    """One row tile that meets every column block among short ones (n = 40,000,
    32 full rows): the block product's partial sums stay within 16 parts of the
    block (350 MB with the operand; by the average list alone, 313 parts and
    6.4 GB), so that it runs, and adds in another order than the row kernel,
    where no more than 400 MiB are to be had."""
    n, k = 40000, 64
    rowptr, col, val = banded_csr(n, 6, 7, rows=range(64, 96))
    X = np.random.default_rng(8).standard_normal((n, k))
    monkeypatch.setenv("TTDFT_ALLOC_LIMIT", str(400 << 20))
    c = E.Context(0)
    try:
        ham = E.Hamiltonian(c, n, rowptr, col, val, 0, None, None, None, None)
        got = {}
        for kk in (7, k):
            dX, dY = dev(c, X[:, :kk]), E.DeviceArray(c, (n, kk))
            c.ham_apply(ham, dX.ptr, kk, dY.ptr, kk, kk, E.F64)
            got[kk] = dY.to_host()
        assert not np.array_equal(got[k][:, :7], got[7])
        # sums of up to 40,000 products of unit normal numbers
        assert rel(got[k], csr_product(n, rowptr, col, val, X)) < 1e-12
        ham.free()
    finally:
        c.close()


@pytest.mark.parametrize("form", ["blocks", "dense"])
def test_filter_without_room_for_partial_sums(monkeypatch, form):
    """Where the split products find no work space (1 MiB at most here; 1.2 MB
    and more needed) the filter runs on the one-kernel products: the row
    kernel's bits, as a Hamiltonian without block storage gives them, or the
    one-kernel dense form's."""
    if form == "blocks":
        n, k = 3000, 20
        rowptr, col, val = banded_csr(n, 15, 5)
    else:
        n, k = 300, 96
        A = np.random.default_rng(9).standard_normal((n, n)) / np.sqrt(n)
        rowptr, col = np.arange(n + 1, dtype=np.int64) * n, np.tile(np.arange(n, dtype=np.int32), n)
        val = (A + A.T).reshape(-1)
    X = np.random.default_rng(10).standard_normal((n, k))
    got = []
    for limited in (False, True):
        c = E.Context(0)
        try:
            if form == "blocks" and not limited:  # no block storage: the row kernel
                monkeypatch.setenv("TTDFT_ALLOC_LIMIT", str(1 << 20))
            ham = E.Hamiltonian(c, n, rowptr, col, val, 0, None, None, None, None)
            monkeypatch.delenv("TTDFT_ALLOC_LIMIT", raising=False)
            dX = dev(c, X)
            if form == "dense":
                monkeypatch.setenv("TTDFT_DENSE_LDS", "16" if limited else "0")
            if limited:
                monkeypatch.setenv("TTDFT_ALLOC_LIMIT", str(1 << 20))
            c.cheb_filter(ham, dX.ptr, k, k, 5, -2.0, 30.0, -10.0, 1, E.F64)
            got.append(dX.to_host())
            monkeypatch.delenv("TTDFT_ALLOC_LIMIT", raising=False)
            ham.free()
        finally:
            c.close()
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("dtype", [E.F64, E.F32])
@pytest.mark.parametrize("p", [4, 60])
@pytest.mark.parametrize("bx,k,ld", [(3, 300, 300), (3, 250, 251), (7, 260, 260), (3, 16, 16),
                                     (2, 16, 17)])
def test_band_epilogue_over_projector_rows(ctx, dtype, p, bx, k, ld):
    """The state-group forms of the band product (aligned rows, unaligned rows,
    the widest band) and one tile of states, the last x-brick's tiles split over
    two waves, with rows of up to four entries of C^T on average and with more,
    in a filter, so that the recurrence is in the epilogue too."""
    s = E.SynthHam(18, 10, 9, bx, 3, 3, p, seed=61)
    assert (s.nnz_c > 4 * s.n) == (p == 60)
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=True)
    assert ham.format()[0] == 1
    npdt, tol = (np.float64, 1e-12) if dtype == E.F64 else (np.float32, 5e-5)
    X = np.random.default_rng(k).standard_normal((s.n, ld)).astype(npdt)
    dX = dev(ctx, X, npdt)
    ctx.cheb_filter(ham, dX.ptr, ld, k, 4, -0.5, 30.0, -3.0, 1, dtype)
    got = dX.to_host().reshape(s.n, ld)
    ref = oracle.cheb_filter(oracle.Ham.from_synth(s),
                             np.ascontiguousarray(X[:, :k]).astype(np.float64), 4, -0.5, 30.0,
                             -3.0, 1)
    assert rel(got[:, :k].astype(np.float64), ref) < tol
    assert np.array_equal(got[:, k:], X[:, k:])
    ham.free()


@pytest.mark.parametrize("dtype", [E.F64, E.F32])
@pytest.mark.parametrize("k,blocks", [(64, 2), (48, 3), (102, 2)])
def test_band_filter_in_column_blocks(ctx, dtype, k, blocks):
    """A band filter in column blocks narrower than the kernel's state tiles (32,
    16 and 51 states): blocks past the first start inside the rows, and the
    last one's rows end where the block's memory ends (2 MiB to the byte for
    4,096 x 64 FP64).  Against the filter in one block and the oracle's."""
    s = E.SynthHam(16, 16, 16, 3, 3, 3, 4, seed=51)
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=True)
    assert ham.format()[0] == 1
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = np.random.default_rng(k).standard_normal((s.n, k)).astype(npdt)
    got = []
    for b in (1, blocks):
        dX = dev(ctx, X, npdt)
        ctx.cheb_filter(ham, dX.ptr, k, k, 6, -0.5, 30.0, -3.0, b, dtype)
        got.append(dX.to_host())
    assert rel(got[1].astype(np.float64), got[0].astype(np.float64)) < 10 * np.finfo(npdt).eps
    ref = oracle.cheb_filter(oracle.Ham.from_synth(s), X.astype(np.float64), 6, -0.5, 30.0, -3.0, 1)
    assert rel(got[1].astype(np.float64), ref) < (1e-12 if dtype == E.F64 else 5e-5)
    ham.free()


def test_dense_storage_reuse_across_hamiltonians(ctx):
    """Hamiltonians of different sizes built and freed in turn on one context:
    the dense storage and the projector fold come from the context's block
    cache (a freed block of the same size class is reused), and every product
    still matches the oracle."""
    for dims in [(9, 8, 7), (4, 3, 5), (11, 10, 13), (9, 8, 7), (8, 8, 8), (4, 3, 5)]:
        s = E.SynthHam(*dims, dims[0] - 1, dims[1] - 1, dims[2] - 1, 5, seed=sum(dims))
        H = oracle.Ham.from_synth(s)
        ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=False)
        assert ham.format()[0] == 2
        X = np.random.default_rng(sum(dims)).standard_normal((s.n, 40))
        dX, dY = dev(ctx, X), E.DeviceArray(ctx, (s.n, 40))
        print(f"reuse n={s.n}", flush=True)
        ctx.ham_apply(ham, dX.ptr, 40, dY.ptr, 40, 40, E.F64)
        assert rel(dY.to_host(), oracle.ham_apply(H, X)) < 1e-13
        ham.free()


@pytest.mark.parametrize("dims,bands,k", [((50, 6, 5), (6, 2, 2), 300), ((22, 9, 7), (3, 2, 3), 81),
                                          ((50, 8, 9), (6, 3, 2), 96)])
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_band_spmm_light_chunks_last_same_bits(ctx, monkeypatch, dims, bands, k, dtype):
    """TTDFT_BRICK_ORDER=1 dispatches the ragged last x-chunk's workgroups
    after all full ones on every XCD; every output is still computed once, by
    the same code: bitwise the default order's result."""
    s = E.SynthHam(*dims, *bands, 4, seed=sum(dims) + k)
    ham = ctx.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=True)
    assert ham.format()[0] == 1
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = np.random.default_rng(k).standard_normal((s.n, k)).astype(npdt)
    dX = dev(ctx, X, npdt)
    out = {}
    for order in ("0", "1"):
        monkeypatch.setenv("TTDFT_BRICK_ORDER", order)
        dY = dev(ctx, np.full((s.n, k), np.nan), npdt)  # every output must be written
        ctx.ham_apply(ham, dX.ptr, k, dY.ptr, k, k, dtype)
        out[order] = dY.to_host()
    assert np.array_equal(out["0"], out["1"])
    if dtype == E.F64:
        H = oracle.Ham.from_synth(s)
        assert rel(out["1"], oracle.ham_apply(H, X)) < 1e-13


@pytest.mark.parametrize("n,k,ld", [(3000, 40, 40), (5000, 300, 301)])
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_random_subspace_matches_oracle(ctx, n, k, ld, dtype):
    """The initial block (main.cc:807-829 with a seeded generator): the
    library's N(0,1) sequence is the oracle's bit for bit, and the block is
    two Cholesky-QR passes of it -- in FP64 the oracle's twice-orthonormalized
    block to 1e-11, in FP32 (split-BF16 Gram, whose XᵀX diagonal carries a
    2^-18 one-signed bias) orthonormal to 3e-5."""
    seed = 1234 + k
    assert np.array_equal(E.rng_normal(seed, 1000), oracle.rng_normal(seed, 1000))
    npdt = np.float64 if dtype == E.F64 else np.float32
    dX = E.DeviceArray(ctx, (n, ld), npdt)
    ctx.random_subspace(dX.ptr, ld, n, k, seed=seed, dtype=dtype)
    X = dX.to_host().reshape(n, ld)[:, :k].astype(np.float64)
    ref = oracle.orth(oracle.orth(oracle.rng_normal(seed, n * k).reshape(n, k)))
    if dtype == E.F64:
        assert rel(X, ref) < 1e-11
    else:
        assert rel(X, ref) < 1e-4
    assert np.abs(X.T @ X - np.eye(k)).max() < (1e-12 if dtype == E.F64 else 3e-5)
