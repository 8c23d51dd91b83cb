"""ttdft_ham_apply_noalloc against ttdft_ham_apply, through the C ABI.

The allocation-free entry point runs the same kernels with the nonlocal
projections in the library's static per-GPU work space, so its result must
equal ttdft_ham_apply's bit for bit (a split dense or block product whose partial
sums do not fit that work space takes fewer parts, or one kernel, and agrees to
rounding).  Two calls in a row, the second on a
smaller input (fewer basis functions, projectors and states), show that the
work space left by one call does not leak into the next.
"""
import numpy as np
import pytest

from ttdft_public_amd import engine as E

pytestmark = pytest.mark.gpu


def _apply_both(c, ham, n, k, ld, dtype, seed):
    npdt = np.float64 if dtype == E.F64 else np.float32
    X = np.random.default_rng(seed).standard_normal((n, ld)).astype(npdt)
    dX = E.DeviceArray.from_host(c, X, npdt)
    dY = E.DeviceArray.from_host(c, np.full((n, ld), 3.0, npdt), npdt)
    dZ = E.DeviceArray.from_host(c, np.full((n, ld), 5.0, npdt), npdt)
    c.ham_apply(ham, dX.ptr, ld, dY.ptr, ld, k, dtype)
    c.ham_apply_noalloc(ham, dX.ptr, ld, dZ.ptr, ld, k, dtype)
    Y = dY.to_host().reshape(n, ld)
    Z = dZ.to_host().reshape(n, ld)
    for d in (dX, dY, dZ):
        d.free()
    return Y, Z


@pytest.mark.parametrize("dtype", [E.F64, E.F32])
def test_noalloc_matches_ham_apply_two_calls(dtype):
    c = E.Context(0)
    try:
        # band format with projectors (the work space holds W and its split partials)
        big = E.SynthHam(12, 10, 9, 3, 3, 3, 9, seed=31)
        ham = c.ham_upload(big, E.HAM_F64 | E.HAM_F32)
        assert ham.format()[0] == 1
        print(f"noalloc call 1: n={big.n} p=9 k=300 dtype={dtype}", flush=True)
        Y, Z = _apply_both(c, ham, big.n, 300, 301, dtype, 1)
        assert np.array_equal(Y[:, :300], Z[:, :300])
        assert np.all(Z[:, 300:] == 5.0)
        ham.free()
        # smaller: fewer functions, projectors and states; CSR format
        small = E.SynthHam(6, 5, 7, 2, 2, 2, 3, seed=32)
        ham = c.ham_upload(small, E.HAM_F64 | E.HAM_F32, tucker=False)
        print(f"noalloc call 2: n={small.n} p=3 k=40 dtype={dtype}", flush=True)
        Y, Z = _apply_both(c, ham, small.n, 40, 40, dtype, 2)
        assert np.array_equal(Y, Z)
        ham.free()
    finally:
        c.close()


def test_noalloc_dense_storage():
    """Dense storage folds C^T D C into H, so no work space is used."""
    c = E.Context(0)
    try:
        s = E.SynthHam(9, 8, 7, 8, 7, 6, 5, seed=17)
        ham = c.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=False)
        assert ham.format()[0] == 2
        for dtype in (E.F64, E.F32):
            Y, Z = _apply_both(c, ham, s.n, 96, 96, dtype, 3)
            assert np.array_equal(Y, Z)
        ham.free()
    finally:
        c.close()


def test_noalloc_dense_storage_past_the_work_space():
    """A dense product whose partial sums (41 MB here for four parts in FP64)
    exceed the static work space takes fewer parts: it agrees with
    ttdft_ham_apply up to the order of the additions."""
    c = E.Context(0)
    try:
        s = E.SynthHam(30, 30, 30, 14, 14, 14, 55, seed=3)
        ham = c.ham_upload(s, E.HAM_F64 | E.HAM_F32, tucker=False)
        assert ham.format()[0] == 2
        k = 48
        assert 4 * s.n * k * 8 > 32 << 20
        for dtype, tol in ((E.F64, 1e-13), (E.F32, 1e-5)):
            print(f"noalloc dense past the work space: n={s.n} k={k} dtype={dtype}", flush=True)
            Y, Z = _apply_both(c, ham, s.n, k, k, dtype, 4)
            Y, Z = Y.astype(np.float64), Z.astype(np.float64)
            assert np.abs(Y - Z).max() <= tol * np.abs(Y).max()
        ham.free()
    finally:
        c.close()


def _csr_blocks(c, n, half, copies, p=3, rows=()):
    """Banded CSR whose 32 x 32 blocks are full enough to be stored, `rows` full."""
    rng = np.random.default_rng(n)
    col = [np.arange(n) if r in rows else np.arange(max(0, r - half), min(n, r + half + 1))
           for r in range(n)]
    rowptr = np.concatenate([[0], np.cumsum([len(x) for x in col])])
    crp = 50 * np.arange(p + 1)
    ccol = np.concatenate([100 + 60 * q + np.arange(50) for q in range(p)])
    return E.Hamiltonian(c, n, rowptr, np.concatenate(col).astype(np.int32),
                         rng.standard_normal(rowptr[-1]), p, crp, ccol.astype(np.int32),
                         rng.standard_normal(50 * p), rng.standard_normal(p), copies=copies)


def _dense(c, n, copies, p=3):
    rng = np.random.default_rng(n)
    crp, ccol = 50 * np.arange(p + 1), np.tile(np.arange(50, dtype=np.int32), p)
    return E.Hamiltonian(c, n, np.arange(n + 1, dtype=np.int64) * n,
                         np.tile(np.arange(n, dtype=np.int32), n),
                         rng.standard_normal(n * n) / np.sqrt(n), p, crp, ccol,
                         rng.standard_normal(50 * p), rng.standard_normal(p), copies=copies)


@pytest.mark.parametrize("form", ["blocks", "dense"])
@pytest.mark.parametrize("dtype", [E.F64, E.F32])
@pytest.mark.parametrize("k", [40, 97])
def test_noalloc_split_products(monkeypatch, form, dtype, k):
    """The block and the split dense product with all they need in the static
    work space, behind the projections (the dense one in FP32 only: an FP32-only
    matrix keeps its projectors apart), leading dimension above k."""
    c = E.Context(0)
    try:
        copies = E.HAM_F64 if dtype == E.F64 else E.HAM_F32
        n = 1000
        ham = _csr_blocks(c, n, 9, copies) if form == "blocks" else _dense(c, n, copies)
        monkeypatch.setenv("TTDFT_DENSE_LDS", "3")
        Y, Z = _apply_both(c, ham, n, k, k + 3, dtype, 5)
        assert np.array_equal(Y[:, :k], Z[:, :k])
        assert np.all(Z[:, k:] == 5.0)
        ham.free()
    finally:
        c.close()


@pytest.mark.parametrize("form,n,k", [("dense", 4300, 240), ("blocks", 40000, 24)])
def test_noalloc_takes_the_parts_that_fit(monkeypatch, form, n, k):
    """Split products whose parts do not all fit the static work space keep those
    that do (dense: 5 parts of 8.3 MB; blocks: 16 parts of 7.7 MB as 32 full rows
    make one long list) rather than fall back to one kernel: not the one-kernel
    form's bits, but its result."""
    c = E.Context(0)
    try:
        if form == "dense":
            ham = _dense(c, n, E.HAM_F64)
        else:
            ham = _csr_blocks(c, n, 6, E.HAM_F64, rows=range(64, 96))
        Y, Z = _apply_both(c, ham, n, k, k, E.F64, 6)
        if form == "dense":
            monkeypatch.setenv("TTDFT_DENSE_LDS", "0")
            one = _apply_both(c, ham, n, k, k, E.F64, 6)[0]
            differ = not np.array_equal(one, Z)
        else:  # the row kernel takes the first seven states
            X = np.random.default_rng(6).standard_normal((n, k))
            dX = E.DeviceArray.from_host(c, X[:, :7].copy(), np.float64)
            dY = E.DeviceArray(c, (n, 7))
            c.ham_apply(ham, dX.ptr, 7, dY.ptr, 7, 7, E.F64)
            differ = not np.array_equal(dY.to_host().reshape(n, 7), Z[:, :7])
        assert differ
        assert np.abs(Y - Z).max() <= 1e-13 * np.abs(Y).max()
        ham.free()
    finally:
        c.close()
