"""aclblasSgetrfBatched for 256 < n: blocked over many workgroups per matrix, bit-identical to the oracle's
unblocked order (every multiplier a / p and every update fma(-l, u, a) in ascending column order).

Sizes at the edges of the 32-column panels and update strips, of one and two rows per thread (1024 panel rows) and
of the path itself (2048 / 2049); row padding; exact zero pivots at the start, inside and at the end of a panel
(info, pivots and stopping state); no pivoting with and without info; exact ties and NaN columns.
"""
import numpy as np
import pytest

import aclblas as B
import oracle as O
from common import to_dev, to_host

pytestmark = pytest.mark.gpu


def _getrf(handle, A, pivot=True, info=True):
    import torch
    dA = to_dev(A)
    batch, n, lda = A.shape
    piv = torch.full((batch, n), -7, dtype=torch.int32, device="cuda") if pivot else None
    inf = torch.full((batch,), -1, dtype=torch.int32, device="cuda") if info else None
    pa = B.ptr_array(dA)
    st = B.sgetrf_batched(handle.value, n, pa.data_ptr(), lda, piv.data_ptr() if pivot else None,
                          inf.data_ptr() if info else None, batch)
    assert st == 0
    torch.cuda.synchronize()
    return to_host(dA), to_host(piv) if pivot else None, to_host(inf) if info else None


def _random(n, batch, pad=0, seed=0, shift=0.0):
    rng = np.random.default_rng(seed + n)
    A = rng.standard_normal((batch, n, n + pad)).astype(np.float32)
    i = np.arange(n)
    A[:, i, i] += np.float32(shift)
    return A


def _check(A, got, pivot=True):
    LU, piv, info = got
    n = A.shape[1]
    gLU, gpiv, ginfo = O.getrf_batched(A.copy(), pivot=pivot)
    assert np.array_equal(LU[:, :, :n], gLU[:, :, :n], equal_nan=True)
    assert np.array_equal(LU[:, :, n:], A[:, :, n:])
    if info is not None:
        assert np.array_equal(info, ginfo)
    for b in range(A.shape[0]):
        if pivot:
            done = n if ginfo[b] == 0 else int(ginfo[b])
            assert np.array_equal(piv[b, :done], gpiv[b, :done])
            assert (piv[b, done:] == -7).all()


@pytest.mark.parametrize("n,batch,pad", [(257, 3, 0), (287, 2, 5), (288, 2, 0), (289, 9, 1), (320, 1, 0), (511, 2, 3),
                                         (1000, 2, 0), (1024, 1, 0), (1057, 1, 2), (1090, 1, 0)])
def test_large_lu_bitwise(handle, n, batch, pad):
    A = _random(n, batch, pad)
    _check(A, _getrf(handle, A))


@pytest.mark.parametrize("n", [2048, 2049])
def test_large_lu_path_edge(handle, n):
    """Either side of the last order of the blocked path: P A = L U and multipliers at most 1."""
    A = _random(n, 1, shift=2.0)
    LU, piv, info = _getrf(handle, A)
    assert info[0] == 0
    M = LU[0].T.astype(np.float64)
    L, U = np.tril(M, -1) + np.eye(n), np.triu(M)
    P = A[0].T.astype(np.float64)
    for k in range(n):
        r = piv[0, k] - 1
        P[[k, r]] = P[[r, k]]
    assert np.abs(np.tril(M, -1)).max() <= 1.0
    # |P A - L U| <= gamma_n |L| |U| entry by entry (FP32 multiply-adds, n of them)
    gamma = (n + 2) * 2.0 ** -24
    assert (np.abs(P - L @ U) <= 1.01 * gamma * (np.abs(L) @ np.abs(U))).all()


@pytest.mark.parametrize("zero_col", [0, 31, 32, 45, 290, 299])
def test_large_lu_zero_pivot_state(handle, zero_col):
    A = _random(300, 3, shift=2.0)
    A[1, zero_col, :] = 0.0
    _check(A, _getrf(handle, A))


@pytest.mark.parametrize("info", [True, False])
def test_large_lu_without_pivoting(handle, info):
    A = _random(333, 2, 2, shift=400.0)
    _check(A, _getrf(handle, A, pivot=False, info=info), pivot=False)
    A[0, 40, :] = 0.0     # stops inside the second panel
    _check(A, _getrf(handle, A, pivot=False, info=info), pivot=False)


def test_large_lu_ties_and_nan(handle):
    rng = np.random.default_rng(3)
    A = rng.integers(-2, 3, size=(2, 300, 300)).astype(np.float32)
    _check(A, _getrf(handle, A))
    A = _random(300, 2)
    A[0, 5, 17] = np.nan
    A[1, 100, 100:] = np.nan
    _check(A, _getrf(handle, A))


@pytest.mark.parametrize("n,batch", [(66, 1030), (127, 3), (128, 1025), (192, 3), (192, 770), (193, 515)])
def test_blocked_lu_instances(handle, n, batch):
    """64 < n <= 256: the instances of the blocked kernel (largest order 128, 192, 256) at their edges, with batches
    past the persistent grid of each.  Pivots as the oracle's, P A = L U to the multiply-adds' rounding."""
    A = _random(n, batch, shift=float(n) ** 0.5)
    LU, piv, info = _getrf(handle, A)
    assert not info.any()
    some = np.unique(np.linspace(0, batch - 1, 9).astype(int))
    _, gpiv, _ = O.getrf_batched(A[some].copy())
    assert np.array_equal(piv[some], gpiv)
    gamma = (n + 2) * 2.0 ** -24
    for b in some:
        M = LU[b].T.astype(np.float64)
        L, U = np.tril(M, -1) + np.eye(n), np.triu(M)
        P = A[b].T.astype(np.float64)
        for k in range(n):
            P[[k, piv[b, k] - 1]] = P[[piv[b, k] - 1, k]]
        # U12 = inv(L11) A12 with an explicit inverse: its rounding is of the same order with |inv(L11)| |L11| terms
        Li = np.abs(np.linalg.inv(L))
        bound = 4 * gamma * (np.abs(L) @ Li @ np.abs(L) @ np.abs(U))
        assert (np.abs(P - L @ U) <= bound).all()
