"""aclblasSgetrsBatched (N, T) and aclblasSgetriBatched for orders above 64: bit-identical to the oracle's
column-oriented substitution.

Orders at the edges of the 16-row tiles, of the 64-swap permutation groups, of the two workgroup sizes (256 / 257) and
of the tile path (2048 / 2049), and batches large enough for one wave per 16 right-hand sides (1536 units);
right-hand sides around the 16 of a workgroup; factors and pivots made directly
(pivots at random rows below, some out of range, which the solves skip), padded leading dimensions.
"""
import ctypes

import numpy as np
import pytest

import aclblas as B
import oracle as O
from common import to_dev, to_host

pytestmark = pytest.mark.gpu


def _factors(n, batch, pad, seed):
    rng = np.random.default_rng(seed)
    LU = (rng.standard_normal((batch, n, n + pad)) / np.sqrt(n)).astype(np.float32)
    i = np.arange(n)
    LU[:, i, i] += np.where(LU[:, i, i] >= 0, 1.5, -1.5).astype(np.float32)
    piv = (i + 1 + rng.integers(0, n - i, size=(batch, n))).astype(np.int32)
    piv[:, 3] = n + 5
    piv[:, 7] = 0
    return LU, piv


@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("n,nrhs,batch,pad", [(65, 1, 5, 0), (79, 16, 2, 1), (80, 17, 3, 0), (128, 8, 9, 0),
                                              (129, 33, 2, 3), (256, 5, 2, 0), (257, 16, 2, 0), (500, 3, 2, 2),
                                              (1024, 2, 1, 0), (2048, 3, 1, 0), (2049, 1, 1, 0),
                                              (100, 3, 1601, 1), (200, 19, 800, 0)])
def test_solve_bitwise(handle, trans, n, nrhs, batch, pad):
    import torch
    LU, piv = _factors(n, batch, pad, n + nrhs)
    rng = np.random.default_rng(nrhs)
    rhs = rng.standard_normal((batch, nrhs, n + 2)).astype(np.float32)
    rhs[:, 0, : n // 2] = 0.0
    dA, dB, dp = to_dev(LU), to_dev(rhs), to_dev(piv)
    pa, pb = B.ptr_array(dA), B.ptr_array(dB)
    inf = ctypes.c_int(-1)
    assert B.sgetrs_batched(handle.value, B.OPS[trans], n, nrhs, pa.data_ptr(), n + pad, dp.data_ptr(),
                            pb.data_ptr(), n + 2, inf, batch) == 0
    torch.cuda.synchronize()
    X = to_host(dB)
    gold = O.getrs_batched(0 if trans == "N" else 1, LU, piv, rhs)
    assert np.array_equal(X[:, :, :n], gold[:, :, :n], equal_nan=True)
    assert np.array_equal(X[:, :, n:], rhs[:, :, n:])


@pytest.mark.parametrize("pivot", [True, False])
@pytest.mark.parametrize("n,batch,zero", [(65, 4, None), (100, 3, 40), (144, 2, 143), (257, 2, None), (300, 2, 0),
                                          (72, 400, 71)])
def test_inverse_bitwise(handle, n, batch, zero, pivot):
    import torch
    LU, piv = _factors(n, batch, 1, 7 * n)
    if zero is not None:
        LU[1, zero, zero] = 0.0
    dA, dp = to_dev(LU), to_dev(piv)
    C = torch.full((batch, n, n + 2), 9.0, dtype=torch.float32, device="cuda")
    info = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
    pa, pc = B.ptr_array(dA), B.ptr_array(C)
    assert B.sgetri_batched(handle.value, n, pa.data_ptr(), n + 1, dp.data_ptr() if pivot else None, pc.data_ptr(),
                            n + 2, info.data_ptr(), batch) == 0
    torch.cuda.synchronize()
    got = to_host(C)
    gold, ginfo = O.getri_batched(LU, piv if pivot else None, ldc=n + 2)
    assert np.array_equal(to_host(info), ginfo)
    assert np.array_equal(got[:, :, :n], gold[:, :, :n], equal_nan=True)
    assert (got[:, :, n:] == 9.0).all()


@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("n,nrhs,batch", [(257, 1, 257), (257, 16, 256), (512, 256, 17), (513, 250, 17),
                                          (1024, 256, 17), (1025, 256, 17)])
def test_solve_many_units_past_256(handle, trans, n, nrhs, batch):
    """Orders past 256 with more than 256 units of 16 right-hand sides: four waves a unit to order 512, eight to 1024,
    sixteen beyond."""
    test_solve_bitwise(handle, trans, n, nrhs, batch, 0)


@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("n,nrhs,batch", [(257, 1, 300), (300, 4, 257), (300, 5, 257), (512, 2, 257), (513, 3, 257),
                                          (1000, 1, 257), (1024, 4, 257), (1025, 4, 257)])
def test_solve_many_units_of_few_right_hand_sides(handle, trans, n, nrhs, batch):
    """Up to four right-hand sides of many systems past order 256 run in units of four columns."""
    test_solve_bitwise(handle, trans, n, nrhs, batch, 0)


@pytest.mark.parametrize("n,batch,zero", [(257, 16, 200), (520, 8, None)])
def test_inverse_many_units_past_256(handle, n, batch, zero):
    test_inverse_bitwise(handle, n, batch, zero, True)
