"""Grouped GEMM calls of many problems: the search for a tile's problem.

Operands are small integers, so that every product, sum and result is exact: equality with FP64 on the host.
"""
import pytest
import torch

import aclblas as B

pytestmark = pytest.mark.gpu

SMALL = [(130, 70, 8), (5, 3, 8), (64, 64, 4), (1, 1, 1), (16, 130, 3)]
LARGE = [(512, 256, 24), (256, 256, 8), (5, 3, 8)]


def _problems(count, dtype, shapes):
    """count problems of the shapes in turn: operands by shape, and the device address of each problem's A, B and C."""
    g = torch.Generator(device="cuda")
    g.manual_seed(count)
    ops, ptrs = [], [[0] * count for _ in range(3)]
    for s, (m, n, k) in enumerate(shapes):
        own = len(range(s, count, len(shapes)))
        x = [torch.randint(-3, 4, d, generator=g, device="cuda").to(dtype) for d in ((own, k, m), (own, n, k))]
        x.append(torch.zeros(own, n, m, dtype=dtype, device="cuda"))
        for p, t in zip(ptrs, x):
            p[s::len(shapes)] = [t.data_ptr() + i * t.stride(0) * t.element_size() for i in range(own)]
        ops.append(x)
    dims = [[shapes[i % len(shapes)][j] for i in range(count)] for j in range(3)]
    return ops, ptrs, dims


def _run(handle, count, dtype, shapes):
    ops, ptrs, (m, n, k) = _problems(count, dtype, shapes)
    op, one, zero, size = [B.OP_N] * count, [1.0] * count, [0.0] * count, [1] * count
    if dtype is torch.float32:
        st = B.sgemm_grouped_batched(handle.value, op, op, m, n, k, one, ptrs[0], m, ptrs[1], k, zero, ptrs[2], m, size)
    else:
        pa, pb, pc = (torch.tensor(p, dtype=torch.int64, device="cuda") for p in ptrs)
        st = B.gemm_grouped_batched_ex(handle.value, op, op, m, n, k, one, pa.data_ptr(), B.ACL_BF16, m, pb.data_ptr(),
                                       B.ACL_BF16, k, zero, pc.data_ptr(), B.ACL_BF16, m, size,
                                       B.COMPUTE["COMPUTE_32F"])
    assert st == 0, st
    torch.cuda.synchronize()
    for a, b, c in ops:
        assert torch.equal(c.cpu().double(), torch.matmul(b.cpu().double(), a.cpu().double()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 4095, 4096, 4097, 9001])
def test_tile_lookup_over_many_problems(handle, count, dtype):
    """Numbers of problems around those where the search takes another step (64 and 4096 records)."""
    _run(handle, count, dtype, SMALL)


def test_tile_lookup_direct_to_lds(handle):
    """Enough 256 x 256 tiles for the direct-to-LDS launch, over 200 problems; every third problem beside it."""
    _run(handle, 300, torch.bfloat16, LARGE)
