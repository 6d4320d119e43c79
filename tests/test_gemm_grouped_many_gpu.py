"""Grouped GEMM calls of many problems (the search for a tile's problem) and of many tiles.

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


def test_more_tiles_than_a_direct_launch(handle):
    """One problem wide enough for 2^23 - 1 tiles of 256 columns beside one whose work lets the pair qualify for the
    direct-to-LDS launch, which cannot hold that many: they take the persistent kernel."""
    n = 8388607 * 256
    big = 16384
    a = torch.ones(8, 8, dtype=torch.bfloat16, device="cuda")
    b = torch.ones(n, 8, dtype=torch.bfloat16, device="cuda")
    c = torch.zeros(n, 8, dtype=torch.bfloat16, device="cuda")
    a2 = torch.zeros(2 * big, big, dtype=torch.bfloat16, device="cuda")
    a2[0] = 1.0
    b2 = torch.zeros(big, 2 * big, dtype=torch.bfloat16, device="cuda")
    b2[:, 0] = torch.arange(big, device="cuda") % 256
    c2 = torch.zeros(big, big, dtype=torch.bfloat16, device="cuda")
    pa, pb, pc = (torch.tensor([x.data_ptr(), y.data_ptr()], dtype=torch.int64, device="cuda")
                  for x, y in ((a, a2), (b, b2), (c, c2)))
    st = B.gemm_grouped_batched_ex(handle.value, [B.OP_N] * 2, [B.OP_N] * 2, [8, big], [n, big], [8, 2 * big],
                                   [1.0] * 2, pa.data_ptr(), B.ACL_BF16, [8, big], pb.data_ptr(), B.ACL_BF16,
                                   [8, 2 * big], [0.0] * 2, pc.data_ptr(), B.ACL_BF16, [8, big], [1] * 2,
                                   B.COMPUTE["COMPUTE_32F"])
    assert st == 0, st
    torch.cuda.synchronize()
    for at in range(0, n, 1 << 28):
        assert bool((c[at:at + (1 << 28)] == 8.0).all()), at
    want = (torch.arange(big, device="cuda") % 256).to(torch.bfloat16)
    assert torch.equal(c2, want[:, None].expand(big, big))
    del a, b, c, a2, b2, c2
    torch.cuda.empty_cache()
