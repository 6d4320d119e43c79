"""GEMM operands at any alignment, and the direct-to-LDS kernel behind pointer arrays and groups.

The element order of every sum is fixed (same instruction sequence per 16 x 16 accumulator in every kernel), so results
are compared bit for bit: odd leading dimensions and bases one element off against the aligned copy of the same
matrices; batches and groups on the direct-to-LDS kernel against the register-staged kernels (launch choice forced on
the handle); ragged k (partial last stages), edge tiles, every transpose pair, pointers the DMA cannot read.
"""
import numpy as np
import pytest
import torch

import aclblas as B

pytestmark = pytest.mark.gpu

TYPES = {"fp32": (torch.float32, B.ACL_FLOAT), "bf16": (torch.bfloat16, B.ACL_BF16),
         "fp16": (torch.float16, B.ACL_FLOAT16), "e4m3": (torch.uint8, B.ACL_FLOAT8_E4M3FN)}


def _values(g, t, cols, rows, ld, off):
    """Column-major rows x cols matrix at leading dimension ld, `off` elements into its buffer; flat view."""
    dt = TYPES[t][0]
    buf = torch.zeros(off + cols * ld, dtype=dt, device="cuda")
    if t == "e4m3":
        v = torch.randint(0, 120, (cols, rows), generator=g, device="cuda", dtype=torch.uint8)
    else:
        v = torch.randn(cols, rows, generator=g, device="cuda").to(dt)
    view = buf[off:].view(cols, ld)
    view[:, :rows] = v
    return buf, view


def _gemm(handle, t, ct, ta, tb, m, n, k, A, lda, Bm, ldb, C, ldc):
    st = B.gemm_ex(handle.value, B.OPS[ta], B.OPS[tb], m, n, k, 1.0, A.data_ptr(), TYPES[t][1], lda, Bm.data_ptr(),
                   TYPES[t][1], ldb, 0.5, C.data_ptr(), TYPES[ct][1], ldc, B.COMPUTE["COMPUTE_32F"])
    assert st == 0


@pytest.mark.parametrize("t,ct", [("fp32", "fp32"), ("bf16", "fp32"), ("fp16", "fp16"), ("e4m3", "fp16")])
@pytest.mark.parametrize("trans", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("m,n,k", [(5, 3, 7), (200, 300, 129), (520, 300, 193)])
def test_unaligned_operands_bitwise(handle, t, ct, trans, m, n, k):
    ta, tb = trans
    ra, ca = (m, k) if ta == "N" else (k, m)
    rb, cb = (k, n) if tb == "N" else (n, k)
    out = []
    for pad, off in ((None, 0), (1, 1), (3, 5)):
        g = torch.Generator(device="cuda")
        g.manual_seed(m + n + k)
        ld = lambda r: (r + 15) // 16 * 16 if pad is None else r + pad
        _, A = _values(g, t, ca, ra, ld(ra), off)
        _, Bm = _values(g, t, cb, rb, ld(rb), off)
        _, C = _values(g, ct, n, m, ld(m), off)
        before = C.clone()
        _gemm(handle, t, ct, ta, tb, m, n, k, A, ld(ra), Bm, ld(rb), C, ld(m))
        torch.cuda.synchronize()
        assert torch.equal(C[:, m:], before[:, m:])
        out.append(C[:, :m].clone())
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


@pytest.mark.parametrize("trans", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("m,n,k,off", [(264, 272, 200, 0), (264, 272, 64, 3), (16, 8, 40, 0)])
def test_batched_direct_tiles(handle, trans, m, n, k, off):
    """256 tiles over a pointer array: the second problem's operands start `off` elements off 16 bytes."""
    ta, tb = trans
    ra, ca = (m, k) if ta == "N" else (k, m)
    rb, cb = (k, n) if tb == "N" else (n, k)
    g = torch.Generator(device="cuda")
    g.manual_seed(k)
    ops = [[_values(g, "bf16", c, r, r, off * (i == 1))[1] for c, r in ((ca, ra), (cb, rb))] for i in range(3)]
    C = [torch.zeros(n, m, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    ptr = lambda ts: torch.tensor([x.data_ptr() for x in ts], dtype=torch.int64, device="cuda")
    pa, pb, pc = ptr([o[0] for o in ops]), ptr([o[1] for o in ops]), ptr(C)
    got = []
    for tile in (256, 64):
        assert B.set_tuning_override(handle.value, B.TUNE_GEMM, tile, 8) == 0
        st = B.gemm_batched_ex(handle.value, B.OPS[ta], B.OPS[tb], m, n, k, 1.0, pa.data_ptr(), B.ACL_BF16, ra,
                               pb.data_ptr(), B.ACL_BF16, rb, 0.0, pc.data_ptr(), B.ACL_BF16, m, 3,
                               B.COMPUTE["COMPUTE_32F"])
        assert st == 0
        torch.cuda.synchronize()
        got.append([c.clone() for c in C])
    assert B.set_tuning_override(handle.value, B.TUNE_GEMM, -1, 0) == 0
    for x, y in zip(*got):
        assert torch.equal(x, y)


@pytest.mark.parametrize("t", ["bf16", "fp16"])
def test_grouped_direct_segments(handle, t):
    """Groups of every transpose pair that go to the direct-to-LDS kernel, beside ones that cannot (odd leading
    dimension) and one without products, against the persistent kernel."""
    rng = np.random.default_rng(4)
    groups = []
    for i in range(24):
        m, n, k = (int(x) * 8 for x in rng.integers(30, 120, 3))
        groups.append(("NT"[i % 2], "NT"[(i // 2) % 2], m, n, k + (5 if i % 5 == 0 else 0), 0))
    groups.append(("N", "N", 301, 77, 200, 1))
    groups.append(("N", "N", 64, 64, 0, 0))
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    ops, lds = [], []
    for ta, tb, m, n, k, odd in groups:
        ra, ca = (m, k) if ta == "N" else (k, m)
        rb, cb = (k, n) if tb == "N" else (n, k)
        pad = lambda r: r + odd if odd else max(8, (r + 7) // 8 * 8)
        ops.append((_values(g, t, max(1, ca), ra, pad(ra), 0)[1], _values(g, t, cb, max(1, rb), pad(rb), 0)[1],
                    torch.randn(n, m, generator=g, device="cuda").to(TYPES[t][0])))
        lds.append((pad(ra), pad(rb), m))
    start = [o[2].clone() for o in ops]
    ptr = lambda i: torch.tensor([o[i].data_ptr() for o in ops], dtype=torch.int64, device="cuda")
    pa, pb, pc = ptr(0), ptr(1), ptr(2)
    col = lambda i: [x[i] for x in groups]
    got = []
    for forced in (False, True):
        if forced:
            assert B.set_tuning_override(handle.value, B.TUNE_GROUPED, 64, 2) == 0
        for o, s in zip(ops, start):
            o[2].copy_(s)
        st = B.gemm_grouped_batched_ex(
            handle.value, [B.OPS[x] for x in col(0)], [B.OPS[x] for x in col(1)], col(2), col(3), col(4),
            [1.0] * len(groups), pa.data_ptr(), TYPES[t][1], [x[0] for x in lds], pb.data_ptr(), TYPES[t][1],
            [x[1] for x in lds], [0.5] * len(groups), pc.data_ptr(), TYPES[t][1], [x[2] for x in lds],
            [1] * len(groups), B.COMPUTE["COMPUTE_32F"])
        assert st == 0
        torch.cuda.synchronize()
        got.append([o[2].clone() for o in ops])
    assert B.set_tuning_override(handle.value, B.TUNE_GROUPED, -1, 0) == 0
    for x, y, s in zip(got[0], got[1], start):
        assert torch.equal(x, y)
        assert not torch.equal(x, s)
