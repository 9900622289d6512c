"""Operands and rows whose extents are no multiple of 16 bytes: the padding copy (mi355q_pad_rows) byte for byte, the
products that go through it, and quantize_rows on rows that are no whole number of vectors."""
import ctypes

import pytest
import torch

from helpers import E4, E5

pytestmark = pytest.mark.gpu


class Desc(ctypes.Structure):
    _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p)] + [(n, ctypes.c_int64) for n in
                                                                      ("batch", "rows", "cols", "src_ld", "src_stride", "dst_rows", "dst_ld")]


@pytest.mark.parametrize("batch,rows,cols,offset", [(1, 1, 1, 0), (1, 5, 15, 3), (1, 7, 16, 1), (3, 33, 17, 5), (1, 1000, 3000, 0), (2, 65, 4099, 7), (1, 2049, 31, 0)])
def test_pad_rows(pkg, dev, batch, rows, cols, offset):
    lib = pkg.capi()
    g = torch.Generator().manual_seed(rows + cols)
    raw = torch.randint(0, 256, (offset + batch * rows * cols,), generator=g, dtype=torch.uint8).to(dev)
    src = raw[offset:].reshape(batch, rows, cols)
    dr, dl = rows + 3, (cols + 15) // 16 * 16
    dst = torch.full((batch, dr, dl), 0xAA, dtype=torch.uint8, device=dev)
    second = torch.full((1, 4, 32), 0xAA, dtype=torch.uint8, device=dev)
    jobs = (Desc * 2)(Desc(src.data_ptr(), dst.data_ptr(), batch, rows, cols, cols, rows * cols, dr, dl),
                      Desc(raw.data_ptr(), second.data_ptr(), 1, 1, 1, 1, 0, 4, 32))
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mi355q_pad_rows(ctypes.byref(jobs), 2, st) == 0
    want = torch.zeros(batch, dr, dl, dtype=torch.uint8)
    want[:, :rows, :cols] = src.cpu()
    assert torch.equal(dst.cpu(), want)
    assert int(second.count_nonzero()) <= 1 and second[0, 0, 0] == raw[0]


# around the size from which operands are copied, one and both operands ragged, every layout, batches
@pytest.mark.parametrize("M,K,N", [(1, 95, 33), (1, 97, 33), (1, 127, 33), (1, 129, 33), (300, 63, 501), (3, 1111, 999), (17, 4096, 257), (130, 333, 144), (64, 100, 5)])
@pytest.mark.parametrize("trans_a,trans_b", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batch", [0, 3])
def test_ragged_products_are_exact(dev, M, K, N, trans_a, trans_b, batch):
    g = torch.Generator().manual_seed(M + K + N)
    bs = (batch,) if batch else ()
    a = torch.randint(-3, 4, bs + (M, K), generator=g).float()
    b = torch.randint(-3, 4, bs + (K, N), generator=g).float()
    a8 = (a.transpose(-1, -2).contiguous() if trans_a else a).to(E4).to(dev)
    b8 = (b.transpose(-1, -2).contiguous() if trans_b else b).to(E5).to(dev)
    c = torch.ops.hpu.fp8_gemm_v2(a8, trans_a, b8, trans_b, None, torch.float32, None, None, None, False)
    assert torch.equal(c.cpu(), a @ b)


# both sides of each line of the rule: the operands are copied where that is faster than the kernel for any shape
@pytest.mark.parametrize("M,K,N,trans_b,copied", [(1, 97, 33, False, 0), (1, 127, 33, True, 0), (1, 129, 33, False, 2), (1, 129, 33, True, 2),
                                                  (300, 81, 501, False, 0), (300, 81, 501, True, 2), (5000, 49, 31, True, 0), (30, 81, 33, True, 0),
                                                  (300, 126, 501, False, 0), (2000, 20, 2001, False, 2), (64, 128, 5, False, 1)])
def test_which_ragged_products_are_copied(dev, M, K, N, trans_b, copied):
    a8, b8 = torch.zeros(M, K, device=dev).to(E4), torch.zeros((N, K) if trans_b else (K, N), device=dev).to(E4)

    def call():
        return torch.ops.hpu.fp8_gemm_v2(a8, False, b8, trans_b, None, torch.float32, None, None, None, False)

    call()
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    c = call()
    assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == 1 + copied and c.shape == (M, N)


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (2, 9), (5, 1021), (600, 515), (1, 16383), (2, 8191)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_ragged_rows_quantised(oracle, dev, rows, cols, dtype):
    if dtype == torch.float32 and cols > 8192:
        cols //= 2
    g = torch.Generator().manual_seed(rows * cols)
    x = (torch.randn(rows, cols, generator=g) * 2).to(dtype)
    for fmt in (E4, E5):
        y, inv = torch.ops.mi355q.quantize_rows(x.to(dev), fmt)
        y_ref, inv_ref = oracle.quantize_rows(x, fmt)
        assert torch.equal(y.cpu().view(torch.uint8), y_ref.view(torch.uint8)) and torch.equal(inv.cpu(), inv_ref)
