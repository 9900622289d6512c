"""Products whose operands begin anywhere (the ring kernel's loads through registers, or straight into LDS where rows begin at whole
dwords): exact at every height of the tile, both layouts of B, lengths of K around whole stages, parts of K, batches; NaN next to
the operands and in the padding of their rows stays out of the result."""
import ctypes

import pytest
import torch

from helpers import E4, E5

pytestmark = pytest.mark.gpu


def operands(gen, batch, M, K, N, trans_b, lda, ldb, offset, dev):
    """A and B inside buffers full of NaN, rows lda and ldb bytes apart, the first one `offset` bytes from an aligned address."""
    a = torch.randint(-3, 4, (batch, M, K), generator=gen).float()
    b = torch.randint(-3, 4, (batch, K, N), generator=gen).float()
    a[..., -1], b[:, -1] = 3.0, 2.0      # the last k carries weight
    rows, cols = (N, K) if trans_b else (K, N)
    out = []
    for v, r, c, ld, fmt in ((a, M, K, lda, E4), (b.transpose(1, 2) if trans_b else b, rows, cols, ldb, E5)):
        stride = r * ld
        raw = torch.full((offset + batch * stride + 64,), 0x7f, dtype=torch.uint8)
        view = raw[offset:offset + batch * stride].reshape(batch, r, ld)
        view[..., :c] = v.to(fmt).view(torch.uint8)
        out.append((raw.to(dev), stride))
    return a, b, out


def call(pkg, dev, batch, M, K, N, trans_b, lda, ldb, offset, out_dtype=torch.float32):
    lib = pkg.capi()
    gen = torch.Generator().manual_seed(M + K + N + offset)
    a, b, ((araw, sa), (braw, sb)) = operands(gen, batch, M, K, N, trans_b, lda, ldb, offset, dev)
    size = ctypes.c_size_t()
    assert lib.mi355q_fp8_gemm_unaligned_workspace_bytes(0, lda, int(trans_b), ldb, M, N, K, batch, ctypes.byref(size)) == 0
    need = size.value
    ws = torch.zeros(max(need, 16), dtype=torch.uint8, device=dev)
    c = torch.full((batch, M, N), -7.0, dtype=out_dtype, device=dev)
    st = lib.mi355q_fp8_gemm_unaligned_ws(
        araw.data_ptr() + offset, pkg.E4M3FN, 0, lda, braw.data_ptr() + offset, pkg.E5M2, int(trans_b), ldb, c.data_ptr(),
        pkg.F32 if out_dtype == torch.float32 else pkg.BF16, N, M, N, K, None, 1.0, pkg.GS_NONE, None, 1.0, pkg.GS_NONE, None, 0, 0, None, 0, batch,
        sa, sb, M * N, 0, 0, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    assert st == 0
    ref = a @ b
    assert ref.abs().max() < 2 ** 24
    assert torch.equal(c.cpu().float(), ref.to(out_dtype).float()), (M, K, N, trans_b, offset)
    assert need == 0 or not ws[:65536].any()


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("offset", [0, 4, 3])
@pytest.mark.parametrize("M,K,N", [
    (1, 257, 33), (16, 384, 16), (17, 511, 129), (33, 512, 140), (64, 300, 1000), (100, 1025, 260), (129, 640, 131), (190, 383, 700),
    (256, 2300, 1000), (40, 4100, 200), (3, 3001, 500),
])
def test_exact(pkg, dev, M, K, N, trans_b, offset):
    gap = 4 if offset != 3 else 1
    lda, ldb = (K + 3) // 4 * 4 + gap, ((K if trans_b else N) + 3) // 4 * 4 + gap
    if offset == 0:
        lda, ldb = K, K if trans_b else N     # dense rows, the end of the operand in the middle of a chunk
    call(pkg, dev, 1, M, K, N, trans_b, lda, ldb, offset)


@pytest.mark.parametrize("trans_b", [False, True])
def test_batches_and_bf16(pkg, dev, trans_b):
    call(pkg, dev, 3, 37, 413, 145, trans_b, 415, (413 if trans_b else 145) + 2, 1, torch.bfloat16)
    call(pkg, dev, 2, 200, 516, 260, trans_b, 520, (516 if trans_b else 260) + 4, 8)


@pytest.mark.parametrize("batch,room", [(65536, True), (65600, True), (65600, False), (1, False)])
def test_a_product_that_the_query_accepts_is_served(pkg, dev, batch, room):
    """More matrices than a launch takes, whose last piece alone would not be worth it, and calls without a workspace."""
    lib = pkg.capi()
    gen = torch.Generator().manual_seed(batch)
    M, N, K = 1, 64, 2801
    a, b, ((araw, _), (braw, _)) = operands(gen, 1, M, K, N, True, K, K, 0, dev)
    size = ctypes.c_size_t()
    assert lib.mi355q_fp8_gemm_unaligned_workspace_bytes(0, K, 1, K, M, N, K, batch, ctypes.byref(size)) == 0
    ws = torch.zeros(max(size.value, 16), dtype=torch.uint8, device=dev)
    c = torch.full((batch, M, N), -7.0, device=dev)
    st = lib.mi355q_fp8_gemm_unaligned_ws(
        araw.data_ptr(), pkg.E4M3FN, 0, K, braw.data_ptr(), pkg.E5M2, 1, K, c.data_ptr(), pkg.F32, N, M, N, K, None, 1.0, pkg.GS_NONE, None, 1.0, pkg.GS_NONE,
        None, 0, 0, None, 0, batch, 0, 0, M * N, 0, 0, ws.data_ptr() if room else None, size.value if room else 0, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert st == 0
    assert torch.equal(c, (a @ b).to(dev).expand(batch, M, N))


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("offset", [1, 8, 15])
@pytest.mark.parametrize("M,K,N", [(1, 1024, 64), (33, 512, 160), (200, 400, 272), (256, 2304, 512)])
def test_whole_pitches_off_the_grid(pkg, dev, M, K, N, trans_b, offset):
    """Extents of whole chunks, and only the addresses are not."""
    call(pkg, dev, 1, M, K, N, trans_b, K, K if trans_b else N, offset)
    call(pkg, dev, 3, M, K, N, trans_b, K + 16, (K if trans_b else N) + 32, offset)


@pytest.mark.parametrize("M,K,N,off_a,off_b,copied", [
    (16, 8191, 4096, 0, 0, 0), (300, 2049, 1008, 0, 0, 0),                              # only K is ragged: B is filled up along it too
    (1000, 3001, 5008, 0, 0, 2), (1000, 3008, 5008, 4, 4, 0), (1000, 3008, 5001, 0, 0, 0),
    (1000, 3008, 5008, 1, 0, 1), (300, 2048, 1024, 1, 0, 0), (1000, 3008, 5008, 0, 1, 0), (1000, 3000, 5000, 1, 0, 2),
])
def test_what_is_copied_looks_at_addresses_and_at_what_a_copy_holds(dev, M, K, N, off_a, off_b, copied):
    a8 = torch.zeros(M * K + 64, dtype=torch.uint8, device=dev)[off_a:off_a + M * K].view(M, K).view(E4)
    b8 = torch.zeros(K * N + 64, dtype=torch.uint8, device=dev)[off_b:off_b + K * N].view(K, N).view(E4)
    run = lambda: torch.ops.hpu.fp8_gemm_v2(a8, False, b8, False, None, torch.bfloat16, None, None, None, False)  # noqa: E731
    run()
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    c = run()
    assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == 1 + copied
    assert not c.any()


def test_what_is_copied_and_what_is_not(pkg, dev):
    """Both sides of the rule, by the buffers that a call allocates: the result alone, or two copies as well."""
    for M, K, N, copied in [(1, 3001, 8000, 0), (300, 2049, 1003, 0), (64, 4100, 9999, 0), (1000, 3000, 5000, 0), (1000, 3001, 5001, 2), (2600, 2999, 6001, 2), (300, 255, 1003, 2)]:
        a8, b8 = torch.zeros(M, K, device=dev).to(E4), torch.zeros(K, N, device=dev).to(E4)
        run = lambda: torch.ops.hpu.fp8_gemm_v2(a8, False, b8, False, None, torch.bfloat16, None, None, None, False)  # noqa: E731
        run()
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        c = run()
        assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == 1 + copied, (M, K, N)
        assert not c.any()
