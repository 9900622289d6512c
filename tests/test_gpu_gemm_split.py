"""Products of few rows of A on the ring kernel (gemm_ring.h) and the split of K over workgroups; test_gpu_gemm_stream.py has
the kernel that streams B into registers.  Operands are small integers and scales powers of two, so that every
fp32 sum is exact in any order and the result must match bit for bit."""
import ctypes

import pytest
import torch

import isa_check
from helpers import E4, E5

# rows at the edges of the kernels' tiles; N off the strips' 128 and 256 columns; K from one unit of 16 up, off the
# stages' 128, and long enough for many parts
CASES = [(1, 16, 8), (1, 4096, 1024), (15, 4112, 1000), (16, 14336, 520), (16, 8192, 4104), (17, 2064, 384), (32, 4096, 264),
         (33, 2048, 1016), (64, 14336, 256), (65, 1040, 2048), (128, 8192, 640), (3, 272, 33288)]


def operands(M, K, N, trans_b, fa, fb, dev):
    g = torch.Generator().manual_seed(M * 7 + K * 3 + N)
    a = torch.randint(-3, 4, (M, K), generator=g).float()
    b = torch.randint(-3, 4, (K, N), generator=g).float()
    return a, b, a.to(fa).to(dev), (b.t().contiguous() if trans_b else b).to(fb).to(dev)


@pytest.mark.gpu
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,K,N", CASES)
def test_split_products_are_exact(M, K, N, trans_b, dev):
    fa, fb = ((E4, E4), (E4, E5), (E5, E4), (E5, E5))[(M + K + N) % 4]
    a, b, a8, b8 = operands(M, K, N, trans_b, fa, fb, dev)
    ops = torch.ops.hpu
    sa, sb = (torch.arange(M) % 3 - 1.0).exp2(), (torch.arange(N) % 2 - 1.0).exp2()
    bias = (torch.arange(N) % 5 - 2).float()
    ref = ((a @ b) * sa[:, None]) * sb[None] + bias
    for out_dtype in (torch.float32, torch.bfloat16):
        for _ in range(2):  # the counters of the first call are back at zero
            c = ops.fp8_gemm_v2(a8, False, b8, trans_b, None, out_dtype, sa[:, None].to(dev), sb.to(dev), bias.to(out_dtype).to(dev), False, [1, N])
            assert torch.equal(c.cpu(), ref.to(out_dtype)), (M, K, N, out_dtype)
    # accumulate input, full bias, scalar scales
    d = torch.randint(-4, 5, (M, N)).bfloat16()
    c = ops.fp8_gemm_v2(a8, False, b8, trans_b, d.to(dev), torch.bfloat16, torch.tensor(0.5).to(dev), torch.tensor(2.0).to(dev), d.to(dev), True)
    assert torch.equal(c.cpu(), (a @ b + d.float() * 2).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 8, 17])
@pytest.mark.parametrize("exponent", [70, -72])
@pytest.mark.parametrize("kind_a", ["scalar", "row", "col"])
@pytest.mark.parametrize("kind_b", ["scalar", "row", "col"])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_scales_are_applied_one_after_the_other(M, exponent, kind_a, kind_b, out, dev):
    """Results whose scales multiply to something outside fp32's range, while sums and results lie inside it: 2^140
    is infinite and 2^-144 has five bits left of a scale with seven."""
    K = N = 4096
    unit = 2.0 ** -14 if exponent > 0 else 2.0 ** 9
    a, b = torch.full((M, K), unit), torch.full((K, N), unit)
    a[M - 1, 1:] = 0.0
    b[:, 5] = 0.0
    sums = torch.full((M, N), K * unit * unit, dtype=torch.float64)
    sums[M - 1] = unit * unit
    sums[:, 5] = 0.0

    def scale(kind, mantissa):
        s = torch.tensor(mantissa * 2.0 ** exponent)
        if kind == "row":
            return (s * (1.0 - 0.25 * (torch.arange(M) % 2)))[:, None]
        return s if kind == "scalar" else (s * (1.0 - 0.25 * (torch.arange(N) % 2)))[None]

    sa, sb = scale(kind_a, 1.0 + 2.0 ** -6), scale(kind_b, 1.0)
    c = torch.ops.hpu.fp8_gemm_v2(a.to(E5).to(dev), False, b.to(E5).to(dev), False, None, out, sa.to(dev), sb.to(dev), None, False,
                                  list(sb.shape) if kind_b != "scalar" else None)
    ref = (sums * sa.double() * sb.double()).float()
    assert bool(ref.isfinite().all()) and int((ref == 0).sum()) == M
    # results below 2^-126 are rounded to a whole number of 2^-149 (bf16: 2^-133); of 1 + 2^-6 and its 0.75 and 0.5625, bf16's eight
    # bits hold the first two, and the third is half a unit off at most
    rtol, atol = (2.0 ** -22, 2.0 ** -149) if out == torch.float32 else (2.0 ** -8, 2.0 ** -133)
    assert torch.allclose(c.float().cpu(), ref, rtol=rtol, atol=atol)


@pytest.mark.gpu
def test_one_workspace_serves_several_shapes(pkg, dev):
    """The C entry with a caller's workspace: shapes one after the other, counters left zero, too small a workspace
    refused, and no workspace accepted."""
    lib = pkg.capi()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    shapes = [(1, 4096, 1024), (16, 8192, 4096), (64, 4096, 512), (2, 2048, 2048)]
    need = max(lib.mi355q_fp8_gemm_workspace_bytes(0, k, 0, n, m, n, k, 1) for m, k, n in shapes)
    assert need > 64 * 1024
    ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    for m, k, n in shapes:
        a, b, a8, b8 = operands(m, k, n, False, E4, E4, dev)
        ref = a @ b
        c = torch.empty(m, n, device=dev)
        for ptr, size, want in ((ws.data_ptr(), need, 0), (None, 0, 0), (ws.data_ptr(), 1024, None)):
            status = lib.mi355q_fp8_gemm_ws(a8.data_ptr(), pkg.E4M3FN, 0, k, b8.data_ptr(), pkg.E4M3FN, 0, n, c.data_ptr(), pkg.F32, n, m, n, k,
                                            None, 1.0, pkg.GS_NONE, None, 1.0, pkg.GS_NONE, None, pkg.BIAS_NONE, 0, None, 0, 1, 0, 0, 0, 0, 0,
                                            ptr, size, st)
            if want is None:
                assert status != 0
                continue
            assert status == 0
            assert torch.equal(c.cpu(), ref)
        assert int(ws[: 64 * 1024].count_nonzero()) == 0


# per kernel that splits K: rows, K off the stages' 128, N off 16
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,name", [(1, 4112, 1000, b"split_ring16"), (16, 4112, 16378, b"split_ring16"), (40, 4112, 1000, b"split_ring32"),
                                        (128, 14352, 250, b"split_ring32"), (300, 8208, 1000, b"split_ring64"), (100, 8208, 11250, b"split_ring128"),
                                        (700, 8208, 4090, b"split_ring192"), (2000, 14352, 1000, b"split_ring256")])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_what_lies_beside_the_operands_stays_out(pkg, dev, M, K, N, name, ta, tb):
    """Operands in wider rows with NaN codes behind every row, and a row of NaN behind the last: exact results all the same.
    Then an infinity and a NaN in the last k and the last column: they reach their own rows and columns and no others."""
    lib = pkg.capi()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator().manual_seed(M + N)
    a, b = torch.randint(-2, 3, (M, K), generator=g).float(), torch.randint(-2, 3, (K, N), generator=g).float()

    def beside(x):  # (rows rounded up to 16 for a transposed one, which is read in chunks of 16 along m or n)
        rows, cols = x.shape
        wide = torch.full((rows + 1, (cols + 15) // 16 * 16 + 32), float("nan"))
        wide[:rows, :cols] = x
        return wide

    def product(a, b):
        aw, bw = beside(a.t() if ta else a).to(E5).to(dev), beside(b.t() if tb else b).to(E5).to(dev)
        lda, ldb = aw.shape[1], bw.shape[1]
        variant = lib.mi355q_fp8_gemm_ws_variant(ta, lda, tb, ldb, M, N, K, 1)
        # (an A [K, M] has tiles of 128 and 256 rows alone, cut or not)
        assert variant.startswith(name + b"x") or (ta and variant.replace(b"split_", b"").startswith((b"ring128x", b"ring256x"))), variant
        need = lib.mi355q_fp8_gemm_workspace_bytes(ta, lda, tb, ldb, M, N, K, 1)
        ws = torch.full((need,), 255, dtype=torch.uint8, device=dev)  # NaN where the sums will lie
        ws[: 64 * 1024] = 0
        c = torch.full((M + 1, N), 7.0, device=dev)
        assert lib.mi355q_fp8_gemm_ws(aw.data_ptr(), pkg.E5M2, ta, lda, bw.data_ptr(), pkg.E5M2, tb, ldb, c.data_ptr(), pkg.F32, N, M, N, K, None, 1.0,
                                      pkg.GS_NONE, None, 1.0, pkg.GS_NONE, None, pkg.BIAS_NONE, 0, None, 0, 1, 0, 0, 0, 0, 0, ws.data_ptr(), need, st) == 0
        assert bool((c[M] == 7.0).all())
        return c[:M].cpu()

    assert torch.equal(product(a, b), a @ b)
    a[:, K - 1], b[K - 1, :] = 1.0, 1.0
    want = a @ b
    a[M - 1, K - 1] = float("inf")
    b[K - 1, N - 1] = float("nan")
    got = product(a, b)
    assert bool(got[:, N - 1].isnan().all()) and bool((got[M - 1, : N - 1] == float("inf")).all())
    assert torch.equal(got[: M - 1, : N - 1], want[: M - 1, : N - 1])


def test_short_products_stay_whole(pkg):
    """K below which a product was slower in parts than whole, and longer ones that stay in parts; without a workspace none is."""
    need = pkg.capi().mi355q_fp8_gemm_workspace_bytes
    bytes_of = lambda m, k, n, nk: need(0, k, nk, k if nk else n, m, n, k, 1)  # noqa: E731
    for m in (1, 4, 8, 16, 17, 64, 128):
        for n in (128, 512, 2048, 4096, 11264):
            for nk in (0, 1):
                assert all(bytes_of(m, k, n, nk) == 0 for k in (16, 512, 1024, 1280, 1536, 1776)), (m, n, nk)
                assert bytes_of(m, 8192, n, nk) > 0, (m, n, nk)
    counters = 64 * 1024
    for n in (512, 1024, 4096):  # sums of 16 rows and 128 columns a strip
        parts = (bytes_of(1, 4096, n, 0) - counters) // (n * 16 * 4)
        assert 2 <= parts <= 8, (n, parts)


def test_large_batches_are_streamed(pkg):
    """Few rows against many matrices [K, N]: on the 16-row tiles of the ring 25 of 1 x 4096 x 4096 took a third longer."""
    name = pkg.capi().mi355q_fp8_gemm_ws_variant
    kernel = lambda m, k, n, batch: name(0, k, 0, n, m, n, k, batch)  # noqa: E731
    for m, k, n, batch in [(1, 4096, 4096, 16), (16, 4096, 2048, 64), (4, 2048, 2048, 100)]:
        assert b"registers" in kernel(m, k, n, batch), (m, k, n, batch)
    for m, k, n, batch in [(1, 4096, 4096, 15), (1, 512, 512, 1600), (16, 1024, 1024, 400), (17, 4096, 4096, 25)]:
        assert b"ring" in kernel(m, k, n, batch), (m, k, n, batch)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16])
def test_large_batches_are_exact(M, dev):
    g = torch.Generator(device=dev).manual_seed(M)
    a = torch.randint(-2, 3, (17, M, 4096), generator=g, device=dev).float()
    b = torch.randint(-2, 3, (17, 4096, 4080), generator=g, device=dev).float()
    want = a @ b
    for out in (torch.float32, torch.bfloat16):
        assert torch.equal(torch.ops.hpu.fp8_gemm_v2(a.to(E4), False, b.to(E5), False, None, out), want.to(out))


def test_few_rows_of_an_mn_major_a_stay_whole_longer(pkg):
    """A [K, M] runs on tiles of 128 rows, whose parts send all their sums: 16 x 1792 x 128 takes 12.0 us whole and 16.4 in parts."""
    need = pkg.capi().mi355q_fp8_gemm_workspace_bytes
    for k in (1792, 2048):
        for n in (128, 1024, 4096, 14336):
            for nk in (0, 1):
                assert need(1, 16, nk, k if nk else n, 16, n, k, 1) == 0, (k, n, nk)
    assert need(1, 16, 0, 1024, 16, 1024, 8192, 1) > 0


@pytest.mark.timeout(600)
def test_parts_of_k_meet_by_device_scope_accesses_in_order():
    """Sums stored (sc1), acknowledged, barrier, ticket, barrier, counter reset, sums read (sc1); nothing cache-wide."""
    import re
    from concurrent.futures import ThreadPoolExecutor
    # the ring kernel has six heights with an A [M, K] and two with an A [K, M], each for four pairs of formats and B with the nontemporal hint or not
    sources = (("gemm_stream.hip", 4), ("gemm_inst_kk.hip", 48), ("gemm_inst_km.hip", 48), ("gemm_inst_mk.hip", 16), ("gemm_inst_mm.hip", 16))
    with ThreadPoolExecutor(max_workers=4) as ex:
        texts = list(ex.map(isa_check.compile_to_isa, [src for src, _ in sources]))
    for (src, least), text in zip(sources, texts):
        orders = isa_check.exchange_order(text)
        assert len(orders) >= least and isa_check.scratch_bytes(text) == {}, src
        for name, seq in orders.items():
            assert "F" not in seq and seq.count("A") == 1, name
            assert re.search(r"S+W+BAW?BS?W?L+", seq), (name, seq)


@pytest.mark.gpu
def test_split_products_in_flight_on_two_streams(dev):
    """Each stream has a workspace of its own: products of three kernels, interleaved without a wait."""
    g = torch.Generator().manual_seed(8)
    work = []
    for m, k, n in ((1, 4096, 1024), (64, 14336, 256), (300, 8192, 1024)):
        a, w = torch.randn(m, k, generator=g).to(E4).to(dev), torch.randn(k, n, generator=g).to(E4).to(dev)
        work.append((a, w, torch.ops.hpu.fp8_gemm_v2(a, False, w, False, None, torch.float32)))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for i in range(60):
        with torch.cuda.stream(streams[i % 2]):
            a, w, want = work[(i // 2 + i % 2) % 3]
            got.append((torch.ops.hpu.fp8_gemm_v2(a, False, w, False, None, torch.float32), want))
    torch.cuda.synchronize()
    assert all(torch.equal(c, want) for c, want in got)


@pytest.mark.gpu
def test_workspaces_that_are_given_back(dev):
    """More (stream, operator) pairs than buffers are kept: the least recently used one goes, and calls on its stream start
    from a fresh one.  torch has 32 streams to hand out, so three operators with a workspace take part."""
    g = torch.Generator().manual_seed(9)
    a, w = torch.randn(1, 4096, generator=g).to(E4).to(dev), torch.randn(4096, 1024, generator=g).to(E4).to(dev)
    x = torch.randn(8, 4096, generator=g).to(dev)
    packed = torch.randint(-2 ** 31, 2 ** 31 - 1, (4096, 64), generator=g, dtype=torch.int64).to(torch.int32).to(dev)
    scale = (torch.rand(32, 512, generator=g) * 0.01).bfloat16().to(dev)

    def run():
        return (torch.ops.hpu.fp8_gemm_v2(a, False, w, False, None, torch.float32),
                torch.ops.mi355q.w4a8_gemm(x.to(E4), packed, scale, None, False, torch.bfloat16, None, None),
                torch.ops.mi355q.w4a16_gemm(x.bfloat16(), packed, scale, None, False, torch.bfloat16, None))

    want = run()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(32)]
    assert len({s.cuda_stream for s in streams}) * 3 > 64
    got = []
    for _ in range(3):
        for s in streams:
            with torch.cuda.stream(s):
                got.append(run())
    torch.cuda.synchronize()
    assert all(torch.equal(c, r) for outs in got for c, r in zip(outs, want))
