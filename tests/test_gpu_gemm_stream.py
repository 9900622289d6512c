"""The kernel that streams B [K, N] into registers (gemm_stream.h): at most 16 rows against more than 96 MiB.  Operands are small
integers and scales powers of two, so that every fp32 sum is exact in any order and the result must match bit for bit."""
import ctypes

import pytest
import torch

from helpers import E4, E5

pytestmark = pytest.mark.gpu

# one row, an odd number and all of a tile; K off the kernel's steps of 32, N off its strips of 256 and off 16; a strip's last
# columns alone; long K in parts and K in one piece
CASES = [(1, 4112, 24570), (3, 4112, 24586), (16, 4112, 24570), (7, 24592, 4104), (16, 48, 2097169), (2, 16400, 6401)]


def streams(pkg, M, K, N, ldb=None):
    up = lambda x: (x + 15) // 16 * 16  # noqa: E731
    return b"registers" in pkg.capi().mi355q_fp8_gemm_ws_variant(0, up(K), 0, ldb or up(N), M, N, up(K), 1)


def operands(M, K, N, dev, low=-2):
    g = torch.Generator(device=dev).manual_seed(M * 7 + K * 3 + N)
    return tuple(torch.randint(low, 3, shape, generator=g, device=dev, dtype=torch.int8).float() for shape in ((M, K), (K, N)))


@pytest.mark.parametrize("fa", [E4, E5])
@pytest.mark.parametrize("fb", [E4, E5])
@pytest.mark.parametrize("M,K,N", CASES)
def test_streamed_products_are_exact(pkg, M, K, N, fa, fb, dev):
    assert streams(pkg, M, K, N)
    a, b = operands(M, K, N, dev)
    a8, b8, p = a.to(fa), b.to(fb), a @ b
    del b
    gemm = torch.ops.hpu.fp8_gemm_v2
    sa, sb = (torch.arange(M, device=dev) % 3 - 1.0).exp2(), (torch.arange(N, device=dev) % 2 - 1.0).exp2()
    bias = (torch.arange(N, device=dev) % 5 - 2).float()
    for out in (torch.float32, torch.bfloat16):
        for _ in range(2):  # the counters of the first call are back at zero
            c = gemm(a8, False, b8, False, None, out, sa[:, None], sb, bias.to(out), False, [1, N])
            assert torch.equal(c, (p * sa[:, None] * sb + bias).to(out))
        d = torch.randint(-4, 5, (M, N), device=dev).to(out)
        half, two = torch.tensor(0.5, device=dev), torch.tensor(2.0, device=dev)
        assert torch.equal(gemm(a8, False, b8, False, d, out, half, two, d, True), (p + 2 * d.float()).to(out))  # accumulate input and full bias
        assert torch.equal(gemm(a8, False, b8, False, None, out, half, two, bias.to(out), False), (p + bias).to(out))


@pytest.mark.parametrize("exponent", [70, -72])
@pytest.mark.parametrize("kind_a", ["scalar", "row", "col"])
@pytest.mark.parametrize("kind_b", ["scalar", "row", "col"])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_scales_are_applied_one_after_the_other(pkg, exponent, kind_a, kind_b, out, dev):
    """Results whose scales multiply to something outside fp32's range, while sums and results lie inside it, with both scales per
    row, both per column, and every other pair."""
    M, K, N = 3, 4096, 24592
    assert streams(pkg, M, K, N)
    unit = 2.0 ** -14 if exponent > 0 else 2.0 ** 9
    a, b = torch.full((M, K), unit, device=dev), torch.full((K, N), unit, device=dev)
    a[M - 1, 1:] = 0.0
    b[:, 5] = 0.0
    sums = torch.full((M, N), K * unit * unit, dtype=torch.float64, device=dev)
    sums[M - 1] = unit * unit
    sums[:, 5] = 0.0

    def scale(kind, mantissa):
        s = torch.tensor(mantissa * 2.0 ** exponent, device=dev)
        if kind == "row":
            return (s * (1.0 - 0.25 * (torch.arange(M, device=dev) % 2)))[:, None]
        return s if kind == "scalar" else (s * (1.0 - 0.25 * (torch.arange(N, device=dev) % 2)))[None]

    sa, sb = scale(kind_a, 1.0 + 2.0 ** -6), scale(kind_b, 1.0)
    c = torch.ops.hpu.fp8_gemm_v2(a.to(E5), False, b.to(E5), False, None, out, sa, sb, None, False, list(sb.shape) if kind_b != "scalar" else None)
    ref = (sums * sa.double() * sb.double()).float()
    assert bool(ref.isfinite().all()) and int((ref == 0).sum()) == M
    # results below 2^-126 are rounded to a whole number of 2^-149 (bf16: 2^-133); bf16 rounds once, half a unit of eight bits
    rtol, atol = (2.0 ** -22, 2.0 ** -149) if out == torch.float32 else (2.0 ** -8, 2.0 ** -133)
    assert torch.allclose(c.float(), ref, rtol=rtol, atol=atol)


@pytest.mark.parametrize("M", [1, 16])
def test_what_lies_beside_the_operands_stays_out(pkg, dev, M):
    """Operands in wider rows with NaN codes behind every row, a row of NaN behind the last, NaN where the sums will lie: exact
    results all the same.  Then an infinity and a NaN in the last k and the last column: they reach their own rows and columns."""
    lib, (K, N) = pkg.capi(), (4112, 24570)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    a, b = operands(M, K, N, dev)

    def beside(x):
        rows, cols = x.shape
        wide = torch.full((rows + 1, (cols + 15) // 16 * 16 + 32), float("nan"), device=dev)
        wide[:rows, :cols] = x
        return wide.to(E5)

    def product(a, b):
        aw, bw = beside(a), beside(b)
        lda, ldb = aw.shape[1], bw.shape[1]
        assert streams(pkg, M, K, N, ldb)
        need = lib.mi355q_fp8_gemm_workspace_bytes(0, lda, 0, ldb, M, N, K, 1)
        ws = torch.full((need,), 255, dtype=torch.uint8, device=dev)
        ws[: 64 * 1024] = 0
        c = torch.full((M + 1, N), 7.0, device=dev)
        assert lib.mi355q_fp8_gemm_ws(aw.data_ptr(), pkg.E5M2, 0, lda, bw.data_ptr(), pkg.E5M2, 0, ldb, c.data_ptr(), pkg.F32, N, M, N, K, None, 1.0,
                                      pkg.GS_NONE, None, 1.0, pkg.GS_NONE, None, pkg.BIAS_NONE, 0, None, 0, 1, 0, 0, 0, 0, 0, ws.data_ptr(), need, st) == 0
        assert bool((c[M] == 7.0).all()) and int(ws[: 64 * 1024].count_nonzero()) == 0
        return c[:M]

    assert torch.equal(product(a, b), a @ b)
    a[:, K - 1], b[K - 1, :] = 1.0, 1.0
    want = a @ b
    a[M - 1, K - 1] = float("inf")
    b[K - 1, N - 1] = float("nan")
    got = product(a, b)
    assert bool(got[:, N - 1].isnan().all()) and bool((got[M - 1, : N - 1] == float("inf")).all())
    assert torch.equal(got[: M - 1, : N - 1], want[: M - 1, : N - 1])


def test_streamed_products_in_flight_on_two_streams(pkg, dev):
    work = []
    for M, K, N in ((1, 4112, 24592), (16, 16400, 6416)):
        assert streams(pkg, M, K, N)
        a, b = operands(M, K, N, dev)
        work.append((a.to(E4), b.to(E4), a @ b))
    torch.cuda.synchronize()
    two, got = [torch.cuda.Stream(), torch.cuda.Stream()], []
    for i in range(40):
        with torch.cuda.stream(two[i % 2]):
            a, b, want = work[(i // 2 + i % 2) % 2]
            got.append((torch.ops.hpu.fp8_gemm_v2(a, False, b, False, None, torch.float32), want))
    torch.cuda.synchronize()
    assert all(torch.equal(c, want) for c, want in got)
