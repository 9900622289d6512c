"""Products of more than 128 rows with K in parts over workgroups (gemm_ring.h), and the choice of tiles for them.
Operands are small integers and scales powers of two, so that every fp32 sum is exact in any order and the result must
match bit for bit."""
import pytest
import torch

from helpers import E4, E5

# rows and columns at the edges of the 128- and 256-row tiles; K of one pair of stages and a remainder, of an odd number of
# pairs, and long enough for two to eight parts, three and five among them; narrow N
CASES = [(129, 4112, 136), (256, 14336, 1024), (257, 2576, 520), (384, 16384, 264), (300, 7168, 7168), (513, 8192, 4104),
         (1024, 14336, 1032), (700, 8192, 4096), (4000, 6160, 24), (130, 528, 8), (1500, 16384, 1024), (200, 1296, 3000)]


@pytest.mark.gpu
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,K,N", CASES)
def test_split_tiles_are_exact(M, K, N, trans_b, dev):
    fa, fb = ((E4, E4), (E4, E5), (E5, E4), (E5, E5))[(M + K // 16 + N) % 4]
    g = torch.Generator().manual_seed(M * 7 + K * 3 + N)
    a, b = torch.randint(-2, 3, (M, K), generator=g).float(), torch.randint(-2, 3, (K, N), generator=g).float()
    a8, b8 = a.to(fa).to(dev), (b.t().contiguous() if trans_b else b).to(fb).to(dev)
    ops = torch.ops.hpu
    sa, sb = (torch.arange(M) % 3 - 1.0).exp2(), (torch.arange(N) % 2 - 1.0).exp2()
    bias = (torch.arange(N) % 5 - 2).float()
    p = a @ b
    ref = (p * sa[:, None]) * sb[None] + bias
    for out_dtype in (torch.float32, torch.bfloat16):
        for _ in range(2):  # the counters of the first call are back at zero
            c = ops.fp8_gemm_v2(a8, False, b8, trans_b, None, out_dtype, sa[:, None].to(dev), sb.to(dev), bias.to(out_dtype).to(dev), False, [1, N])
            assert torch.equal(c.cpu(), ref.to(out_dtype)), (M, K, N, out_dtype)
    d = torch.randint(-4, 5, (M, N), generator=g).bfloat16()
    c = ops.fp8_gemm_v2(a8, False, b8, trans_b, d.to(dev), torch.bfloat16, torch.tensor(0.5).to(dev), torch.tensor(2.0).to(dev), d.to(dev), True)
    assert torch.equal(c.cpu(), (p + d.float() * 2).bfloat16())
    at8 = a.t().contiguous().to(fa).to(dev)  # K contiguous in neither operand
    if M % 16 == 0 and N % 16 == 0:
        c = ops.fp8_gemm_v2(at8, True, b8, trans_b, None, torch.float32, None, None, None, False)
        assert torch.equal(c.cpu(), p)


@pytest.mark.gpu
def test_batches_and_repeated_calls(dev):
    """Separate products in one launch, and results that are the same from run to run whoever arrives last."""
    g = torch.Generator().manual_seed(5)
    a, b = torch.randint(-2, 3, (3, 144, 4096), generator=g).float(), torch.randint(-2, 3, (3, 4096, 256), generator=g).float()
    c = torch.ops.hpu.fp8_gemm_v2(a.to(E4).to(dev), False, b.to(E4).to(dev), False, None, torch.float32, None, None, None, False)
    assert torch.equal(c.cpu(), a @ b)
    x, w = torch.randn(300, 8192, generator=g).to(E4).to(dev), torch.randn(8192, 1024, generator=g).to(E4).to(dev)
    first = torch.ops.hpu.fp8_gemm_v2(x, False, w, False, None, torch.float32, None, None, None, False)
    for _ in range(20):
        assert torch.equal(torch.ops.hpu.fp8_gemm_v2(x, False, w, False, None, torch.float32, None, None, None, False), first)


def test_plans_of_the_cases(pkg):
    """The shapes above do split (they need a workspace), products that fill the chip do not, and the sums' room is bounded."""
    need = pkg.capi().mi355q_fp8_gemm_workspace_bytes
    split = [c for c in CASES if need(0, c[1], 0, (c[2] + 15) // 16 * 16, *(c[0], c[2], c[1]), 1) > 0]
    assert len(split) >= 9, split
    assert need(0, 4096, 0, 14336, 8192, 14336, 4096, 1) == 0
    for m in (129, 200, 256, 300, 512, 1000, 2000):
        for n in (128, 1024, 4096, 8192):
            for k in (1024, 4096, 14336):
                assert need(0, k, 0, n, m, n, k, 1) <= 64 * 1024 + 256 * 256 * 128 * 4


def test_few_and_long_parts(pkg):
    """Short products on a chip that their parts fill are cut in two at most (in four they took up to 57 % longer than whole), and
    nothing into more than 16 parts."""
    need = pkg.capi().mi355q_fp8_gemm_workspace_bytes
    sums = lambda m, k, n: need(0, k, 0, n, m, n, k, 1)  # noqa: E731
    for m, k, n in [(130, 3072, 4096), (256, 3072, 4096), (384, 3072, 2048), (500, 3072, 2048), (768, 3072, 1024), (1000, 3072, 1024)]:
        tiles = (m + 127) // 128 * (n // 128)
        assert sums(m, k, n) <= 64 * 1024 + 2 * tiles * 128 * 128 * 4, (m, k, n)
    for k in (14336, 16384, 32768):
        assert 64 * 1024 < sums(130, k, 128) <= 64 * 1024 + 16 * 2 * 128 * 128 * 4, k


def test_products_that_fill_the_chip_keep_the_largest_tiles(pkg):
    """From one and a half 256 x 256 tiles per compute unit on the 256-row tiles of the ring took up to a fifth longer, and below that
    with rows off the 128-byte lines or few stages; the 192-row tile and the other products below it gained."""
    name = pkg.capi().mi355q_fp8_gemm_ws_variant
    tile = lambda m, k, n, nk=0: name(0, k, nk, k if nk else n, m, n, k, 1).decode().split("_")[0]  # noqa: E731
    for m, k, n in [(4096, 4096, 14336), (3636, 2816, 14752), (1792, 1536, 21248), (5888, 3072, 9728), (2409, 3824, 9600), (7836, 512, 3072),
                    (8192, 4096, 14336), (4096, 14336, 4096)]:
        assert tile(m, k, n) == tile(m, k, n, 1) == "tile256x256x128", (m, k, n)
    assert tile(7341, 896, 2176) == tile(3840, 3712, 6144, 1) == "ring256x128x128"
    assert tile(8005, 3968, 2304, 1) == tile(1766, 896, 9632) == "ring192x128x128"
