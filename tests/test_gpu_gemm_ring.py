"""The ring kernel (gemm_ring.h) at the edges of its tiles: rows and columns beside the tile heights and strips, K of less than a
stage, of a ragged last stage and of more and fewer stages than the ring holds, each height whole and in parts, all layouts.
Operands are small integers and scales powers of two, so that every fp32 sum is exact in any order and the result must match
bit for bit."""
import ctypes

import pytest
import torch

from helpers import E4, E5

# M, K, N, trans_a, trans_b by the tile height that the plan gives them; whole, then in parts
CASES_OF = {
    "ring16": [(16, 144, 130, 0, 0), (1, 16, 256, 0, 1)],
    "split_ring16": [(16, 2064, 129, 0, 0), (3, 8176, 8210, 0, 1), (1, 8192, 8208, 0, 1)],
    "ring32": [(17, 128, 128, 0, 0), (33, 400, 1000, 0, 0), (65, 768, 9000, 0, 0), (49, 896, 384, 0, 1)],
    "split_ring32": [(64, 4112, 4100, 0, 0), (32, 2064, 130, 0, 1)],
    "ring64": [(257, 1040, 5000, 0, 0), (65, 144, 11570, 0, 0), (128, 1168, 13000, 0, 1)],
    "split_ring64": [(35, 2720, 6598, 0, 0), (64, 14336, 4096, 0, 0), (33, 3024, 5789, 0, 1)],
    "ring128": [(129, 512, 12000, 0, 0), (257, 272, 8200, 0, 1), (600, 1303, 3000, 1, 0), (1000, 4096, 4096, 1, 0), (144, 1040, 5000, 1, 1)],
    "split_ring128": [(100, 8192, 11264, 0, 0), (72, 4640, 8612, 0, 1), (65, 2576, 250, 1, 0), (16, 4096, 256, 1, 1)],
    "ring192": [(129, 1040, 20000, 0, 0), (385, 272, 9366, 0, 0), (513, 2576, 7168, 0, 1)],
    "split_ring192": [(300, 7168, 7168, 0, 0), (700, 8208, 4090, 0, 0), (520, 8208, 2190, 0, 1)],
    "ring256": [(249, 1040, 20000, 0, 0), (1000, 2576, 6400, 0, 1), (275, 260, 10996, 1, 0), (258, 272, 11841, 1, 1)],
    "split_ring256": [(249, 7168, 13000, 0, 0), (200, 6672, 8488, 0, 1), (130, 6538, 8787, 1, 0), (129, 6576, 8357, 1, 1)],
}
CASES = [c for cases in CASES_OF.values() for c in cases]


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,ta,tb", CASES)
def test_ring_tiles_are_exact(M, K, N, ta, tb, dev):
    g = torch.Generator().manual_seed(M * 5 + K * 3 + N)
    a, b = torch.randint(-2, 3, (M, K), generator=g).float(), torch.randint(-2, 3, (K, N), generator=g).float()
    fa, fb = ((E4, E4), (E4, E5), (E5, E4), (E5, E5))[(M + K + N) % 4]
    a8, b8 = (a.t().contiguous() if ta else a).to(fa).to(dev), (b.t().contiguous() if tb else b).to(fb).to(dev)
    gemm = torch.ops.hpu.fp8_gemm_v2
    p = (a.to(dev) @ b.to(dev)).cpu()  # (small integers: exact in fp32)
    sa, sb = (torch.arange(M) % 3 - 1.0).exp2(), (torch.arange(N) % 2 - 1.0).exp2()
    bias = (torch.arange(N) % 5 - 2).float()
    ref = (p * sa[:, None]) * sb[None] + bias
    for out in (torch.float32, torch.bfloat16):
        for _ in range(2):
            c = gemm(a8, bool(ta), b8, bool(tb), None, out, sa[:, None].to(dev), sb.to(dev), bias.to(out).to(dev), False, [1, N])
            assert torch.equal(c.cpu(), ref.to(out))
    d = torch.randint(-4, 5, (M, N), generator=g).bfloat16()
    half, two = torch.tensor(0.5).to(dev), torch.tensor(2.0).to(dev)
    assert torch.equal(gemm(a8, bool(ta), b8, bool(tb), d.to(dev), torch.bfloat16, half, two, None, True).cpu(), (p + d.float()).bfloat16())
    assert torch.equal(gemm(a8, bool(ta), b8, bool(tb), None, torch.bfloat16, half, two, bias.bfloat16().to(dev), False).cpu(), (p + bias).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(1, 256, 4), (16, 2048, 300), (31, 256, 132), (60, 14336, 516), (100, 512, 12004), (190, 1024, 12004), (1000, 512, 6404)])
@pytest.mark.parametrize("f32", [True, False])
def test_rows_in_pieces_of_four(pkg, dev, M, K, N, f32):
    """fp32 results, accumulate inputs and scales per column of A or row of B, C and D in rows of their own pitch, two products a
    launch; pitches that are and are not multiples of four: the same values, and nothing beside them."""
    lib, out = pkg.capi(), torch.float32 if f32 else torch.bfloat16
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator().manual_seed(M + K + N)
    a, b = torch.randint(-2, 3, (2, M, K), generator=g).float(), torch.randint(-2, 3, (2, N, K), generator=g).float()
    a8, b8 = a.to(E4).to(dev), b.to(E5).to(dev)
    p = (a.to(dev) @ b.to(dev).transpose(1, 2).contiguous()).cpu()  # (small integers: exact in fp32)
    rows, cols = (torch.arange(M) % 3 - 1.0).exp2(), (torch.arange(N) % 2 - 1.0).exp2()
    vec, d = (torch.arange(N) % 5 - 2).to(out).to(dev), torch.randint(-4, 5, (2, M, N), generator=g).to(out)
    rs, cs = rows.to(dev), cols.to(dev)
    need = lib.mi355q_fp8_gemm_workspace_bytes(0, K, 1, K, M, N, K, 2)
    ws = torch.zeros(max(need, 16), dtype=torch.uint8, device=dev)
    for pitch in (N + 4, N + 3):
        wide = torch.full((2, M, pitch), float("nan"), dtype=out)
        wide[..., :N] = d
        wide = wide.to(dev)
        for a_rows, with_d, bias in ((1, 1, 0), (0, 1, 1), (0, 0, 1), (1, 0, 0)):
            c = torch.full((2, M, pitch), 7.0, dtype=out, device=dev)
            sa, sb = ((rs, pkg.GS_PER_ROW), (cs, pkg.GS_PER_COL)) if a_rows else ((cs, pkg.GS_PER_COL), (rs, pkg.GS_PER_ROW))
            assert lib.mi355q_fp8_gemm_ws(a8.data_ptr(), pkg.E4M3FN, 0, K, b8.data_ptr(), pkg.E5M2, 1, K, c.data_ptr(), pkg.F32 if f32 else pkg.BF16, pitch, M, N, K,
                                          sa[0].data_ptr(), 1.0, sa[1], sb[0].data_ptr(), 1.0, sb[1], vec.data_ptr() if bias else None,
                                          pkg.BIAS_ROW_VECTOR if bias else pkg.BIAS_NONE, 0, wide.data_ptr() if with_d else None, pitch if with_d else 0, 2,
                                          M * K, N * K, M * pitch, M * pitch if with_d else 0, 0, ws.data_ptr(), need, st) == 0
            ref = p * rows[:, None] * cols + (vec.float().cpu() if bias else 0.0) + (d.float() if with_d else 0.0)
            assert torch.equal(c[..., :N].cpu(), ref.to(out)), (pitch, a_rows, with_d, bias)
            assert bool((c[..., N:] == 7.0).all())


def test_every_height_is_reached(pkg):
    """The cases above run on the tile heights they stand under: all six, whole and in parts, with both layouts of B."""
    name = pkg.capi().mi355q_fp8_gemm_ws_variant
    up = lambda x: (x + 15) // 16 * 16  # noqa: E731
    for want, cases in CASES_OF.items():
        for M, K, N, ta, tb in cases:
            # (A [K, M] with a ragged K is the one form whose K is not rounded up before the launch)
            got = name(ta, up(M if ta else K), tb, up(K if tb else N), M, N, K if ta and not tb else up(K), 1).decode()
            assert got.startswith(want + "x"), (want, M, K, N, ta, tb, got)
        assert {c[4] for c in cases} == {0, 1}, want
