"""The 4-bit products of at most 16 rows (w4_stream.hip): bit-exact where the arithmetic is exact, at the edges of strips, stages and
parts; sums that depend on the order the same whichever part adds them up; and the generated code's order of the exchange."""
import ctypes
import re

import pytest
import torch

import isa_check
from helpers import gemm_errors
from test_gpu_w4a8_gemm import weights

E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["bf16", "e4m3fn", "e5m2"])
@pytest.mark.parametrize("M,K,N,signed,zp", [
    (1, 128, 32, False, True),        # one stage, one slot of a strip
    (16, 256, 512, True, False),      # two stages, a whole strip
    (15, 384, 544, False, False),     # three; a second strip of one slot
    (7, 1024, 1056, True, True),      # four parts of two stages
    (16, 4224, 992, False, True),     # uneven parts, a last strip that ends inside its last wave
    (2, 4096, 480, False, True),      # sixteen parts of two stages
    (9, 640, 66048, False, True),     # 129 strips: whole
    (16, 2176, 13312, True, True),    # 26 strips
])
def test_exact(oracle, dev, M, K, N, signed, zp, act):
    gen = torch.Generator().manual_seed(M + K + N + signed)
    q, z, s, pk, pz = weights(oracle, gen, K, N, 128, signed, zp, pow2=True)
    top = {"bf16": 255, "e4m3fn": 15, "e5m2": 7}[act]      # integers that the format holds
    a = torch.randint(-top, top + 1, (M, K), generator=gen).float()
    bias = torch.randint(-8, 9, (N,), generator=gen).float()
    w = (q - (z.repeat_interleave(128, 0) if zp else 0)).double() * s.double().repeat_interleave(128, 0)
    pkd, sd, pzd = pk.to(dev), s.to(dev), pz.to(dev) if zp else None
    if act == "bf16":
        expect = a.double() @ w + bias.double()
        run = lambda dt, b: torch.ops.mi355q.w4a16_gemm(a.bfloat16().to(dev), pkd, sd, pzd, signed, dt, b.to(dev))  # noqa: E731
    else:
        x = a.to(E4 if act == "e4m3fn" else E5)
        assert torch.equal(x.float(), a)
        sa = torch.exp2(torch.randint(-2, 3, (M, 1), generator=gen).float())
        expect = a.double() @ w * sa.double() + bias.double()
        run = lambda dt, b: torch.ops.mi355q.w4a8_gemm(x.to(dev), pkd, sd, pzd, signed, dt, sa.to(dev), b.to(dev))  # noqa: E731
    assert expect.abs().max() < 2 ** 24
    for _ in range(2):
        assert torch.equal(run(torch.float32, bias).cpu().double(), expect)
    assert torch.equal(run(torch.bfloat16, bias.bfloat16()).cpu(), expect.float().bfloat16())


@pytest.mark.gpu
def test_extreme_activations_in_bf16(oracle, dev):
    """Rows of the largest and of very small bf16 values next to ordinary ones; a row with an infinity and one with a NaN keep them to themselves."""
    gen = torch.Generator().manual_seed(5)
    M, K, N = 6, 512, 544
    q, z, s, pk, pz = weights(oracle, gen, K, N, 128, False, True)
    x = torch.randn(M, K, generator=gen)
    x[1] = torch.where(x[1] > 0, 1.0, -1.0) * 3.0e38
    x[2] *= 1e-30
    x[3, 5], x[4, 300] = float("inf"), float("nan")
    x = x.bfloat16()
    s = (s.float() * 2.0 ** -10).bfloat16()
    out = torch.ops.mi355q.w4a16_gemm(x.to(dev), pk.to(dev), s.to(dev), pz.to(dev), False, torch.float32, None).cpu()
    w = (q - z.repeat_interleave(128, 0)).double() * s.double().repeat_interleave(128, 0)
    ref = x.double() @ w
    for m in (0, 1, 2, 5):
        # fp32 sums of K products: at most K roundings of 2^-24 of the sum of magnitudes, of q a and z a apart
        bound = (x[m].double().abs() @ (15 * s.double().repeat_interleave(128, 0))) * (2 * K * 2.0 ** -24)
        assert ((out[m].double() - ref[m]).abs() <= bound).all(), m
    assert torch.isnan(out[4]).all() and not torch.isfinite(out[3]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("K", [512, 4096])      # in one part, in several
@pytest.mark.parametrize("scale", [-27, 0])
def test_rows_of_small_activations(oracle, dev, K, scale):
    """Results down to fp32's smallest values keep the bits that fp32 has for them, beside rows near the largest bf16 values."""
    gen = torch.Generator().manual_seed(K + scale)
    M, N = 16, 1056
    q, z, s, pk, pz = weights(oracle, gen, K, N, 128, False, True)
    s = (s.float() * 2.0 ** scale).bfloat16()
    x = (torch.randn(M, K, generator=gen).double() * torch.exp2(torch.tensor([*range(-90, -132, -3), 118, 120]).double())[:, None]).bfloat16()
    out = torch.ops.mi355q.w4a16_gemm(x.to(dev), pk.to(dev), s.to(dev), pz.to(dev), False, torch.float32, None).cpu()
    ref = x.double() @ ((q - z.repeat_interleave(128, 0)).double() * s.double().repeat_interleave(128, 0))
    # 2^-24 of the sum of magnitudes for each of K products, of q a and z a apart, and half of fp32's smallest value wherever a group or a
    # part is added (sixteen parts at most)
    bound = (x.double().abs() @ (15 * s.double().repeat_interleave(128, 0))) * (2 * K * 2.0 ** -24) + (K // 128 + 16) * 2.0 ** -150
    assert ((out.double() - ref).abs() <= bound).all(), ((out.double() - ref).abs() / bound).amax(1)


@pytest.mark.gpu
def test_sums_past_the_range(oracle, dev):
    """Groups whose sums are past fp32's largest value: an infinity of the result's sign, and a finite result stays finite."""
    gen = torch.Generator().manual_seed(6)
    M, K, N = 8, 512, 544
    q, z, s, pk, pz = weights(oracle, gen, K, N, 128, False, True)
    x = torch.randn(M, K, generator=gen)
    x[:, 256:] = -x[:, :256]             # with the weights below: the last two groups take the first two back, but for one activation
    q[256:], z[2:], s[2:] = q[:256], z[:2], s[:2]
    pk, pz = oracle.pack_nibbles(q), oracle.pack_nibbles(z)
    x[1::2, 300] += 4.0
    s = (s.float() * 2.0 ** 20).bfloat16()
    x = (x * 2.0 ** 110).bfloat16()
    out = torch.ops.mi355q.w4a16_gemm(x.to(dev), pk.to(dev), s.to(dev), pz.to(dev), False, torch.float32, None).cpu()
    ref = x.double() @ ((q - z.repeat_interleave(128, 0)).double() * s.double().repeat_interleave(128, 0))
    top = torch.finfo(torch.float32).max
    assert (ref[1::2].abs() > 2 * top).any() and (ref.abs() < top / 2).any()
    assert torch.isfinite(out[ref.abs() < top / 2]).all()
    past = ref.abs() > 2 * top
    assert torch.equal(out[past].double(), ref[past].sign() * float("inf"))


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["bf16", "e5m2"])
@pytest.mark.parametrize("K", [256, 2048])      # in one part, in several
def test_scales_near_the_end_of_the_range(oracle, dev, K, act):
    """Scales of 2^120 beside ordinary ones, in the last group and in others: rows of zeros stay zeros, small activations give what they should."""
    gen = torch.Generator().manual_seed(K)
    M, N = 16, 544
    q, z, s, pk, pz = weights(oracle, gen, K, N, 128, False, True, pow2=True)
    s[0, 1::2] = s[-1, 2::4] = 2.0 ** 120
    x = torch.randint(-3, 4, (M, K), generator=gen).double()
    x[3] = x[8, -128:] = 0.0
    tiny = 2.0 ** (-100 if act == "bf16" else -16)
    x *= torch.where(torch.arange(M) < 12, tiny, 1.0)[:, None]
    ref = x @ ((q - z.repeat_interleave(128, 0)).double() * s.double().repeat_interleave(128, 0))
    if act == "bf16":
        out = torch.ops.mi355q.w4a16_gemm(x.bfloat16().to(dev), pk.to(dev), s.to(dev), pz.to(dev), False, torch.float32, None).cpu()
    else:
        out = torch.ops.mi355q.w4a8_gemm(x.to(E5).to(dev), pk.to(dev), s.to(dev), pz.to(dev), False, torch.float32, None, None).cpu()
    assert (out[3] == 0).all()
    # fp32 sums: a rounding of 2^-24 of the sum of magnitudes per group and part
    bound = (x.abs() @ (15 * s.double().repeat_interleave(128, 0))) * ((K // 128 + 16) * 2.0 ** -23)
    inside = (x.abs() @ (15 * s.double().repeat_interleave(128, 0))) < torch.finfo(torch.float32).max / 2   # every partial sum too
    assert inside[:12].all()
    assert torch.isfinite(out[inside]).all() and ((out.double() - ref).abs() <= bound)[inside].all()


@pytest.mark.gpu
def test_same_bits_whoever_adds_the_parts_up(oracle, pkg, dev):
    """The parts share the sum, or the last one adds all of them up (split_k < 0); the counters are zero afterwards; fewer parts where
    the workspace has less room than the plan wants."""
    lib = pkg.capi()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    gen = torch.Generator().manual_seed(9)
    for M, K, N in [(16, 4096, 14336), (3, 8192, 1024), (11, 2432, 5152)]:
        q, z, s, pk, pz = weights(oracle, gen, K, N, 128, False, True)
        x = torch.randn(M, K, generator=gen).bfloat16().to(dev)
        pkd, sd, pzd = pk.to(dev), s.to(dev), pz.to(dev)
        nbytes = lib.mi355q_w4a16_gemm_workspace_bytes(M, N, K, 128, pkg.BF16)
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
        outs = []
        for split in (1, -1, 1, -1, -1, 1):
            C = torch.full((M, N + 8), -5.0, device=dev)
            assert lib.mi355q_w4a16_gemm(x.data_ptr(), pkg.BF16, K, pkd.data_ptr(), N // 8, sd.data_ptr(), pkg.BF16, pzd.data_ptr(), 0, 128,
                                         C.data_ptr(), pkg.F32, N + 8, M, N, K, None, ws.data_ptr(), nbytes, split, st) == 0
            outs.append(C)
        torch.cuda.synchronize()
        assert not ws[:1024].any() and (outs[0][:, N:] == -5.0).all()
        assert all(torch.equal(outs[0], o) for o in outs[1:]), (M, K, N)
        rel, ok = gemm_errors(outs[0][:, :N], oracle.torch_w4a16_gemm(x.cpu(), pk, s, pz, False, torch.float32))
        assert rel < 2e-4 and ok, rel
    # fp8 activations with room for two parts only, and with none at all
    M, K, N = 16, 4096, 1024
    q, z, s, pk, pz = weights(oracle, gen, K, N, 128, False, True, pow2=True)
    a = torch.randint(-4, 5, (M, K), generator=gen).float()
    expect = a.double() @ ((q - z.repeat_interleave(128, 0)).double() * s.double().repeat_interleave(128, 0))
    Ad, pkd, sd, pzd = a.to(E4).to(dev), pk.to(dev), s.to(dev), pz.to(dev)
    least = 4 * 4 * 32 * 256 * 4 + 1024                  # what the shape needed in parts of eight stages and strips of 256 columns
    need = lib.mi355q_w4a8_gemm_workspace_bytes(M, N, K, 128, pkg.BF16)
    assert need >= least
    for nbytes in (need, least, 0):
        ws = torch.zeros(max(nbytes, 16), dtype=torch.uint8, device=dev)
        C = torch.full((M, N), -5.0, device=dev)
        assert lib.mi355q_w4a8_gemm(Ad.data_ptr(), pkg.E4M3FN, K, pkd.data_ptr(), N // 8, sd.data_ptr(), pkg.BF16, pzd.data_ptr(), 0, 128,
                                    C.data_ptr(), pkg.F32, N, M, N, K, None, ctypes.c_float(1.0), pkg.GS_NONE, None,
                                    ws.data_ptr() if nbytes else None, nbytes, st) == 0
        torch.cuda.synchronize()
        assert torch.equal(C.cpu().double(), expect), nbytes


@pytest.mark.timeout(300)
def test_generated_code():
    text = isa_check.compile_to_isa("w4_stream.hip")
    assert isa_check.scan(text) == [] and isa_check.scratch_bytes(text) == {}
    orders = isa_check.exchange_order(text)
    assert len(orders) == 6
    for name, seq in orders.items():
        # sums stored past the XCD's caches, acknowledged, barrier, arrival; then a barrier before the others' sums are read
        assert "F" not in seq and re.search(r"S{8}WBA", seq) and re.search(r"A.*B.*L{8}", seq), (name, seq)
