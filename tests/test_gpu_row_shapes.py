"""The row kernels (quantize_rows, silu_mul_quantize_rows) at the edges of how they spread a row over a workgroup: one
vector per thread and two, four from 512 rows on, rows that end inside a wave, and a target past the largest code."""
import ctypes

import pytest
import torch

from helpers import E4, E5, assert_fp8_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 8), (1, 512), (3, 8192), (2, 8200), (1, 16384), (511, 520), (512, 520), (600, 2056), (513, 16384)])
@pytest.mark.parametrize("fmt", [E4, E5])
def test_rows_of_every_shape(oracle, dev, rows, cols, fmt):
    g = torch.Generator().manual_seed(rows + cols)
    gate = (torch.randn(rows, cols, generator=g) * 3).bfloat16()
    up = torch.randn(rows, cols, generator=g).bfloat16()
    own = torch.ops.mi355q
    y, inv = own.quantize_rows(gate.to(dev), fmt)
    y_ref, inv_ref = oracle.quantize_rows(gate, fmt)
    assert torch.equal(y.cpu().view(torch.uint8), y_ref.view(torch.uint8)) and torch.equal(inv.cpu(), inv_ref)
    h, h_inv = own.silu_mul_quantize_rows(gate.to(dev), up.to(dev), fmt)
    h_ref, h_inv_ref = oracle.quantize_rows(oracle.c_silu_mul_bf16(gate, up), fmt)
    assert torch.equal(h.cpu().view(torch.uint8), h_ref.view(torch.uint8)) and torch.equal(h_inv.cpu(), h_inv_ref)


@pytest.mark.parametrize("rows,cols", [(1, 16392), (511, 16448), (600, 20808), (3, 32768), (2, 32776)])  # the last: three steps again
def test_rows_of_more_than_two_vectors_per_thread(oracle, dev, rows, cols):
    g = torch.Generator().manual_seed(rows + cols)
    gate = (torch.randn(rows, cols, generator=g) * 3).bfloat16()
    own = torch.ops.mi355q
    for x in (gate, gate[:, : cols // 2].float()):
        y, inv = own.quantize_rows(x.to(dev), E4)
        y_ref, inv_ref = oracle.quantize_rows(x, E4)
        assert torch.equal(y.cpu().view(torch.uint8), y_ref.view(torch.uint8)) and torch.equal(inv.cpu(), inv_ref)
    if cols > 32768:
        return  # aten's silu there
    up = torch.randn(rows, cols, generator=g).bfloat16()
    up[-1, 5] = float("inf")  # the row's scale is 0 and its codes as the oracle has them
    h, h_inv = own.silu_mul_quantize_rows(gate.to(dev), up.to(dev), E5)
    h_ref, h_inv_ref = oracle.quantize_rows(oracle.c_silu_mul_bf16(gate, up), E5)
    assert_fp8_equal(h, h_ref, E5, f"{rows} x {cols}")
    assert torch.equal(h_inv.cpu(), h_inv_ref)


def test_target_past_the_largest_code_saturates(pkg, dev):
    lib = pkg.capi()
    x = torch.tensor([[1.0, -2.0, 3.0, 4.0, -4.0, 0.5, 0.0, 1.5]]).bfloat16().to(dev)
    y = torch.empty(1, 8, dtype=E4, device=dev)
    inv = torch.empty(1, device=dev)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mi355q_quantize_rows(x.data_ptr(), pkg.BF16, 1, 8, y.data_ptr(), pkg.E4M3FN, 1024.0, None, inv.data_ptr(), st) == 0
    assert y.cpu().float()[0].tolist() == [256.0, -448.0, 448.0, 448.0, -448.0, 128.0, 0.0, 384.0]


@pytest.mark.parametrize("target", [-448.0, -1024.0, -60000.0, -1e5, 1e5, float("-inf")])
@pytest.mark.parametrize("fmt", [E4, E5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_target_of_any_sign_saturates(oracle, pkg, dev, target, fmt, dtype):
    """Codes past the largest finite one are that code, whatever the sign of the target, on aligned rows, on ragged ones and
    behind silu(gate) * up."""
    lib = pkg.capi()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator().manual_seed(9)
    gate, up = torch.randn(5, 136, generator=g).to(dtype), torch.randn(5, 136, generator=g).to(dtype)

    def reference(x):
        amax = x.float().abs().amax(1)
        scale = torch.clamp_max(torch.full_like(amax, target) / amax, oracle.ROW_SCALE_CAP)
        return oracle.c_cast_to_fp8(x, scale, fmt, scale_shape=[x.shape[0], 1])[0]

    code = {E4: pkg.E4M3FN, E5: pkg.E5M2}[fmt]
    for cols in (136, 133):
        x = gate[:, :cols].contiguous()
        y, xd = torch.empty(5, cols, dtype=fmt, device=dev), x.to(dev)
        assert lib.mi355q_quantize_rows(xd.data_ptr(), pkg.BF16 if dtype == torch.bfloat16 else pkg.F32, 5, cols, y.data_ptr(), code, target, None,
                                        None, st) == 0
        assert_fp8_equal(y, reference(x), fmt, f"{cols} columns")
    if dtype == torch.bfloat16:
        y, gd, ud = torch.empty(5, 136, dtype=fmt, device=dev), gate.to(dev), up.to(dev)
        assert lib.mi355q_silu_mul_quantize_rows(gd.data_ptr(), 136, ud.data_ptr(), 136, 5, 136, y.data_ptr(), code, target, None, None, None, st) == 0
        assert_fp8_equal(y, reference(oracle.c_silu_mul_bf16(gate, up)), fmt, "silu")


@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 8192), (2, 8200), (511, 520), (512, 520), (513, 16384)])
def test_saturating_form_at_every_row_shape(oracle, pkg, dev, rows, cols):
    """The codes of a target past the largest finite one at the row shapes of the first test."""
    lib = pkg.capi()
    g = torch.Generator().manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=g).bfloat16()
    xd, y = x.to(dev), torch.empty(rows, cols, dtype=E4, device=dev)

    def call(target):
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert lib.mi355q_quantize_rows(xd.data_ptr(), pkg.BF16, rows, cols, y.data_ptr(), pkg.E4M3FN, target, None, None, st) == 0

    call(1024.0)
    amax = x.float().abs().amax(1)
    ref = oracle.c_cast_to_fp8(x, torch.full_like(amax, 1024.0) / amax, E4, scale_shape=[rows, 1])[0]
    assert_fp8_equal(y, ref, E4)


def test_saturating_form_is_as_fast(pkg, dev):
    lib = pkg.capi()
    rows, cols = 8192, 512
    x, y = torch.randn(rows, cols, device=dev).bfloat16(), torch.empty(rows, cols, dtype=E4, device=dev)

    def best(target):
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        times = []
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(40):
                lib.mi355q_quantize_rows(x.data_ptr(), pkg.BF16, rows, cols, y.data_ptr(), pkg.E4M3FN, target, None, None, st)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    assert best(1024.0) < 2.0 * best(448.0)  # 7.8 with 1024 threads for every row, 1.1 with the rows' own shape
