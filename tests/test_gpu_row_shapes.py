"""The row kernels (quantize_rows, silu_mul_quantize_rows) at the edges of how they spread a row over a workgroup: one
vector per thread and two, four from 512 rows on, rows that end inside a wave, and a target past the largest code."""
import ctypes

import pytest
import torch

from helpers import E4, E5

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


def test_target_past_the_largest_code_saturates(pkg, dev):
    lib = pkg.capi()
    x = torch.tensor([[1.0, -2.0, 3.0, 4.0, -4.0, 0.5, 0.0, 1.5]]).bfloat16().to(dev)
    y = torch.empty(1, 8, dtype=E4, device=dev)
    inv = torch.empty(1, device=dev)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mi355q_quantize_rows(x.data_ptr(), pkg.BF16, 1, 8, y.data_ptr(), pkg.E4M3FN, 1024.0, None, inv.data_ptr(), st) == 0
    assert y.cpu().float()[0].tolist() == [256.0, -448.0, 448.0, 448.0, -448.0, 128.0, 0.0, 384.0]
