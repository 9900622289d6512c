"""The order in which a causal prefill's workgroups take heads and query blocks (sdpa_place): every block is served, once; and the
form of the kernel for many workgroups (MANY).

A block of query rows does not depend on which workgroup served it, so the whole call equals its heads called one by one, which
are too few workgroups for the order to be changed or for that form, bit for bit.
"""
import math

import pytest
import torch

from helpers import E4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,length,keys,dim", [
    (90, 90, 300, 300, 128),       # heads that 8 does not divide: one group over all XCDs
    (33, 33, 1025, 1025, 128),     # as well, a number of workgroups that 8 does not divide, a short last round
    (88, 22, 385, 385, 128),       # all resident, every second round backwards, shared K and V
    (16, 4, 2100, 2100, 256),      # 17 query blocks of 16 heads: one round more than the first
    (544, 136, 300, 300, 64),      # more workgroups than are resident
    (144, 36, 1000, 1000, 64),     # five per CU, resident: every second round backwards
    (160, 160, 1000, 1000, 64),    # as many as are
    (136, 136, 130, 8192, 128),    # 17 heads per XCD in groups of 4, the last one of 1
    (24, 24, 1500, 1500, 72),      # rows through registers
])
def test_every_block_once(dev, heads, kv_heads, length, keys, dim):
    gen = torch.Generator(device=dev).manual_seed(heads)
    q = torch.randn((kv_heads, heads // kv_heads, length, dim), generator=gen, device=dev).to(E4)
    k = torch.randn((kv_heads, 1, keys, dim), generator=gen, device=dev).to(E4)
    v = torch.randn((kv_heads, 1, keys, dim), generator=gen, device=dev).to(E4)

    def run(q, k, v):
        return torch.ops.hpu.fp8_sdpa_recomp_fwd.scalar(q, k, v, None, 0.0, 1.0 / math.sqrt(dim), True, False, "None",
                                                        1.0, 1.0, 1.0, 128.0, 0.0, 1.0 / 128.0, False, False, None, "left")[0]
    out = run(q, k, v)
    assert torch.isfinite(out.float()).all()
    for a in range(kv_heads):
        for b in range(heads // kv_heads):
            assert torch.equal(out[a, b], run(q[a:a + 1, b:b + 1], k[a:a + 1], v[a:a + 1])[0, 0]), (a, b)


@pytest.mark.parametrize("dim", [128, 112, 64, 48])
@pytest.mark.parametrize("keys", [1, 63, 65, 128, 500])
@pytest.mark.parametrize("causal,scale,p_scale,pad", [
    (False, 0.1, 128.0, None),
    (True, 0.1, 128.0, None),
    (True, -0.1, 128.0, None),      # scores scaled in place: a scale that is not positive
    (False, 0.0, 1.0, None),
    (True, 0.1, 1000.0, None),      # probabilities that have to be limited
    (True, 0.1, 128.0, "left"),     # a first key
    (True, 0.1, 128.0, "right"),
])
def test_many_workgroups(dev, dim, keys, causal, scale, p_scale, pad):
    batch, heads, length = 4, 50, 500  # 800 workgroups: more than three per CU
    gen = torch.Generator(device=dev).manual_seed(keys)
    q, k, v = (torch.randn((batch, heads, n, dim), generator=gen, device=dev).to(E4) for n in (length, keys, keys))
    valid = None if pad is None else torch.tensor([keys, (keys + 1) // 2, max(keys - 64, 0), 1], dtype=torch.int32, device=dev)

    def run(q, k, v, valid):
        return torch.ops.hpu.fp8_sdpa_recomp_fwd.scalar(q, k, v, None, 0.0, scale, causal, False, "None", 1.0, 1.0, 1.0,
                                                        p_scale, 0.0, 1.0 / p_scale, False, False, valid, pad or "left")[0]
    out = run(q, k, v, valid)
    for b in range(batch):
        one = slice(b, b + 1)
        assert torch.equal(out[one], run(q[one], k[one], v[one], None if valid is None else valid[one])), b
