"""cast_to_fp8 with amax at the edges of its launch shapes (one workgroup, up to 2^21 elements, one logical block per
workgroup, several), many calls in a row (each clears the next one's word), streams, threads, and the C entries that
raise a running maximum and chain calls."""
import ctypes
import threading

import pytest
import torch

from helpers import E4

pytestmark = pytest.mark.gpu
SIZES = [1, 8, 4096, 16384, 16392, 2 ** 21, 2 ** 21 + 8, 2 ** 22, 2 ** 22 + 8, 2 ** 23, 2 ** 23 + 40, 2 ** 24 + 3]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_amax_and_codes(oracle, dev, n, dtype):
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, generator=g).to(dtype)
    x[torch.randint(0, n, (1,), generator=g)] = -7.25  # the maximum somewhere
    scale = torch.tensor(40.0)
    y, amax = torch.ops.hpu.cast_to_fp8_v2(x.to(dev), scale.to(dev), False, True, E4)
    y_ref, _ = oracle.c_cast_to_fp8(x, scale, E4, True)
    assert amax.shape == () and amax.item() == 7.25
    assert torch.equal(y.cpu().view(torch.uint8), y_ref.view(torch.uint8))


# rows at the edges of how many vectors a thread asks for: 512, 1024 and 2048 vectors a row, one more, and short ones; small
# tensors (up to 2^21 elements) and larger ones
@pytest.mark.parametrize("rows,cols", [(3, 64), (5, 16384), (600, 4096), (513, 4104), (300, 8192), (260, 8200), (140, 16384), (130, 16392), (2100, 1000),
                                       (20000, 120), (100, 40960)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("per_row", [False, True])
def test_amax_and_codes_with_row_and_column_scales(oracle, dev, rows, cols, dtype, per_row):
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, cols, generator=g).to(dtype)
    x.view(-1)[torch.randint(0, rows * cols, (1,), generator=g)] = 9.5
    scale, shape = (torch.rand(rows, 1, generator=g) + 20, [rows, 1]) if per_row else (torch.rand(cols, generator=g) + 20, [1, cols])
    y, amax = torch.ops.hpu.cast_to_fp8_v2(x.to(dev), scale.to(dev), False, True, E4, shape)
    y_ref, amax_ref = oracle.c_cast_to_fp8(x, scale.reshape(-1), E4, True, scale_shape=shape)
    assert amax.item() == 9.5 == float(amax_ref)
    assert torch.equal(y.cpu().view(torch.uint8), y_ref.view(torch.uint8))


# no whole vectors in a row: an element per thread without amax, eight with it (2048 a workgroup)
@pytest.mark.parametrize("rows,cols", [(1, 3), (3, 683), (2048, 1), (293, 7), (3001, 1001)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("is_amax", [False, True])
def test_ragged_rows_with_column_scales(oracle, dev, rows, cols, dtype, is_amax):
    g = torch.Generator().manual_seed(cols)
    x = torch.randn(rows, cols, generator=g).to(dtype)
    x.view(-1)[-1] = 9.5  # in the last element
    scale = torch.rand(cols, generator=g) + 20
    y, amax = torch.ops.hpu.cast_to_fp8_v2(x.to(dev), scale.to(dev), False, is_amax, E4, [1, cols])
    y_ref, _ = oracle.c_cast_to_fp8(x, scale, E4, True, scale_shape=[1, cols])
    assert torch.equal(y.cpu().view(torch.uint8), y_ref.view(torch.uint8))
    assert amax.item() == 9.5 if is_amax else amax.shape == (0,)


def test_column_scales_cost_little_more_than_one_scale(dev):
    x, scale = torch.randn(4096, 4096, device=dev).bfloat16(), torch.rand(4096, device=dev) + 0.5

    def best(s, shape):
        times = []
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(40):
                torch.ops.hpu.cast_to_fp8_v2(x, s, False, True, E4, shape)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    # 1.5 measured; 4.6 with eight vectors in flight per thread where a row holds one
    assert best(scale, [1, 4096]) < 3.0 * best(scale[:1].reshape(()), None)


def test_every_call_has_its_own_word(dev):
    """Many calls on two streams, all results kept."""
    xs = [torch.full((5,), float(i + 1), device=dev).bfloat16() for i in range(8)]
    side = torch.cuda.Stream()
    got = []
    for i in range(600):
        if i % 3 == 2:
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                got.append((i, torch.ops.hpu.cast_to_fp8_v2(xs[i % 8], None, False, True, E4)[1]))
        else:
            got.append((i, torch.ops.hpu.cast_to_fp8_v2(xs[i % 8], None, False, True, E4)[1]))
    torch.cuda.synchronize()
    assert all(a.item() == i % 8 + 1 for i, a in got)
    got[0][1].fill_(99.0)  # writing to one result leaves the others alone
    assert all(a.item() == i % 8 + 1 for i, a in got[1:])


def test_amax_is_an_ordinary_tensor(dev):
    """Whatever mode the call was made in that cleared the word: own storage and version, resizable, an inference tensor only by the call's own mode."""
    x = torch.tensor([-3.0, 1.0], device=dev).bfloat16()
    call = lambda: torch.ops.hpu.cast_to_fp8_v2(x, None, False, True, E4)[1]  # noqa: E731
    for _ in range(70):
        with torch.inference_mode():
            inside = call()
        first, second = call(), call()
        assert inside.is_inference() and not first.is_inference()
        assert first.untyped_storage().nbytes() == 4 and first.storage_offset() == 0 and first._base is None
        assert first.untyped_storage().device == x.device == first.device and first.untyped_storage().resizable()
        version = second._version
        first.mul_(2)  # refused for an inference tensor
        assert second._version == version
        first.resize_(100).fill_(-1.0)
        assert second.item() == 3.0 and inside.item() == 3.0


def test_no_call_pays_for_others(dev):
    """Every call allocates its codes, and its own or the next call's word: no call makes a stock for later ones."""
    x = torch.ones(4096, device=dev).bfloat16()
    kept = []
    for _ in range(200):
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        kept.append(torch.ops.hpu.cast_to_fp8_v2(x, None, False, True, E4))
        assert torch.cuda.memory_stats()["allocation.all.allocated"] - before <= 3
    assert all(a.item() == 1.0 for _, a in kept)


def test_threads_on_one_stream_and_on_their_own(dev):
    """Threads that share a stream find no word now and then and clear their own; none sees another's."""
    tops = [float(2 ** i) for i in range(8)]
    xs = [torch.full((1000 + i,), t, device=dev).bfloat16() for i, t in enumerate(tops)]
    torch.cuda.synchronize()
    shared = torch.cuda.Stream()
    got, errors = [[] for _ in tops], []

    def work(i):
        try:
            with torch.cuda.stream(shared if i < 5 else torch.cuda.Stream()):
                for _ in range(100):
                    got[i].append(torch.ops.hpu.cast_to_fp8_v2(xs[i], None, False, True, E4)[1])
                torch.cuda.current_stream().synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for i, t in enumerate(tops):
        assert torch.stack(got[i]).cpu().eq(t).all()


@pytest.mark.parametrize("n", [0, 5, 4096, 4099, 2 ** 22 + 3])
def test_chained_calls(pkg, dev, n):
    """The C entry: each call's maximum in the word that the call before it cleared, tails and empty tensors among them."""
    lib = pkg.capi()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    words = torch.full((4,), 77.0, device=dev)
    y = torch.empty(n, dtype=E4, device=dev)
    word = lambda i: words.data_ptr() + 4 * i  # noqa: E731
    for i, top in enumerate((5.0, 3.0, 4.0)):
        x = torch.full((n,), -top, device=dev).bfloat16()
        assert lib.mi355q_cast_to_fp8_amax_chain(x.data_ptr(), pkg.BF16, y.data_ptr(), pkg.E4M3FN, None, 1.0, pkg.SCALE_NONE, n, 1, 1, word(i),
                                                 int(i > 0), word(i + 1) if i < 2 else None, st) == 0
    assert words.tolist() == ([5.0, 3.0, 4.0] if n else [0.0, 0.0, 0.0]) + [77.0]
    for amax, following in ((None, word(0)), (word(0), word(0))):
        assert lib.mi355q_cast_to_fp8_amax_chain(x.data_ptr(), pkg.BF16, y.data_ptr(), pkg.E4M3FN, None, 1.0, pkg.SCALE_NONE, n, 1, 1, amax, 1, following,
                                                 st) != 0


def test_running_maximum(pkg, dev):
    lib = pkg.capi()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    am = torch.tensor([2.0], device=dev)
    y = torch.empty(64, dtype=E4, device=dev)
    for top, want in ((1.0, 2.0), (3.5, 3.5), (0.25, 3.5)):
        x = torch.full((64,), -top, device=dev)
        assert lib.mi355q_cast_to_fp8_running_amax(x.data_ptr(), pkg.F32, y.data_ptr(), pkg.E4M3FN, None, 1.0, pkg.SCALE_NONE, 64, 1, 1,
                                                   am.data_ptr(), st) == 0
        assert am.item() == want
    assert lib.mi355q_cast_to_fp8_running_amax(x.data_ptr(), pkg.F32, y.data_ptr(), pkg.E4M3FN, None, 1.0, pkg.SCALE_NONE, 64, 1, 1, None, st) != 0
