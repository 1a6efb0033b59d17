"""More elements than a launch has threads (2^32 in one dimension of a grid, which is cut off without an error beyond): kernels
with one thread per element, on unaligned buffers or sizes that no vector kernel takes.  Patterns that repeat every P elements,
the whole result against its first P, and those against what the same entry point gives for a small tensor."""
import pytest

pytestmark = pytest.mark.gpu
P = 127
N = (1 << 32) // P * P + 40 * P   # a little over 2^32


def need(gib):
    import torch
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < gib << 30:
        pytest.skip("needs %d GiB" % gib)


def repeats(t, n):
    rows = t[:n].view(-1, P)
    return all(bool((part == rows[:1]).all()) for part in rows.split(1 << 22))


def filled(dev, pattern, n):
    """pattern over n elements, one element off the buffer's alignment"""
    import torch
    buf = torch.empty(n + 1, dtype=pattern.dtype, device=dev)
    buf[1:].view(-1, P).copy_(pattern.view(1, -1))
    return buf


def test_fill(hip, dev):
    import ctypes as C
    import torch
    need(20)
    n = (1 << 34) + 4096
    buf = torch.zeros(n, dtype=torch.uint8, device=dev)
    hip._check(hip.raw().itexhip_memset8_async(C.c_void_p(buf.data_ptr()), C.c_uint8(0x5a), C.c_size_t(n), C.c_void_p(0)))
    torch.cuda.synchronize()
    assert all(bool((part == 0x5a).all()) for part in buf.split(1 << 30))
    hip._check(hip.raw().itexhip_memset32_async(C.c_void_p(buf.data_ptr()), C.c_uint32(0x01020304), C.c_size_t(n), C.c_void_p(0)))
    torch.cuda.synchronize()
    assert all(bool((part == 0x01020304).all()) for part in buf.view(torch.int32).split(1 << 28))


def test_copy(hip, dev):
    import torch
    need(12)
    src = filled(dev, torch.arange(P, dtype=torch.uint8, device=dev), N)
    dst = torch.full((N + 1,), 255, dtype=torch.uint8, device=dev)
    hip.memcpy_d2d_async(dst[1:], src[1:], N)
    torch.cuda.synchronize()
    assert torch.equal(dst[1:P + 1], src[1:P + 1]) and repeats(dst[1:], N)


@pytest.mark.parametrize("per_channel", [False, True])
def test_quantize_and_dequantize(hip, dev, per_channel):
    import torch
    need(48)
    pattern = torch.linspace(-1.0, 1.0, P, device=dev)
    scales = torch.linspace(50.0, 127.0, P, device=dev)
    x = filled(dev, pattern, N)[1:]
    q = torch.full((N + 1,), 99, dtype=torch.int8, device=dev)[1:]
    small = torch.empty(P + 1, dtype=torch.int8, device=dev)[1:]
    if per_channel:
        hip.quantize_axis(x, q, N // P, P, 1, hip.QINT8, scales)
        hip.quantize_axis(x, small, 1, P, 1, hip.QINT8, scales)
    else:
        hip.quantize(x, q, N, hip.QINT8, 100.0)
        hip.quantize(x, small, P, hip.QINT8, 100.0)
    torch.cuda.synchronize()
    assert torch.equal(q[:P], small) and repeats(q, N)
    x.fill_(7.0)
    small = torch.empty(P + 1, device=dev)[1:]
    if per_channel:
        hip.dequantize_axis(q, x, N // P, P, 1, hip.QINT8, scales)
        hip.dequantize_axis(q, small, 1, P, 1, hip.QINT8, scales)
    else:
        hip.dequantize(q, x, N, hip.QINT8, 0.01)
        hip.dequantize(q, small, P, hip.QINT8, 0.01)
    torch.cuda.synchronize()
    assert torch.equal(x[:P], small) and repeats(x, N)


@pytest.mark.parametrize("per_channel", [False, True])
def test_16_bit_quantize_and_dequantize(hip, dev, per_channel):
    import torch
    need(24)
    scales = torch.linspace(50.0, 127.0, P, device=dev)
    x = filled(dev, torch.linspace(-1.0, 1.0, P, device=dev).bfloat16(), N)[1:]
    q = torch.full((N + 1,), 99, dtype=torch.int8, device=dev)[1:]
    small = torch.empty(P + 1, dtype=torch.int8, device=dev)[1:]
    if per_channel:
        hip.quantize_axis_bf16(x, q, N // P, P, 1, hip.QINT8, scales)
        hip.quantize_axis_bf16(x, small, 1, P, 1, hip.QINT8, scales)
    else:
        hip.quantize_bf16(x, q, N, hip.QINT8, 100.0)
        hip.quantize_bf16(x, small, P, hip.QINT8, 100.0)
    torch.cuda.synchronize()
    assert torch.equal(q[:P], small) and repeats(q, N)
    x.fill_(7.0)
    small = torch.empty(P + 1, dtype=torch.bfloat16, device=dev)[1:]
    if per_channel:
        hip.dequantize_axis16(q, x, N // P, P, 1, hip.QINT8, hip.BFLOAT16, scales)
        hip.dequantize_axis16(q, small, 1, P, 1, hip.QINT8, hip.BFLOAT16, scales)
    else:
        hip.dequantize16(q, x, N, hip.QINT8, hip.BFLOAT16, 0.01)
        hip.dequantize16(q, small, P, hip.QINT8, hip.BFLOAT16, 0.01)
    torch.cuda.synchronize()
    assert torch.equal(x[:P], small) and repeats(x, N)


def test_requantize(hip, dev):
    import torch
    need(48)
    x = filled(dev, torch.arange(P, dtype=torch.int32, device=dev) * 1000 - 60000, N)[1:]
    q = torch.full((N + 1,), 99, dtype=torch.int8, device=dev)[1:]
    small = torch.empty(P + 1, dtype=torch.int8, device=dev)[1:]
    hip.requantize(x, q, N, hip.QINT8, 2e-3)
    hip.requantize(x, small, P, hip.QINT8, 2e-3)
    torch.cuda.synchronize()
    assert torch.equal(q[:P], small) and repeats(q, N)


def test_rows_quantized_one_by_one(hip, dev):
    """2^22 rows: a workgroup of 1024 threads each."""
    import torch
    rows = (1 << 22) // P * P + 2 * P
    x = (torch.linspace(-1.0, 1.0, 4 * P, device=dev).view(P, 4) ** 3).repeat(rows // P, 1)
    q = torch.full((rows, 4), 99, dtype=torch.uint8, device=dev)
    lo, hi = (torch.full((rows,), 9.0, device=dev) for _ in range(2))
    hip.quantize_dynamic_rows(x, q, rows, 4, hip.QUINT8, hip.MIN_FIRST, 0.01, lo, hi)
    sq, slo, shi = torch.empty(P, 4, dtype=torch.uint8, device=dev), *(torch.empty(P, device=dev) for _ in range(2))
    hip.quantize_dynamic_rows(x, sq, P, 4, hip.QUINT8, hip.MIN_FIRST, 0.01, slo, shi)
    torch.cuda.synchronize()
    for got, want in ((q, sq), (lo, slo), (hi, shi)):
        got = got.view(rows // P, P, -1)
        assert torch.equal(got[0], want.view(P, -1)) and bool((got == got[:1]).all())


def test_matmul_per_output(hip, dev):
    """itexhip_qgemm_naive: 2^32 outputs of 33 columns."""
    import torch
    need(12)
    rows, n = (1 << 32) // 33 // P + 9, 33
    M = rows * P
    a = torch.arange(P, dtype=torch.int8, device=dev).repeat(rows)
    w = torch.arange(-16, 17, dtype=torch.int8, device=dev)
    ep = hip.Epilogue()
    ep.n_scales = 1
    scale, bias = torch.full((1,), 1.0 / 16.0, device=dev), torch.zeros(n, device=dev)
    out = torch.full((rows, P, n), 99, dtype=torch.int8, device=dev)
    small = torch.empty(P, n, dtype=torch.int8, device=dev)
    for o, m in ((out, M), (small, P)):
        hip.qgemm_naive(a, hip.QINT8, w, False, m, 1, n, scale, bias, ep, hip.QINT8, o)
    torch.cuda.synchronize()
    assert torch.equal(out[0], small) and bool((out == out[:1]).all())
    want = (torch.arange(P).view(-1, 1) * torch.arange(-16, 17).view(1, -1) / 16.0).round().clamp(-128, 127).to(torch.int8)
    assert torch.equal(small.cpu(), want)


def test_batch_matmul_rows_of_one_column(hip, dev):
    """2^30 rows of one column: 2^24 tiles of one matrix."""
    import torch
    need(8)
    M = (1 << 30) // P * P + 70 * P
    x = torch.arange(P, dtype=torch.int8, device=dev).repeat(M // P)
    y = torch.full((1,), 3, dtype=torch.int8, device=dev)
    p, _ = hip.bmm_params((1, M, 1), (1, 1, 1), False, False, hip.BFLOAT16, 0.25)
    out = torch.full((M,), 99.0, dtype=torch.bfloat16, device=dev)
    hip.qbatch_matmul(p, x, y, out)
    torch.cuda.synchronize()
    assert torch.equal(out[:P].float(), (x[:P].float() * 0.75).bfloat16().float()) and repeats(out, M)
