"""Prepared 4-bit weights past 16 rows: the GEMV's 32-row slabs and the GEMM that
decodes its operand (128- and 256-row tiles), at partial slabs, tiles and K
steps, every block size, both types, with and without zero points, operands that
only the general path takes, and the ONNX packing, which is tiled first.  Small
integers and power-of-two scales, whose sums are exact in any order, against
64-bit products; one-hot rows with random scales, which give the dequantised
weights themselves, bit for bit against the general path (operands 2 bytes off)
and, for that path, against fp32 arithmetic rounded once."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev(olamd):
    olamd.init(0)
    return torch.device("cuda:0")


# rows 17 to 96 are slabs at these sizes, the rest the GEMM
@pytest.mark.parametrize("M,K,N", [(17, 128, 16), (33, 96, 77), (64, 384, 4112), (97, 256, 8208), (257, 32, 8208),
                                   (129, 416, 11024), (1500, 224, 2064), (2049, 160, 2176), (300, 96, 4106), (1300, 64, 2040)], ids=str)
@pytest.mark.parametrize("block", [8, 32, 64, 128, 0, -1])  # 0: a scale per column, -1: one scale
def test_prepared_rows(olamd, dev, M, K, N, block):
    if block > 0 and K % block:
        K = (K + block - 1) // block * block
    g = torch.Generator(device=dev).manual_seed(M + N + block)
    ints = lambda lo, hi, sh: torch.randint(lo, hi, sh, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    shape, axis = ((K // block, N), 0) if block > 0 else (((N,), 1) if block == 0 else ((), 1))
    full = lambda t: t.repeat_interleave(block, 0) if block > 0 else t  # noqa: E731
    pack = lambda t: torch.nn.functional.pad(t.reshape(-1) & 15, (0, t.numel() % 2)).view(-1, 2)  # noqa: E731
    nibbles = lambda t: (pack(t)[:, 0] | pack(t)[:, 1] << 4).to(torch.uint8)  # noqa: E731
    a = ints(-2, 3, (M, K))
    onehot = torch.zeros((M, K), dtype=torch.float16, device=dev)
    onehot[torch.arange(M, device=dev), ints(0, K, (M,)).long()] = 1
    for code, lo in ((olamd.INT4, -8), (olamd.UINT4, 0)):
        w, z = ints(lo, lo + 16, (K, N)), ints(lo, lo + 16, shape)
        s2 = torch.pow(2.0, -ints(0, 4, shape).float()).half()
        rnd = (torch.rand(shape, generator=g, device=dev) * 0.02 + 0.001).half()
        onnx = nibbles(w)
        pw = olamd.prepare_weight(onnx, code, (K, N))
        odd = torch.empty(M * K + 1, dtype=torch.float16, device=dev)[1:].view(M, K)  # 2-byte aligned
        odd.copy_(a)
        for zp in (None, z):
            zb = None if zp is None else nibbles(zp)
            deq = (w - (0 if zp is None else full(zp))).double() * full(s2).double()
            want = (a.double() @ deq).to(torch.float32).half()
            for x in (a.half(), odd):
                y = olamd.dequantize_linear_matmul(x, pw, s2, zb, axis=axis, x_dtype=code)
                assert torch.equal(y, want)
            y = olamd.dequantize_linear_matmul(a.half(), onnx, s2, zb, axis=axis, x_dtype=code, x_shape=(K, N))
            assert torch.equal(y, want)
            y = olamd.dequantize_linear_matmul(onehot, pw, rnd, zb, axis=axis, x_dtype=code)
            odd.copy_(onehot)
            general = olamd.dequantize_linear_matmul(odd, pw, rnd, zb, axis=axis, x_dtype=code)
            assert torch.equal(y, general)
            odd.copy_(a)


@pytest.mark.parametrize("K,N,block", [(8, 8, 8), (264, 24, 8), (96, 648, 32), (264, 1032, 88), (100, 72, 4),
                                       (130, 20, 65), (257, 16, 0), (300, 77, -1)], ids=str)
@pytest.mark.parametrize("bf16", [False, True])
def test_general_weights(olamd, dev, K, N, block, bf16):
    """The general path's dequantisation, value by value: the identity as
    activations (bf16 with FLOAT scales and a Cast, or fp16 2 bytes off), every
    weight type, row-major and tiled, whole and partial groups of rows and columns."""
    g = torch.Generator(device=dev).manual_seed(K + N + block)
    ints = lambda lo, hi, sh: torch.randint(lo, hi, sh, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    dt = torch.bfloat16 if bf16 else torch.float16
    a = torch.empty(K * K + 1, dtype=dt, device=dev)[1:].view(K, K)
    a.copy_(torch.eye(K, device=dev))
    shape, axis = ((K // block, N), 0) if block > 0 else (((N,), 1) if block == 0 else ((), 1))
    full = lambda t: t.repeat_interleave(block, 0) if block > 0 else t  # noqa: E731
    pack = lambda t: torch.nn.functional.pad(t.reshape(-1) & 15, (0, t.numel() % 2)).view(-1, 2)  # noqa: E731
    nibbles = lambda t: (pack(t)[:, 0] | pack(t)[:, 1] << 4).to(torch.uint8)  # noqa: E731
    scale = torch.rand(shape, generator=g, device=dev) * 0.02 + 0.001
    scale = scale if bf16 else scale.half()
    kw = dict(axis=axis, cast_to=olamd.BFLOAT16 if bf16 else 0)
    for code, lo, bits in ((olamd.INT8, -128, 8), (olamd.UINT8, 0, 8), (olamd.INT4, -8, 4), (olamd.UINT4, 0, 4)):
        w, z = ints(lo, lo + (1 << bits), (K, N)), ints(lo, lo + (1 << bits), shape)
        for zp in (None, z):
            want = ((w - (0 if zp is None else full(zp))).float() * full(scale).float()).to(dt)
            store = nibbles if bits == 4 else (lambda t: t.to(torch.int8 if lo else torch.uint8))  # noqa: E731
            zb = None if zp is None else store(zp)
            y = olamd.dequantize_linear_matmul(a, store(w), scale, zb, x_dtype=code, x_shape=(K, N), **kw)
            assert torch.equal(y, want)
            if bits == 4:
                pw = olamd.prepare_weight(nibbles(w), code, (K, N))
                assert torch.equal(olamd.dequantize_linear_matmul(a, pw, scale, zb, x_dtype=code, **kw), want)


@pytest.mark.parametrize("M", [1, 16, 17, 40, 2000])
@pytest.mark.parametrize("K,N", [(32, 48), (160, 80), (640, 272), (1696, 1040)], ids=str)
@pytest.mark.parametrize("block", [8, 32, 0, -1])
def test_padding_of_large_scales(olamd, dev, M, K, N, block):
    """Rows past K, and whole groups past a wave's share, add nothing where a
    padding code times the scale overflows fp16, or the scale is infinite: one-hot
    rows of weights that stay below 65504, then ones times an infinite weight."""
    g = torch.Generator(device=dev).manual_seed(M + K + N + block)
    ints = lambda lo, hi, sh: torch.randint(lo, hi, sh, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    shape, axis = ((K // block, N), 0) if block > 0 else (((N,), 1) if block == 0 else ((), 1))
    full = lambda t: t.repeat_interleave(block, 0) if block > 0 else t  # noqa: E731
    nibbles = lambda t: ((t.reshape(-1, 2)[:, 0] & 15) | (t.reshape(-1, 2)[:, 1] & 15) << 4).to(torch.uint8)  # noqa: E731
    scale = torch.full(shape, 12000.0, dtype=torch.float16, device=dev)
    at = ints(0, K, (M,)).long()
    onehot = torch.zeros((M, K), dtype=torch.float16, device=dev)
    onehot[torch.arange(M, device=dev), at] = 1
    ones = torch.ones((M, K), dtype=torch.float16, device=dev)
    for code, mid in ((olamd.INT4, 0), (olamd.UINT4, 8)):
        w = ints(mid - 5, mid + 6, (K, N))
        for zp in (mid != 0, True):
            z = torch.full((max(2, scale.numel()),), mid, dtype=torch.int32, device=dev)
            zb = (nibbles(z) if scale.numel() > 1 else nibbles(z)[:1]) if zp else None
            pw = olamd.prepare_weight(nibbles(w), code, (K, N))
            want = ((w - mid).float() * 12000.0).half()[at]
            y = olamd.dequantize_linear_matmul(onehot, pw, scale, zb, axis=axis, x_dtype=code)
            assert torch.equal(y, want), (code, zp)
            inf = scale.clone()
            inf[...] = float("inf")
            up = olamd.prepare_weight(nibbles((w - mid).abs().clamp(1, 5) + mid), code, (K, N))
            y = olamd.dequantize_linear_matmul(ones, up, inf, zb, axis=axis, x_dtype=code)
            assert bool((y == float("inf")).all()), (code, zp)
