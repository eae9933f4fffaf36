"""The small-tile GEMM (csrc/tile_gemm.hpp) at the edges of its 64 x 64 and
128 x 128 tiles, its K steps and its guarded last step: rows that end inside a
16-byte piece, matrices of less than one piece, one past and one short of a
tile.  Integers against the oracle, bit for bit.  The 16-bit kinds use small
integers times powers of two, whose fp32 sums are exact in any order, so the
result is the exact sum rounded once to the output type."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 15, 3), (3, 130, 1), (1, 17, 7), (64, 128, 64), (65, 127, 63), (63, 129, 65), (5, 64, 16),
          (129, 200, 130), (200, 1, 77), (31, 256, 15), (7, 2049, 9),
          (1100, 72, 2100), (1025, 131, 2053)]  # more than 512 small tiles: 128 x 128 ones


@pytest.fixture(scope="module")
def dev(olamd):
    olamd.init(0)
    return torch.device("cuda:0")


def _T(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def _offset(t):
    """t at an address that is no multiple of 16 bytes (of its element size only)."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:].copy_(t.reshape(-1))
    return buf[1:].view(t.shape)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("dts", [(np.uint8, np.int8), (np.int8, np.uint8)], ids=["u8s8", "s8u8"])
def test_int8(olamd, oracle, dev, shape, dts):
    M, K, N = shape
    rng = np.random.default_rng(M * 7919 + K * 31 + N)
    a = rng.integers(np.iinfo(dts[0]).min, np.iinfo(dts[0]).max + 1, (M, K)).astype(dts[0])
    b = rng.integers(np.iinfo(dts[1]).min, np.iinfo(dts[1]).max + 1, (K, N)).astype(dts[1])
    za = rng.integers(np.iinfo(dts[0]).min, np.iinfo(dts[0]).max + 1, M).astype(dts[0])
    zb = rng.integers(np.iinfo(dts[1]).min, np.iinfo(dts[1]).max + 1, N).astype(dts[1])
    ta, tb = _offset(_T(a, dev)), _offset(_T(b, dev))
    y = olamd.matmul_integer(ta, tb, _T(za, dev), _T(zb, dev))
    sums = (a.astype(np.int64) - za[:, None]) @ (b.astype(np.int64) - zb)
    if M * K * N < 2_000_000:
        assert np.array_equal(oracle.matmul_integer(a, b, za.tolist(), zb.tolist()), sums)
    assert np.array_equal(y.cpu().numpy(), sums)
    s = [np.array(v, np.float32) for v in (0.02, 0.004, 0.3)]
    yz = np.array(3, dts[0])
    q = olamd.qlinear_matmul(ta, s[0], np.array(za[0]), tb, s[1], np.array(zb[0]), s[2], yz)
    if M * K * N < 2_000_000:
        want = oracle.qlinear_matmul(a, s[0], int(za[0]), b, s[1], int(zb[0]), s[2], yz)
    else:
        sums = (a.astype(np.int64) - int(za[0])) @ (b.astype(np.int64) - int(zb[0]))
        cs = np.float32(np.float32(s[0] * s[1]) / s[2])
        info = np.iinfo(dts[0])
        want = np.clip(np.rint(sums.astype(np.float32) * cs) + np.float32(yz), info.min, info.max).astype(dts[0])
    assert np.array_equal(q.cpu().numpy(), want)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_16_bit(olamd, dev, shape):
    M, K, N = shape
    g = torch.Generator(device=dev).manual_seed(K)
    ints = lambda lo, hi, sh: torch.randint(lo, hi, sh, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    a, b = ints(-2, 3, (2, M, K)), ints(-8, 9, (2, K, N))
    exact = torch.stack([x.double() @ y.double() for x, y in zip(a, b)])
    assert float(torch.stack([x.double().abs() @ y.double().abs() for x, y in zip(a, b)]).max()) < 2 ** 24
    for dt in (torch.float16, torch.bfloat16):
        y = olamd.matmul(_offset(a.to(dt)), _offset(b.to(dt)))
        assert torch.equal(y, exact.to(torch.float32).to(dt)), dt
    # fp8 weights under bf16 activations: codes that are small integers, power-of-two scales
    scale = torch.pow(2.0, -ints(0, 4, (N,)).float())
    w = b[0].to(torch.float8_e4m3fn)
    y = olamd.dequantize_linear_matmul(a[0].to(torch.bfloat16), w, scale if N > 1 else scale.reshape(()), None, 1,
                                       olamd.BFLOAT16)
    assert torch.equal(y, (exact[0] * scale.double()).to(torch.float32).to(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", [(9, 1, 64), (65, 63, 32), (130, 129, 320), (1100, 2101, 96), (65537, 17, 32)])
def test_b_transposed(olamd, dev, M, N, K):
    """The packed-weight product past the GEMVs: its decoded weight is [N, K]."""
    g = torch.Generator(device=dev).manual_seed(N)
    a = torch.randint(-2, 3, (M, K), generator=g, device=dev, dtype=torch.int32)
    q = torch.randint(-8, 9, (N * K // 32, 32), generator=g, device=dev, dtype=torch.int32)
    d = torch.full((N * K // 32, 1), 0.5, dtype=torch.float16, device=dev)
    x = torch.cat((d.view(torch.uint8).view(-1, 2), q.to(torch.int8).view(torch.uint8)), dim=1).reshape(-1)
    y = olamd.dequantize_packed_matmul(a.to(torch.float16), x, "gguf:q8_0", (N, K))
    exact = a.double() @ (q.double().view(N, K) * 0.5).t().contiguous()
    assert torch.equal(y, exact.to(torch.float32).to(torch.float16))


# The core's 128-row tiles: enough outputs for them, rows that end inside one,
# half a K step at the end.
@pytest.mark.parametrize("M,K,N", [(520, 192, 2064), (1100, 64, 1040), (385, 320, 2176)], ids=str)
def test_half_tiles(olamd, dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(M)
    ints = lambda lo, hi, sh: torch.randint(lo, hi, sh, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    for lo_a, dt_a, lo_b, dt_b in ((0, torch.uint8, -128, torch.int8), (-128, torch.int8, 0, torch.uint8)):
        a, b = ints(lo_a, lo_a + 256, (M, K)).to(dt_a), ints(lo_b, lo_b + 256, (K, N)).to(dt_b)
        za, zb = ints(lo_a, lo_a + 256, (M,)).to(dt_a), ints(lo_b, lo_b + 256, (N,)).to(dt_b)
        y = olamd.matmul_integer(a, b, za, zb)
        assert torch.equal(y.double(), (a.double() - za.double().unsqueeze(1)) @ (b.double() - zb.double()))
        assert torch.equal(olamd.matmul_integer(a, b).double(), a.double() @ b.double())
    a, b = ints(-2, 3, (M, K)), ints(-8, 9, (K, N))
    exact = a.double() @ b.double()
    for dt in (torch.float16, torch.bfloat16):
        assert torch.equal(olamd.matmul(a.to(dt), b.to(dt)), exact.to(torch.float32).to(dt))
    scale = torch.pow(2.0, -ints(0, 4, (N,)).float())
    w = b.to(torch.float32).to(torch.float8_e4m3fn)
    y = olamd.dequantize_linear_matmul(a.to(torch.bfloat16), w, scale, None, 1, olamd.BFLOAT16)
    assert torch.equal(y, (exact * scale.double()).to(torch.float32).to(torch.bfloat16))
    # grouped: 16-bit experts given [N, K], and fp8 experts [K, N]
    idx = ints(0, 2, (M, 1))
    e = torch.stack((b, -b)).to(torch.float32)
    want = torch.where(idx.unsqueeze(2) == 0, exact.unsqueeze(1), -exact.unsqueeze(1))
    y = olamd.grouped_matmul(a.to(torch.bfloat16), e.transpose(1, 2).contiguous().to(torch.bfloat16), idx, transB=1)
    assert torch.equal(y, want.to(torch.float32).to(torch.bfloat16))
    y = olamd.dequantize_linear_grouped_matmul(a.to(torch.bfloat16), e.to(torch.float8_e4m3fn),
                                               torch.ones((2, 1, N), device=dev), idx, cast_to=olamd.BFLOAT16)
    assert torch.equal(y, want.to(torch.float32).to(torch.bfloat16))


# Two wave groups per tile (long K, few outputs): K steps that do not split
# evenly, partial last steps, rows off 16 bytes.
@pytest.mark.parametrize("M,K,N", [(40, 3072, 64), (64, 3136, 130), (65, 4089, 96), (130, 1536, 72), (33, 3112, 257),
                                   (7, 1601, 100)], ids=str)
def test_two_groups(olamd, dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(M + K)
    ints = lambda lo, hi, sh: torch.randint(lo, hi, sh, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    a, b = ints(-2, 3, (M, K)), ints(-8, 9, (K, N))
    exact = a.double() @ b.double()
    for dt in (torch.float16, torch.bfloat16):
        assert torch.equal(olamd.matmul(a.to(dt), b.to(dt)), exact.to(torch.float32).to(dt)), dt
    scale = torch.pow(2.0, -ints(0, 4, (N,)).float())
    y = olamd.dequantize_linear_matmul(a.to(torch.bfloat16), b.float().to(torch.float8_e4m3fn), scale, None, 1,
                                       olamd.BFLOAT16)
    assert torch.equal(y, (exact * scale.double()).to(torch.float32).to(torch.bfloat16))


# 64 x 128 tiles: more small tiles than CUs, or more large ones; rows and columns
# that end inside one.
@pytest.mark.parametrize("M,K,N", [(65, 130, 8250), (330, 333, 3137), (1040, 65, 1023), (63, 2049, 16500),
                                   (300, 129, 11007)], ids=str)
def test_wide_tiles(olamd, dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(M + K)
    ints = lambda lo, hi, sh: torch.randint(lo, hi, sh, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    a, b = ints(0, 256, (M, K)).to(torch.uint8), ints(-128, 128, (K, N)).to(torch.int8)
    za, zb = ints(0, 256, (M,)).to(torch.uint8), ints(-128, 128, (N,)).to(torch.int8)
    assert torch.equal(olamd.matmul_integer(a, b).double(), a.double() @ b.double())
    y = olamd.matmul_integer(a, b, za, zb)
    assert torch.equal(y.double(), (a.double() - za.double().unsqueeze(1)) @ (b.double() - zb.double()))
    a, b = ints(-2, 3, (M, K)), ints(-8, 9, (K, N))
    for dt in (torch.float16, torch.bfloat16):
        assert torch.equal(olamd.matmul(a.to(dt), b.to(dt)), (a.double() @ b.double()).to(torch.float32).to(dt)), dt


# K = 0: nothing is read, sums are zero (rows of whole 16-byte pieces and others).
@pytest.mark.parametrize("M,N", [(3, 15), (8, 16), (1, 1), (70, 130), (600, 2053)], ids=str)
def test_empty_k(olamd, dev, M, N):
    empty = lambda *sh, dt: torch.empty(sh, dtype=dt, device=dev)  # noqa: E731
    a, b = empty(M, 0, dt=torch.uint8), empty(0, N, dt=torch.int8)
    za = torch.full((M,), 7, dtype=torch.uint8, device=dev) if M > 1 else None
    zb = torch.full((N,), -3, dtype=torch.int8, device=dev) if N > 1 else None
    assert not olamd.matmul_integer(a, b).any()
    assert not olamd.matmul_integer(a, b, za, zb).any()
    s = [np.array(v, np.float32) for v in (0.02, 0.004, 0.3)]
    for z in (0, 128):  # without and with column sums
        q = olamd.qlinear_matmul(a, s[0], np.array(z, np.uint8), b, s[1], np.array(3, np.int8), s[2], np.array(9, np.uint8))
        assert bool((q == 9).all())
    for dt in (torch.float16, torch.bfloat16):
        assert not olamd.matmul(empty(M, 0, dt=dt), empty(0, N, dt=dt)).any(), dt
    scale = torch.full((N,), 0.5, device=dev) if N > 1 else torch.tensor(0.5, device=dev)
    assert not olamd.dequantize_linear_matmul(empty(M, 0, dt=torch.float16), b, scale.half(), None, 1).any()
    assert not olamd.dequantize_linear_matmul(empty(M, 0, dt=torch.bfloat16), b.view(torch.float8_e4m3fn), scale, None,
                                              1, olamd.BFLOAT16).any()


# fp8 weights with an infinite scale, K no multiple of a step: the padding of the
# last step stays out of the sums.
@pytest.mark.parametrize("M,K,N", [(5, 100, 40), (130, 100, 130), (3, 77, 17), (1100, 33, 2101), (40, 3073, 65)], ids=str)
def test_fp8_infinite_scale(olamd, dev, M, K, N):
    a = torch.ones((M, K), dtype=torch.bfloat16, device=dev)
    w = torch.ones((K, N), device=dev).to(torch.float8_e4m3fn)
    scale = torch.ones(N, device=dev)
    scale[1] = float("inf")
    y = olamd.dequantize_linear_matmul(a, w, scale, None, 1, olamd.BFLOAT16)
    assert torch.equal(y, (scale * K).to(torch.bfloat16).expand(M, N))


# 16-bit groups in 128-row tiles (few pairs, or few tiles) and in 256-row ones, even
# and skewed.
@pytest.mark.parametrize("M,G,K,N", [(50, 8, 96, 2064), (100, 8, 64, 9008), (100, 8, 64, 6016), (300, 8, 64, 6016),
                                     (600, 3, 160, 1040)], ids=str)
def test_grouped_tile_heights(olamd, dev, M, G, K, N):
    g = torch.Generator(device=dev).manual_seed(M + N)
    ints = lambda lo, hi, sh: torch.randint(lo, hi, sh, generator=g, device=dev, dtype=torch.int32)  # noqa: E731
    a, w = ints(-2, 3, (M, K)), ints(-4, 5, (G, K, N))
    for idx in (ints(0, G, (M, 2)), (torch.rand((M, 2), generator=g, device=dev) ** 4 * G).int().clamp(0, G - 1)):
        every = torch.stack([a.double() @ w[e].double() for e in range(G)])  # [G, M, N]
        want = torch.stack([every[idx[:, s].long(), torch.arange(M, device=dev)] for s in range(2)], dim=1).float()
        for dt in (torch.float16, torch.bfloat16):
            y = olamd.grouped_matmul(a.to(dt), w.to(dt), idx, transB=0)
            assert torch.equal(y, want.to(dt)), dt
            y = olamd.grouped_matmul(a.to(dt), w.transpose(1, 2).contiguous().to(dt), idx, transB=1)
            assert torch.equal(y, want.to(dt)), dt


# A weight past 2^31 bytes, N odd: one-hot rows pick rows of it, its last among them.
@pytest.mark.parametrize("M", [8, 40])  # the decode GEMM, tiles
def test_weight_past_two_gib(olamd, dev, M):
    K, N = 32800, 65537
    b = torch.empty((K, N), dtype=torch.int8, device=dev)
    for k in range(0, K, 4100):
        b[k:k + 4100] = torch.randint(-128, 128, (4100, N), device=dev, dtype=torch.int8)
    at = torch.linspace(0, K - 1, M, device=dev).long()
    a = torch.zeros((M, K), dtype=torch.int8, device=dev)
    a[torch.arange(M, device=dev), at] = 3
    assert torch.equal(olamd.matmul_integer(a, b), b[at].int() * 3)
