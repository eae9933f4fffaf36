"""The decode GEMM (csrc/skinny_gemm.hpp): one and two 16-row operands and the
row of ones behind them, 64- and 128-column tiles with partial ones, K that is
no multiple of a chunk and weights whose last lines end inside a load, fewer
chunks than waves.  Integers bit for bit; fp8 with small integers and
power-of-two scales, whose sums are exact in any order.  Grouped calls with
more pairs of one expert than a pass holds, idle experts and pairs outside the
groups."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev(olamd):
    olamd.init(0)
    return torch.device("cuda:0")


def _ints(g, lo, hi, shape, dtype=torch.int32):
    return torch.randint(lo, hi, shape, generator=g, device=g.device, dtype=torch.int32).to(dtype)


@pytest.mark.parametrize("M", [1, 15, 16, 17, 31])
@pytest.mark.parametrize("K,N", [(256, 64), (300, 65), (2048, 130), (2113, 1027), (257, 16500)], ids=str)
def test_int8(olamd, dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(M * K + N)
    for (alo, adt), (blo, bdt) in (((0, torch.uint8), (-128, torch.int8)), ((-128, torch.int8), (0, torch.uint8))):
        a, b = _ints(g, alo, alo + 256, (M, K), adt), _ints(g, blo, blo + 256, (K, N), bdt)
        af, bf = a.double(), b.double()
        assert torch.equal(olamd.matmul_integer(a, b).double(), af @ bf)
        za = _ints(g, alo, alo + 256, (M,), adt) if M > 1 else np.array(7, np.uint8 if alo == 0 else np.int8)
        zb = _ints(g, blo, blo + 256, (N,), bdt)
        fa = za.double().unsqueeze(1) if M > 1 else 7
        assert torch.equal(olamd.matmul_integer(a, b, za, zb).double(), (af - fa) @ (bf - zb.double()))
        s = [np.array(v, np.float32) for v in (0.02, 0.004, 0.3)]
        cs = float(np.float32(np.float32(s[0] * s[1]) / s[2]))
        for z in (128 if alo == 0 else 0, 5):  # with and without column sums
            az = np.array(z, np.uint8 if alo == 0 else np.int8)
            bz = np.array(0 if blo else 128, np.int8 if blo else np.uint8)
            y = olamd.qlinear_matmul(a, s[0], az, b, s[1], bz, s[2], np.array(3, np.int8))
            acc = (af - z) @ (bf - float(bz))
            want = (torch.round(acc.to(torch.float32) * cs) + 3).clamp(-128, 127).to(torch.int8)
            assert torch.equal(y, want)


def test_batched(olamd, dev):
    g = torch.Generator(device=dev).manual_seed(5)
    a, b = _ints(g, -128, 128, (3, 9, 320), torch.int8), _ints(g, -128, 128, (320, 200), torch.int8)
    assert torch.equal(olamd.matmul_integer(a, b).double(), torch.stack([x.double() @ b.double() for x in a]))


@pytest.mark.parametrize("M,K,N", [(1, 256, 64), (16, 288, 80), (17, 2048, 144), (32, 4096, 64), (5, 544, 16512)],
                         ids=str)
def test_fp8(olamd, dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(K + N)
    a, w = _ints(g, -2, 3, (M, K)), _ints(g, -8, 9, (K, N))
    scale = torch.pow(2.0, -_ints(g, 0, 4, (N,)).float())
    y = olamd.dequantize_linear_matmul(a.to(torch.bfloat16), w.float().to(torch.float8_e4m3fn), scale, None, 1,
                                       olamd.BFLOAT16)
    assert torch.equal(y, (a.double() @ w.double() * scale.double()).to(torch.float32).to(torch.bfloat16))


@pytest.mark.parametrize("M,G,K,N", [(1, 3, 64, 64), (40, 4, 288, 112), (64, 16, 256, 1040), (90, 3, 1024, 4112),
                                     (260, 200, 64, 80), (5, 4096, 32, 64)], ids=str)
def test_grouped(olamd, dev, M, G, K, N):
    g = torch.Generator(device=dev).manual_seed(M + N)
    a, w = _ints(g, -2, 3, (M, K)), _ints(g, -4, 5, (G, K, N))
    scale = torch.pow(2.0, -_ints(g, 0, 3, (G, 1, N)).float())
    bias = _ints(g, -8, 9, (G, N)).to(torch.bfloat16)
    idx = _ints(g, 0, max(1, G - 1), (M, 2), torch.int64)  # the last expert idle
    idx[: M // 2] = 0  # one expert with more pairs than a pass holds
    idx[M - 1, 1] = G  # outside the groups: a NaN row
    y = olamd.dequantize_linear_grouped_matmul(a.to(torch.bfloat16), w.float().to(torch.float8_e4m3fn), scale, idx,
                                               cast_to=olamd.BFLOAT16, bias=bias)
    for m in range(M):
        for s in range(2):
            e = int(idx[m, s])
            if e >= G:
                assert bool(torch.isnan(y[m, s]).all())
                continue
            r = (a[m].double() @ w[e].double() * scale[e, 0].double()).to(torch.float32).to(torch.bfloat16)
            assert torch.equal(y[m, s], (r.float() + bias[e].float()).to(torch.bfloat16)), (m, s)


def test_grouped_none_inside(olamd, dev):
    a = torch.ones((9, 64), dtype=torch.bfloat16, device=dev)
    w = torch.ones((5, 64, 144), device=dev).to(torch.float8_e4m3fn)
    for bad in (-1, 5):
        y = olamd.dequantize_linear_grouped_matmul(a, w, torch.ones((5, 1, 144), device=dev),
                                                   torch.full((9, 2), bad, device=dev), cast_to=olamd.BFLOAT16)
        assert bool(torch.isnan(y).all())
