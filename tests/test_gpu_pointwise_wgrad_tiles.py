"""Weight gradient of the 1x1 convolution around its 128 x 128 tiles: one tile and its neighbours, shares of one to some thirty chunks (from 24 on the larger tiles
take over), partial last chunks, samples that begin inside a share, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (batch, in, out, pixels): shares of 256 x 256 tiles hold max(4, chunks / 256) chunks of 64 pixels
CASES = [(1, 127, 128, 8), (1, 128, 128, 64), (2, 128, 127, 264), (3, 129, 128, 1000), (1, 128, 129, 4096), (2, 255, 256, 3048), (1, 257, 128, 9000), (1, 384, 128, 9000),
         (1, 200, 192, 32768), (1, 200, 192, 33800), (5, 256, 64, 2008), (1, 64, 8, 70000), (1, 200, 60, 420000), (1, 130, 100, 420000), (1, 60, 200, 300000), (1, 700, 130, 1200), (2, 40, 300, 504)]


@pytest.mark.parametrize("B,K,O,P", CASES)
@pytest.mark.parametrize("bias", [True, False])
def test_small_tiles(lib_built, B, K, O, P, bias):
    from makani_amd import pointwise as pw

    print(f"case wgrad tiles B={B} K={K} O={O} P={P} bias={bias}", flush=True)
    gen = torch.Generator().manual_seed(K + O)
    x = torch.randn(B, K, P // 8, 8, generator=gen).bfloat16()
    gy = torch.randn(B, O, P // 8, 8, generator=gen).bfloat16()
    xs, gs = x.double().reshape(B, K, P), gy.double().reshape(B, O, P)
    want, size = torch.zeros(O, K, dtype=torch.float64), torch.zeros(O, K, dtype=torch.float64)
    for b in range(B):
        want += gs[b] @ xs[b].T
        size += gs[b].abs() @ xs[b].abs().T
    gw, gb = pw.conv1x1_weight_grad(gy.cuda(), x.cuda(), bias)
    torch.cuda.synchronize()
    # exact products of bf16 values, fp32 sums of B P of them whose rounding errors grow like the root of the number of additions (B P / 16 in a
    # matrix instruction's chain, shares and wavefronts of the second kernel behind it); six standard deviations
    n = B * P
    bound = 6 * 2.0**-24 * (n / 16 + 64) ** 0.5 / n**0.5 * size + 2.0**-24 * size / n**0.5 * 64
    assert bool(((gw.cpu().double() - want).abs() <= bound).all()), float(((gw.cpu().double() - want).abs() / bound).max())
    if bias:
        assert bool(((gb.cpu().double() - gs.sum(dim=(0, 2))).abs() <= 1e-6 * gs.abs().sum(dim=(0, 2))).all())
