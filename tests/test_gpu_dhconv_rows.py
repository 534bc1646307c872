"""The channel mix over its row groups and chunks: one to four blocks of 32 rows in a group of 128 (groups of one or two blocks share the column tiles out to the
wavefronts), one to four chunks of 16 input channels with a last one that is not full, wide and narrow column blocks, rows that begin off a 16-byte
boundary, rows whose magnitude rises late and rows near the smallest numbers, against float64."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# (batch, in, out, degrees, orders): rows of a degree are min(l + 1, orders) * batch
CASES = [(1, 2, 2, 3, 3), (1, 16, 66, 35, 35), (1, 18, 64, 70, 70), (2, 32, 130, 33, 33), (1, 34, 128, 131, 131), (3, 48, 100, 44, 44), (5, 66, 30, 27, 20), (1, 64, 200, 65, 66)]


@pytest.mark.parametrize("B,I,O,L,M", CASES)
@pytest.mark.parametrize("shift", [0, 1])
def test_rows_and_chunks(lib_built, B, I, O, L, M, shift):
    from makani_amd._lib import check, lib
    from makani_amd.contractions import packed_for
    from makani_amd.sht import _stream_ptr

    print(f"case dhconv rows B={B} I={I} O={O} L={L} M={M} shift={shift}", flush=True)
    gen = torch.Generator().manual_seed(1000 * B + I)
    # channels that rise by 2^30 over the chunks in every third row: the scale of the row moves after partial sums exist
    rise = torch.exp2(torch.linspace(0, 30, I))
    x = torch.randn(M, L, B, I, 2, generator=gen)
    x[::3] *= rise[:, None]
    row_scale = torch.exp2(torch.randint(-60, 60, (M, L, 1, 1, 1), generator=gen).float())
    row_scale[1::7] = 2.0**-118                      # (rows whose scale would pass the largest power of two)
    x = x * row_scale
    w = torch.view_as_complex(torch.randn(I, O, L, 2, generator=gen)) / I**0.5
    ld_i, ld_o = int(lib.sfno_spectral_ld(B * I)), int(lib.sfno_spectral_ld(B * O))
    buf = torch.full((M * L * ld_i + 4,), float("nan"), device="cuda")[shift:shift + M * L * ld_i]
    buf.view(M, L, ld_i)[..., :2 * B * I] = x.reshape(M, L, -1).cuda()
    out = torch.full((M, L, ld_o), float("nan"), device="cuda")
    wd = w.cuda()
    check(lib.sfno_dhconv_spectral(packed_for(wd).handle, ctypes.c_void_p(buf.data_ptr()), ctypes.c_void_p(out.data_ptr()), B, M, 1, _stream_ptr(out.device)),
          "sfno_dhconv_spectral")
    torch.cuda.synchronize()
    got = torch.view_as_complex(out[..., :2 * B * O].reshape(M, L, B, O, 2).cpu().double())
    xd, wdd = torch.view_as_complex(x.double()), w.to(torch.complex128)
    # per product 2^-21 |x w| + 2^-38 max|x| max|w|, the row scale of a bound with up to four bits of headroom, and fp32 sums of 2 I terms; rows near the
    # smallest numbers keep 2^-151 in the row and round their results (about 2^-118) to 2^-149
    for l in range(L):
        m = min(l + 1, M)
        ref = torch.einsum("mbi,io->mbo", xd[:m, l], wdd[:, :, l])
        size = torch.einsum("mbi,io->mbo", xd[:m, l].abs(), wdd[:, :, l].abs())
        top = 2 * I * xd[:m, l].abs().amax(-1, keepdim=True) * wdd[:, :, l].abs().amax(0)
        bound = 2 * (2.0**-21 + 2 * I * 2.0**-24) * size + 2.0**-33 * top + 2.0**-140
        err = (got[:m, l] - ref).abs()
        assert bool((err <= bound).all()), (l, float((err / bound).max()))
    # orders past the degree are not written
    for l in range(min(L, M) - 1):
        assert bool(torch.isnan(out[l + 1:, l]).all())
