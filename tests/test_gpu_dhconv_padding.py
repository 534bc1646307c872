"""The channel mix clears the row slots behind the last sample's channels wherever it writes the row, and nothing else: one to fifteen channels short of a whole
row, the tile they end in narrow, wide or shared among the wavefronts, odd channel counts (another kernel) and bf16 compute."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# (batch, in, out, degrees, orders)
CASES = [(1, 8, 1, 5, 5), (1, 16, 138, 70, 70), (1, 16, 31, 33, 20), (3, 16, 31, 40, 44), (2, 16, 104, 30, 30), (3, 16, 17, 9, 9), (5, 16, 65, 12, 12), (1, 16, 64, 6, 6)]


@pytest.mark.parametrize("B,I,O,L,M,compute", [(*c, k) for c in CASES for k in ("fp32", "bf16")] + [(2, 7, 5, 20, 20, "fp32")])
@pytest.mark.parametrize("triangular", [True, False])
def test_padding_is_cleared(lib_built, B, I, O, L, M, triangular, compute):
    from makani_amd._lib import check, lib
    from makani_amd.contractions import packed_for
    from makani_amd.sht import _stream_ptr

    print(f"case dhconv padding B={B} I={I} O={O} L={L} M={M} triangular={triangular} {compute}", flush=True)
    gen = torch.Generator().manual_seed(B * 1000 + O)
    w = torch.view_as_complex(torch.randn(I, O, L, 2, generator=gen)).cuda()
    ld_i, ld_o = int(lib.sfno_spectral_ld(B * I)), int(lib.sfno_spectral_ld(B * O))
    x = torch.zeros(M, L, ld_i)
    x[..., :2 * B * I] = torch.randn(M, L, 2 * B * I, generator=gen)
    x = x.cuda()
    out = torch.full((M * L * ld_o + 64,), float("nan"), device="cuda")
    check(lib.sfno_dhconv_spectral(packed_for(w, compute).handle, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(out.data_ptr()), B, M, int(triangular),
                                   _stream_ptr(out.device)), "sfno_dhconv_spectral")
    torch.cuda.synchronize()
    assert bool(torch.isnan(out[-64:]).all())
    got = out[:-64].view(M, L, ld_o).cpu()
    ref = torch.einsum("mlbi,iol->mlbo", torch.view_as_complex(x[..., :2 * B * I].reshape(M, L, B, I, 2).cpu().double()), w.cpu().to(torch.complex128))
    for l in range(L):
        m = min(l + 1, M) if triangular else M
        assert bool((got[:m, l, 2 * B * O:] == 0).all()), l
        # (the value check is a coarse one, for rows that a misplaced zero would hit; no sum here comes near zero by more than its terms)
        val = torch.view_as_complex(got[:m, l, :2 * B * O].reshape(m, B, O, 2).double())
        assert float((val - ref[:m, l]).abs().max()) <= 2.0**-7 * float(ref[:m, l].abs().max()) * I**0.5, l
        if triangular:
            assert bool(torch.isnan(got[m:, l, :2 * B * O]).all()), l
