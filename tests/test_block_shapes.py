"""Which parameter shapes the native block takes (no device needed)."""
import pytest
import torch


def params(c_in=6, embed=4, hidden=8, lmax=5):
    shapes = [(c_in, embed, lmax), (embed, c_in, 1, 1), (hidden, embed, 1, 1), (hidden,), (embed, hidden, 1, 1)] + 5 * [(embed,)]
    return [torch.empty(s, device="meta") for s in shapes]


def test_matching_and_absent_parameters():
    from makani_amd.block import shapes_fit

    assert shapes_fit(params(), 6, 4, 5)
    p = params()
    for i in (3, 5, 6, 7, 8, 9):
        p[i] = None
    assert shapes_fit(p, 6, 4, 5)
    assert not shapes_fit(params(), 7, 4, 5) and not shapes_fit(params(), 6, 5, 5) and not shapes_fit(params(), 6, 4, 6)


@pytest.mark.parametrize("which", [i for i in range(10) if i != 2])
def test_one_parameter_of_another_size(which):
    from makani_amd.block import shapes_fit

    p = params()
    p[which] = torch.empty((p[which].shape[0] + 1, *p[which].shape[1:]), device="meta")
    assert not shapes_fit(p, 6, 4, 5)
