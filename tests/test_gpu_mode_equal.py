"""Smoothing with the filter applied inside the pass along x equals the transform, the product and the inverse transform
called one after another, bit for bit, at lengths with every kind of radix stage (2, 3, 4, 5 and 8)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [12, 16, 20, 24, 40, 48, 80, 96, 128, 160, 192, 320, 384])
def test_fused_filter_equals_separate_passes(gpu, N):
    from pylians_amd import Pk_library, smoothing_library
    g = torch.Generator("cuda").manual_seed(N)
    f = torch.randn((N, N, N), device="cuda", generator=g)
    k = torch.randn((N, N, N // 2 + 1), device="cuda", dtype=torch.complex64, generator=g)
    c = Pk_library.FFT3Dr_f(f)
    ac, bd, ad, bc = c.real * k.real, c.imag * k.imag, c.real * k.imag, c.imag * k.real   # each rounded by itself
    s = Pk_library.IFFT3Dr_f(torch.complex(ac - bd, ad + bc))
    assert torch.equal(smoothing_library.field_smoothing(f, k), s)
