"""Positions that are NaN or far outside the box, and weights that are not finite, leave the same cells through the sorts of
the ragged and 2-D deposits as through the direct kernel: the same cells NaN and infinite, and the others within the
direct kernel's float32 sums (1e-5 of the largest cell)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

L = 100.0
NAN, INF = float("nan"), float("inf")


def _grid(pos, W, dims, scheme, flags):
    from pylians_amd import _lib
    g = torch.zeros((dims,) * pos.shape[1], device="cuda")
    _lib.check(_lib.lib().pyl_mas_deposit(_lib.ptr(pos), _lib.ptr(W), pos.shape[0], pos.shape[1], dims, L, scheme, flags,
                                          _lib.ptr(g), _lib.stream()))
    return g.cpu().numpy()


@pytest.mark.parametrize("coords, weight", [({0: NAN}, None), ({0: NAN, 1: NAN}, None), ({0: 250.0, 1: -130.5}, None),
                                            ({0: 1e9, 1: -3e8}, None), ({}, INF), ({}, NAN)])
@pytest.mark.parametrize("scheme", [1, 2, 3, 4])
@pytest.mark.parametrize("axes, dims, n", [(3, 100, 2000003), (2, 300, 4000003)])
def test_same_cells(gpu, axes, dims, n, scheme, coords, weight):
    from pylians_amd import _lib
    g = torch.Generator("cuda").manual_seed(scheme)
    pos = torch.rand((n, axes), device="cuda", generator=g) * L
    W = torch.rand(n, device="cuda", generator=g) + 0.5
    for i in (1234, n - 1):
        for a, v in coords.items():
            pos[i, a] = v
        if weight is not None:
            W[i] = weight
    a, b = _grid(pos, W, dims, scheme, _lib.ATOMIC), _grid(pos, W, dims, scheme, 0)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isposinf(a), np.isposinf(b))
    ok = np.isfinite(a)
    assert np.max(np.abs(a[ok] - b[ok])) <= 1e-5 * np.max(np.abs(a[ok]))
