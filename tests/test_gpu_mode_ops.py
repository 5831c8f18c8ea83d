"""Field operations made inside the transform's pass along x (smoothing filter, window, |W delta_k|^2), at the
transform lengths where the pass can go wrong (one radix stage; radices 3 and 5; a partial last block of columns;
no prefetch past 512 points), against the float64 oracle.

Tolerance: a float32 transform is within 2e-6 log2 N of its largest output (the bound of the r2c tests); two of them
and one rounded product leave a field within 4e-6 log2 N + 1e-6 of its largest value; float64: 1e-12."""
import numpy as np
import pytest
import torch

from oracle import fields as F

pytestmark = pytest.mark.gpu


def _field(N, dtype):
    rng = np.random.default_rng(N)
    return (rng.standard_normal((N, N, N)) + 0.5).astype(dtype)


def _close(g, o, N, dtype):
    tol = 4e-6 * np.log2(N) + 1e-6 if dtype == np.float32 else 1e-12
    assert np.max(np.abs(np.asarray(g, np.float64) - o)) <= tol * np.max(np.abs(o))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("N", [8, 12, 16, 20, 40, 48, 80, 96, 160])
def test_window_and_power(gpu, N, dtype):
    from pylians_amd import Pk_library
    f = _field(N, dtype)
    _close(Pk_library.correct_MAS(f, 100.0, MAS="TSC"), F.correct_MAS(f, 100.0, "TSC"), N, dtype)
    x, o = Pk_library.Xi(f, 100.0, MAS="CIC", axis=1), F.Xi(f, 100.0, "CIC", axis=1)
    assert np.array_equal(x.Nmodes3D, o.Nmodes3D)
    _close(x.xi, o.xi, N, dtype)


@pytest.mark.parametrize("N", [8, 12, 16, 20, 40, 48, 80, 96, 160])
def test_filter(gpu, N):
    from pylians_amd import smoothing_library
    f = _field(N, np.float32)
    k = smoothing_library.FT_filter(100.0, 9.0, N, "Top-Hat")
    _close(smoothing_library.field_smoothing(f, k), F.field_smoothing(f, k.astype(np.complex128)), N, np.float32)


@pytest.mark.parametrize("N", [640, 768])
def test_large_lengths(gpu, N):
    """Plane waves along each axis come back times their filter value (no full-size oracle needed)."""
    from pylians_amd import smoothing_library
    x = torch.arange(N, device="cuda", dtype=torch.float64) * (2.0 * np.pi / N)
    f = (torch.cos(3 * x)[:, None, None] + torch.cos(5 * x)[None, :, None] + torch.cos(7 * x)[None, None, :]).float()
    k = torch.zeros((N, N, N // 2 + 1), device="cuda", dtype=torch.complex64)
    k[3, 0, 0] = k[N - 3, 0, 0] = 0.5
    k[0, 5, 0] = k[0, N - 5, 0] = 2.0
    k[0, 0, 7] = -1.0
    g = smoothing_library.field_smoothing(f, k)
    o = 0.5 * torch.cos(3 * x)[:, None, None] + 2.0 * torch.cos(5 * x)[None, :, None] - torch.cos(7 * x)[None, None, :]
    assert float((g.double() - o).abs().max()) <= (4e-6 * np.log2(N) + 1e-6) * 3.5
