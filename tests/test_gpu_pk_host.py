"""Results in host memory, block by block: pyl_pk_particles_host fills an array of sentinels with what the device entry
points leave, with weights and a redshift-space shift as well.

Wave numbers and the NaN of empty bins: equal to 1e-13 and in place; Nmodes: equal; each power block: 1e-5 of its own largest
value (float64 deposit by atomics in another order, one rounding of the overdensity to float32)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

L = 70.0
SENTINEL = -7.25e300


def _blocks(N):
    """(name, slice) of the layout."""
    from pylians_amd.Pk_library import pk_layout
    kpar, kper, kmax, n = pk_layout(N)
    n2 = (kpar + 1) * (kper + 1)
    at, out = 0, []
    for name, size in (("k3D", kmax), ("P0", kmax), ("P2", kmax), ("P4", kmax), ("phase", kmax), ("Nmodes3D", kmax),
                       ("k1D", kpar), ("P1D", kpar), ("Nmodes1D", kpar), ("kpar", n2), ("kper", n2), ("P2D", n2), ("Nmodes2D", n2)):
        out.append((name, slice(at, at + size)))
        at += size
    assert at == n
    return out, n


@pytest.mark.parametrize("weights, rsd", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("flags_all", [True, False])
@pytest.mark.parametrize("N, axis", [(8, 0), (40, 2), (64, 1), (128, 2)])
def test_particles_host(gpu, N, axis, flags_all, weights, rsd):
    from pylians_amd import _lib
    lib = _lib.lib()
    blocks, n = _blocks(N)
    g = torch.Generator("cuda").manual_seed(N)
    pos = torch.rand((4000, 3), device="cuda", generator=g) * L
    vel = 200.0 * torch.randn((4000, 3), device="cuda", generator=g) if rsd else None
    W = torch.rand(4000, device="cuda", generator=g) + 0.5 if weights else None
    flags = (_lib.PK_ALL if flags_all else 0) | _lib.ATOMIC
    dev, host = torch.full((n,), SENTINEL, dtype=torch.float64, device="cuda"), np.full(n, SENTINEL)
    _lib.check(lib.pyl_pk_particles_host(_lib.ptr(pos), _lib.ptr(vel), _lib.ptr(W), 4000, N, L, 100.0, 0.5, 1, 2, axis,
                                         _lib.F32, flags, host.ctypes.data, _lib.stream()))
    if rsd:
        _lib.check(lib.pyl_pk_particles_rsd(_lib.ptr(pos), _lib.ptr(vel), _lib.ptr(W), 4000, N, L, 100.0, 0.5, 1, 2, axis,
                                            _lib.F32, flags, _lib.ptr(dev), _lib.stream()))
    else:
        _lib.check(lib.pyl_pk_particles(_lib.ptr(pos), _lib.ptr(W), 4000, N, L, 2, axis, _lib.F32, flags, _lib.ptr(dev),
                                        _lib.stream()))
    a = dev.cpu().numpy()
    assert np.array_equal(np.isnan(a), np.isnan(host))
    for name, s in blocks:
        x, y = np.nan_to_num(a[s]), np.nan_to_num(host[s])
        if name.startswith("Nmodes"):
            assert np.array_equal(x, y), name
        elif name.startswith("k"):
            assert np.allclose(x, y, rtol=1e-13, atol=0), name
        else:
            sel = slice(1, None) if name == "P2D" else slice(None)   # 2-D bin 0 holds the mean: rounding noise
            assert np.max(np.abs(x[sel] - y[sel])) <= 1e-5 * np.max(np.abs(x[sel])), name
