"""The reduction of the binning pass's rows with the normalisation, at the grid sizes where its tiles have edges (fewer
3-D bins than a workgroup's 8, partial tiles of 2-D entries, fewer rows than the threads that share them), per line of
sight, with and without the 1-D and 2-D histograms, against the float64 oracle; single and batched.

Tolerance: modes are sums of squares in float64, so bins agree to 1e-12 of the largest; counts and k exactly or to 1e-13."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [8, 12, 20, 24, 40, 64, 96, 128]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("N", SIZES)
def test_bins(gpu, N, axis):
    from oracle import pk as P
    from pylians_amd import Pk_library
    f = np.random.default_rng(N).standard_normal((N, N, N))
    g, o = Pk_library.Pk(f, 150.0, axis=axis, MAS="TSC"), P.Pk(f, 150.0, axis=axis, MAS="TSC")
    for name in ("Nmodes3D", "Nmodes1D", "Nmodes2D"):
        assert np.array_equal(getattr(g, name), getattr(o, name)), name
    for name in ("k3D", "k1D", "kpar", "kper"):
        assert np.allclose(getattr(g, name), getattr(o, name), rtol=1e-13, atol=0), name
    for name in ("Pk", "Pk1D", "Pk2D"):
        a, b = getattr(g, name), getattr(o, name)
        assert np.array_equal(np.isnan(a), np.isnan(b))
        a, b = np.nan_to_num(a), np.nan_to_num(b)
        sel = slice(1, None) if name == "Pk2D" else slice(None)   # 2-D bin 0 holds the mean
        assert np.max(np.abs(a[sel] - b[sel])) <= 1e-12 * np.max(np.abs(b[sel])), name


@pytest.mark.parametrize("N", [12, 64])
def test_without_1d_and_2d(gpu, N):
    """Histograms that are left out report the geometry's counts and zero power; the 3-D bins are the same."""
    from pylians_amd import _lib
    from pylians_amd.Pk_library import pk_layout
    f = torch.from_numpy(np.random.default_rng(N).standard_normal((N, N, N))).cuda()
    kpar, kper, kmax, n = pk_layout(N)
    out = []
    for flags in (_lib.PK_ALL, 0):
        o = torch.zeros(n, dtype=torch.float64, device="cuda")
        _lib.check(_lib.lib().pyl_pk(_lib.ptr(f), N, 100.0, 0, 2, _lib.F64, flags, _lib.ptr(o), None, _lib.stream()))
        out.append(o.cpu().numpy())
    a, b = out
    s = kmax
    for i in (0, 1, 2, 3, 5):   # k3D, P0, P2, P4, Nmodes3D
        assert np.allclose(a[i * s:(i + 1) * s], b[i * s:(i + 1) * s], rtol=1e-12, atol=1e-12 * np.abs(a[s:2 * s]).max())
    p1 = 6 * s
    assert np.array_equal(a[p1:p1 + kpar], b[p1:p1 + kpar]) and not b[p1 + kpar:p1 + 2 * kpar].any()
    assert np.array_equal(a[p1 + 2 * kpar:p1 + 3 * kpar], b[p1 + 2 * kpar:p1 + 3 * kpar])
    n2, p2 = (kpar + 1) * (kper + 1), p1 + 3 * kpar
    assert np.array_equal(a[p2:p2 + 2 * n2], b[p2:p2 + 2 * n2])
    assert np.array_equal(a[p2 + 3 * n2:], b[p2 + 3 * n2:])
    assert not np.nan_to_num(b[p2 + 2 * n2:p2 + 3 * n2]).any()


def test_batched_sizes(gpu):
    """Jobs of several sizes and lines of sight share one reduction launch: each equals its own call."""
    from pylians_amd import batch, pipeline
    rng = np.random.default_rng(5)
    jobs = [{"pos": rng.random((4000, 3), dtype=np.float32) * 90, "BoxSize": 90.0, "dims": d, "axis": ax}
            for d, ax in ((16, 2), (64, 0), (96, 2), (32, 1), (64, 2), (16, 0))]
    b = batch.PkBatch(jobs)
    for _ in range(3):
        b.run()
        res = b.results()
        for r, j in zip(res, jobs):
            s = pipeline.PkParticles(j["pos"], 90.0, j["dims"], MAS="CIC", axis=j["axis"])
            assert np.array_equal(r.Nmodes2D, s.Nmodes2D)
            assert np.max(np.abs(r.Pk - s.Pk)) <= 1e-5 * np.max(np.abs(s.Pk))
    b.close()


@pytest.mark.parametrize("axis", [0, 2])
@pytest.mark.parametrize("N", [8, 40, 128])
def test_results_in_host_memory(gpu, N, axis):
    """pyl_pk_host and pyl_pk_particles_host fill the whole layout with what the device entry points leave in device
    memory; an asynchronous call is refused, and so is a null array."""
    from pylians_amd import _lib
    from pylians_amd.Pk_library import pk_layout
    L, n = _lib.lib(), pk_layout(N)[3]
    f = torch.from_numpy(np.random.default_rng(N).standard_normal((N, N, N)).astype(np.float32)).cuda()
    pos = torch.rand((500, 3), device="cuda", generator=torch.Generator("cuda").manual_seed(N)) * 70
    dev, host = torch.zeros(n, dtype=torch.float64, device="cuda"), np.full(n, -1.0)
    for flags in (_lib.PK_ALL, 0):
        _lib.check(L.pyl_pk(_lib.ptr(f), N, 70.0, axis, 2, _lib.F32, flags, _lib.ptr(dev), None, _lib.stream()))
        _lib.check(L.pyl_pk_host(_lib.ptr(f), N, 70.0, axis, 2, _lib.F32, flags, host.ctypes.data, None, _lib.stream()))
        a = dev.cpu().numpy()
        assert np.array_equal(np.isnan(a), np.isnan(host))
        ok = ~np.isnan(a)
        assert np.all(np.abs(a[ok] - host[ok]) <= 1e-12 * np.abs(a[ok]) + 1e-12)   # LDS sums in another order
    args = (_lib.ptr(pos), None, None, 500, N, 70.0, 0.0, 0.0, 0, 2, axis, _lib.F32)
    _lib.check(L.pyl_pk_particles_host(*args, _lib.PK_ALL | _lib.ATOMIC, host.ctypes.data, _lib.stream()))
    _lib.check(L.pyl_pk_particles(_lib.ptr(pos), None, 500, N, 70.0, 2, axis, _lib.F32, _lib.PK_ALL | _lib.ATOMIC,
                                  _lib.ptr(dev), _lib.stream()))
    a = dev.cpu().numpy()
    pw = np.nan_to_num(a - host)
    assert np.max(np.abs(pw)) <= 1e-5 * np.nanmax(np.abs(a))   # float64 deposit, one rounding to float32
    assert L.pyl_pk_particles_host(*args, _lib.PK_ASYNC, host.ctypes.data, _lib.stream()) != 0
    assert L.pyl_pk_host(_lib.ptr(f), N, 70.0, axis, 2, _lib.F32, _lib.PK_ALL, None, None, _lib.stream()) != 0
