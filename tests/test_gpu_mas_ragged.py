"""Mass assignment onto grids whose edge is no multiple of the deposit's 16-cell tiles, against the
FP64 oracle.  The cell sums are float64 and rounded once to the grid type: half a float32 ulp (2^-24
relative) of the oracle's value, plus the float64 rounding of sums in another order (1e-13)."""
import numpy as np
import pytest

from oracle import cpu as C

pytestmark = pytest.mark.gpu

RTOL = 2.0 ** -24 + 1e-13


def _particles(n, dims, L, order, seed):
    """Unordered, or sorted by cell along x, y, z as in a snapshot; edge and corner positions included."""
    rng = np.random.default_rng(seed)
    pos = rng.random((n, 3), dtype=np.float32) * np.float32(L)
    h = L / dims
    edge = np.array([0.0, L, np.nextafter(np.float32(L), np.float32(0)), L - 0.5 * h, 0.5 * h, L - 1.5 * h], np.float32)
    pos[:216] = np.stack(np.meshgrid(edge, edge, edge, indexing="ij"), -1).reshape(-1, 3)
    if order == "sorted":
        c = np.floor(pos.astype(np.float64) / h).astype(np.int64)
        pos = pos[np.lexsort((c[:, 2], c[:, 1], c[:, 0]))]
    return np.ascontiguousarray(pos)


@pytest.mark.parametrize("order", ["unordered", "sorted"])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("scheme", ["NGP", "CIC", "TSC", "PCS"])
@pytest.mark.parametrize("dims", [33, 47, 49, 63, 65, 100])
def test_ragged_grid(gpu, dims, scheme, weighted, order):
    from pylians_amd import MAS_library
    L, n = 310.0, 2400001 if scheme == "NGP" else 900001
    pos = _particles(n, dims, L, order, dims)
    W = np.random.default_rng(3).random(n, dtype=np.float32) + np.float32(0.25) if weighted else None
    start = np.random.default_rng(4).random((dims,) * 3).astype(np.float32)
    g = start.copy()
    MAS_library.MA(pos, g, L, scheme, W=W)
    o = start.astype(np.float64) + C.deposit_f64(pos, dims, L, scheme, W)
    assert np.all(np.abs(g - o) <= RTOL * np.abs(o))


@pytest.mark.parametrize("dims", [64, 97])
@pytest.mark.parametrize("scheme", ["CIC", "PCS"])
def test_many_particles_in_and_out_of_order(gpu, dims, scheme):
    """More particles than the device's look at their order needs, clustered so that buckets overflow;
    the float64 grid too."""
    from pylians_amd import MAS_library
    L, n = 100.0, (1 << 20) + 4099
    rng = np.random.default_rng(11)
    pos = rng.random((n, 3), dtype=np.float32) * np.float32(L)
    pos[: n // 2] = np.mod(30.0 + 4.0 * rng.standard_normal((n // 2, 3)), L).astype(np.float32)
    pos = np.ascontiguousarray(rng.permutation(pos))
    order = np.lexsort(tuple(np.floor(pos[:, a] * (dims / L)).astype(np.int64) for a in (2, 1, 0)))
    o = C.deposit_f64(pos, dims, L, scheme)
    for p in (pos, np.ascontiguousarray(pos[order])):
        g = np.zeros((dims,) * 3, np.float32)
        MAS_library.MA(p, g, L, scheme)
        assert np.all(np.abs(g - o) <= RTOL * np.abs(o))
    if scheme == "CIC":
        W = rng.random(n, dtype=np.float32)
        gd = np.zeros((dims,) * 3, np.float64)
        MAS_library.CICW_d(pos, gd, L, W)
        od = C.deposit_f64(pos, dims, L, scheme, W)
        assert np.allclose(gd, od, rtol=1e-12, atol=1e-12)
