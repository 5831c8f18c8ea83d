"""The device's look at the order of the particles of a deposit: which inputs it groups, and the grids either way.

Tolerance: float64 cell sums, one rounding to float32 (2^-24 relative), plus 1e-13 for sums in another order."""
import numpy as np
import pytest
import torch

from oracle import cpu as C

pytestmark = pytest.mark.gpu

L = 1000.0
RTOL = 2.0 ** -24 + 1e-13


def _lattice(m, seed=1):
    x = (torch.arange(m, device="cuda") + 0.5) * (L / m)
    p = torch.stack(torch.meshgrid(x, x, x, indexing="ij"), -1).reshape(-1, 3)
    g = torch.Generator("cuda").manual_seed(seed)
    return torch.remainder(p + 5.0 * torch.randn(p.shape, device="cuda", generator=g), L).contiguous()


def _unordered(n, seed=2):
    return torch.rand((n, 3), device="cuda", generator=torch.Generator("cuda").manual_seed(seed)) * L


def _in_cell_order(pos, dims):
    c = (pos * (dims / L)).long()
    return pos[torch.argsort((c[:, 0] * dims + c[:, 1]) * dims + c[:, 2])].contiguous()


def _presort_us(pos, dims, calls=20):
    """Least time of the deposit's look and grouping over some calls; None where it does not look."""
    from pylians_amd import MAS_library, _lib
    g, t = torch.zeros((dims,) * 3, device="cuda"), []
    try:
        for _ in range(calls):
            _lib.profile(True)
            MAS_library.MA(pos, g, L, "CIC")
            torch.cuda.synchronize()
            t.append(_lib.profile_read().get("deposit_presort", (0, None))[1])
    finally:
        _lib.profile(False)
    return None if t[0] is None else min(t) * 1e3


@pytest.mark.parametrize("dims", [128, 256, 512])
@pytest.mark.parametrize("order", ["sparse lattice", "2^21 lattice", "sparse, in cell order"])
def test_ordered_particles_are_not_grouped(gpu, order, dims):
    """Counting and copying would take as long as for unordered particles (25 us and more against some 5)."""
    pos = {"sparse lattice": lambda: _lattice(102), "2^21 lattice": lambda: _lattice(128),
           "sparse, in cell order": lambda: _in_cell_order(_unordered(1 << 20), dims)}[order]()
    assert _presort_us(pos, dims) <= 0.6 * _presort_us(_unordered(len(pos)), dims)


@pytest.mark.parametrize("dims", [32, 33, 48])
def test_few_tiles_are_not_looked_at(gpu, dims):
    """A step of unordered particles has few keys there already."""
    assert _presort_us(_unordered(1 << 20), dims) is None


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("dims, n", [(64, (1 << 20) + 1), (80, 1200007), (113, 1200007), (400, 2300003), (512, 1100003)])
def test_groups(gpu, dims, n, weighted):
    """16, 25, 64, 313 and 512 groups of unordered particles."""
    from pylians_amd import MAS_library
    pos = _unordered(n, dims)
    W = torch.rand(n, device="cuda", generator=torch.Generator("cuda").manual_seed(3)) + 0.25 if weighted else None
    o = C.deposit_f64(pos.cpu().numpy(), dims, L, "CIC", None if W is None else W.cpu().numpy())
    g = torch.zeros((dims,) * 3, device="cuda")
    MAS_library.MA(pos, g, L, "CIC", W=W)
    assert np.all(np.abs(g.cpu().numpy() - o) <= RTOL * np.abs(o))


def _stages(axes, dims, scheme, n):
    from pylians_amd import MAS_library, _lib
    pos = torch.rand((n, axes), device="cuda", generator=torch.Generator("cuda").manual_seed(1)) * L
    g = torch.zeros((dims,) * axes, device="cuda")
    try:
        _lib.profile(True)
        MAS_library.MA(pos, g, L, scheme)
        torch.cuda.synchronize()
        return set(_lib.profile_read())
    finally:
        _lib.profile(False)


@pytest.mark.parametrize("axes, dims, scheme, n", [(2, 1000, "CIC", 255000), (2, 250, "PCS", 40000), (2, 500, "NGP", 945000),
                                                   (3, 33, "PCS", 19000), (3, 40, "CIC", 115000), (3, 399, "PCS", 96600)])
def test_direct_kernel_below_the_line(gpu, axes, dims, scheme, n):
    """Ordered particles so few are quicker there; whether they are ordered the host cannot tell."""
    assert "deposit_atomic" in _stages(axes, dims, scheme, n)


@pytest.mark.parametrize("axes, dims, scheme, n", [(2, 1000, "CIC", 330000), (2, 500, "NGP", 2100000), (3, 33, "PCS", 53000),
                                                   (3, 100, "CIC", 131072), (3, 399, "PCS", 113600)])
def test_without_global_atomics_above_it(gpu, axes, dims, scheme, n):
    assert ("deposit_map" if axes == 2 else "deposit_tiles") in _stages(axes, dims, scheme, n)
