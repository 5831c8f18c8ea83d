"""The differentiable P0 with the spectrum saved by its forward pass: against the FP64 gradient over the schemes and
over grid sizes of every kind of radix stage, the one-call adjoint, repeated backward passes, saved-tensor hooks, and
forward passes that need no gradient.

Tolerance: relative L2 1e-5 of the FP64 gradient, as for the one-call adjoint (float32 grid and transforms)."""
import numpy as np
import pytest
import torch

from oracle import adjoint as A
from oracle.pk import MAS_correction, MAS_function, isqrt_array, mode_grid
from pylians_amd import synth

pytestmark = pytest.mark.gpu


def _case(N, seed=5):
    L = 2.0 * N
    pos = synth.zeldovich(32, L, seed=seed, rms_disp=2.0)
    nb = N // 3
    return pos, L, torch.tensor(np.random.default_rng(seed).random(nb), device="cuda"), nb


def _weights(d, scheme, N):
    """[(cell, weight)] of a float64 coordinate in cells, differentiable in d (the B-splines of orders 2 to 4)."""
    S = MAS_function(scheme)
    if S == 2:   # without |.|, whose derivative at a particle on a grid point is neither side's
        lo = torch.floor(d.detach())
        return [(lo.long() % N, 1.0 - (d - lo)), ((lo.long() + 1) % N, d - lo)]
    lo = torch.floor(d.detach() - 0.5 * S) + 1
    out = []
    for j in range(S):
        s = torch.abs(lo + j - d)
        if S == 3:
            w = torch.where(s < 0.5, 0.75 - s * s, 0.5 * torch.clamp(1.5 - s, min=0.0) ** 2)
        else:
            w = torch.where(s < 1.0, (4.0 - 6.0 * s * s + 3.0 * s ** 3) / 6.0, torch.clamp(2.0 - s, min=0.0) ** 3 / 6.0)
        out.append(((lo.long() + j) % N, w))
    return out


def _gradient(pos, N, L, w, scheme):
    """float64 gradient of sum_b w_b P0_b by automatic differentiation on the CPU."""
    p = torch.from_numpy(pos.astype(np.float64)).requires_grad_(True)
    ax = [_weights(p[:, a] * (N / L), scheme, N) for a in range(3)]
    rho = torch.zeros(N ** 3, dtype=torch.float64)
    for i0, w0 in ax[0]:
        for i1, w1 in ax[1]:
            for i2, w2 in ax[2]:
                rho = rho.index_add(0, (i0 * N + i1) * N + i2, w0 * w1 * w2)
    dk = torch.fft.rfftn(rho.reshape(N, N, N) * (N ** 3 / len(pos)) - 1.0)
    kx, ky, kz, ok = mode_grid(N)
    c = np.ones(dk.shape)
    for k in (kx, ky, kz):
        c = c * MAS_correction(np.pi / N * k, MAS_function(scheme))
    bins = torch.from_numpy(isqrt_array(np.broadcast_to(kx * kx + ky * ky + kz * kz, dk.shape)[ok]))
    power = (dk.real ** 2 + dk.imag ** 2)[torch.from_numpy(ok)] * torch.from_numpy(c[ok] ** 2)
    n = torch.bincount(bins).double()
    P0 = (torch.zeros_like(n).index_add(0, bins, power) / n * (L / N ** 2) ** 3)[1:1 + len(w)]
    g, = torch.autograd.grad((torch.from_numpy(w) * P0).sum(), p)
    return g.numpy()


@pytest.mark.parametrize("scheme", ["CIC", "TSC", "PCS"])
@pytest.mark.parametrize("N", [12, 20, 32, 40, 48, 80])
def test_gradient(gpu, N, scheme):
    from pylians_amd import autograd
    pos, L, w, nb = _case(N)
    x = torch.from_numpy(pos).cuda().requires_grad_(True)
    P0 = autograd.pk0(x, L, N, scheme, nbins=nb)
    g, = torch.autograd.grad((w * P0).sum(), x)
    one, P1 = autograd.grad_loss(x.detach(), L, N, w, scheme)
    ref = _gradient(pos, N, L, w.cpu().numpy(), scheme)
    if scheme == "CIC":
        o = A.grad(pos, N, L, w.cpu().numpy())
        assert np.linalg.norm(ref - o) <= 1e-10 * np.linalg.norm(o)
    for got in (g, one):
        assert np.linalg.norm(got.cpu().numpy() - ref) <= 1e-5 * np.linalg.norm(ref)
    assert torch.allclose(P0, P1, rtol=1e-9, atol=0)


def test_repeated_backward_and_hooks(gpu):
    from pylians_amd import autograd
    pos, L, w, nb = _case(48)
    x = torch.from_numpy(pos).cuda().requires_grad_(True)
    with torch.autograd.graph.save_on_cpu():
        a = autograd.pk0(x, L, 48, nbins=nb)
    b = autograd.pk0(x, L, 48, nbins=nb)
    ga, = torch.autograd.grad((w * a).sum(), x, retain_graph=True)
    gb, = torch.autograd.grad((w * b).sum(), x, retain_graph=True)
    gb2, = torch.autograd.grad((w * b).sum(), x)
    ga2, = torch.autograd.grad((2.0 * w * a).sum(), x)
    assert torch.equal(gb, gb2) and torch.allclose(ga, gb, rtol=1e-5, atol=0) and torch.allclose(ga2, 2.0 * ga, rtol=1e-5)


def test_no_gradient(gpu):
    from pylians_amd import autograd
    pos, L, w, nb = _case(32)
    x = torch.from_numpy(pos).cuda()
    p0 = autograd.pk0(x, L, 32, nbins=nb)
    with torch.no_grad():
        p1 = autograd.pk0(x.requires_grad_(True), L, 32, nbins=nb)
    assert not p0.requires_grad and not p1.requires_grad
    assert torch.allclose(p0, p1, rtol=1e-9, atol=0)
