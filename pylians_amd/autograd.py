"""Differentiable P0(k) of a particle set: a torch.autograd.Function around the hand-written
adjoint (pyl_pk_adjoint).  Builder-defined; the reference has no gradients.

    P0 = pk0(pos, BoxSize, dims, MAS="CIC", nbins=64)     # (nbins,) float64, differentiable
    loss = (w * P0).sum(); loss.backward()                 # pos.grad: (n, 3) float32

Forward: fused deposit -> delta = rho/rhobar - 1 -> r2c -> window deconvolution -> binning
(float32 grid and FFT, float64 shell sums); when a gradient is asked for, the corrected half spectrum
is saved for the backward pass (complex64, dims x dims x (dims/2 + 1): 0.54 GB at 512^3), or, where memory is short or
the caller says so, the positions alone: the backward pass then computes the forward pass a second time (256^3: 0.77 ms
for both passes with the spectrum, 1.17 without).  Backward: the gradient spectrum
H_k = (dL/dP0_b) (L/N^2)^3 / Nmodes_b c_k^2 delta_k, an unnormalised c2r and the stencil-derivative
gather at the particles.
"""
import torch

from . import _lib
from .Pk_library import pk_layout


def _kmax(dims):
    return pk_layout(dims)[2]


class _P0(torch.autograd.Function):
    @staticmethod
    def forward(ctx, pos, BoxSize, dims, scheme, nbins, needs_grad, keep):
        p = pos.detach().to(torch.float32).contiguous()
        _, _, kmax, nout = pk_layout(dims)
        out = torch.empty(nout, dtype=torch.float64, device=p.device)
        spec = _spectrum(dims, p.device, keep) if needs_grad else None
        if spec is not None:
            _lib.check(_lib.lib().pyl_pk_forward_keep(_lib.ptr(p), int(p.shape[0]), int(dims), float(BoxSize),
                                                      int(scheme), _lib.ptr(spec), _lib.ptr(out), _lib.stream()))
            ctx.save_for_backward(p, spec)
        else:
            _lib.check(_lib.lib().pyl_pk_particles(_lib.ptr(p), None, int(p.shape[0]), int(dims), float(BoxSize),
                                                   int(scheme), 0, _lib.F32, 0, _lib.ptr(out), _lib.stream()))
            ctx.save_for_backward(p)
        ctx.cfg = (float(BoxSize), int(dims), int(scheme), int(nbins))
        return out[kmax:kmax + nbins].clone()

    @staticmethod
    def backward(ctx, gP0):
        p, *spec = ctx.saved_tensors
        BoxSize, dims, scheme, nbins = ctx.cfg
        w = gP0.detach().to(torch.float64).contiguous()
        grad = torch.empty_like(p)
        if spec:
            _lib.check(_lib.lib().pyl_pk_adjoint_keep(_lib.ptr(p), int(p.shape[0]), dims, BoxSize, scheme, _lib.ptr(w),
                                                      nbins, _lib.ptr(spec[0]), _lib.ptr(grad), _lib.stream()))
        else:
            out = torch.empty(pk_layout(dims)[3], dtype=torch.float64, device=p.device)
            _lib.check(_lib.lib().pyl_pk_adjoint(_lib.ptr(p), int(p.shape[0]), dims, BoxSize, scheme, _lib.ptr(w),
                                                 nbins, _lib.ptr(grad), _lib.ptr(out), _lib.stream()))
        return grad, None, None, None, None, None, None


def _spectrum(dims, device, keep):
    """The buffer of a kept spectrum, or None: the caller wants none, or (keep=None) it would take more than an eighth of
    the memory that is free, so that the spectra of many forward passes never take the room of what follows."""
    shape = (dims, dims, dims // 2 + 1)
    if keep is False or (keep is None and 64 * shape[0] * shape[1] * shape[2] > torch.cuda.mem_get_info(device)[0]):
        return None
    return torch.empty(shape, dtype=torch.complex64, device=device)


def pk0(pos, BoxSize, dims, MAS="CIC", nbins=None, keep_spectrum=None):
    """Monopole P0 of the first `nbins` bins (|k| in [b+1, b+2) kF), differentiable w.r.t. pos.

    keep_spectrum: whether the spectrum is saved for the backward pass (else computed again there); None: while it is no
    more than an eighth of the free memory."""
    _lib.require_gpu()
    if MAS not in _lib.SCHEMES:
        raise ValueError("unknown MAS %r" % (MAS,))
    kmax = _kmax(dims)
    nbins = kmax if nbins is None else int(nbins)
    if not 0 < nbins <= kmax:
        raise ValueError("nbins must be in [1, %d]" % kmax)
    if not (isinstance(pos, torch.Tensor) and pos.is_cuda and pos.ndim == 2 and pos.shape[1] == 3):
        raise ValueError("pos must be a (n, 3) tensor on the GPU")
    needs_grad = torch.is_grad_enabled() and pos.requires_grad
    return _P0.apply(pos, BoxSize, int(dims), _lib.SCHEMES[MAS], nbins, needs_grad, keep_spectrum)


def grad_loss(pos, BoxSize, dims, w, MAS="CIC"):
    """dL/dpos for L = sum_b w_b P0_b without autograd bookkeeping; returns (grad, P0[:len(w)])."""
    p = _lib.to_dev(pos, torch.float32)
    wt = _lib.to_dev(w, torch.float64)
    _, _, kmax, nout = pk_layout(dims)
    grad = torch.empty_like(p)
    out = torch.empty(nout, dtype=torch.float64, device=p.device)
    _lib.check(_lib.lib().pyl_pk_adjoint(_lib.ptr(p), int(p.shape[0]), int(dims), float(BoxSize),
                                         _lib.SCHEMES[MAS], _lib.ptr(wt), int(wt.numel()), _lib.ptr(grad),
                                         _lib.ptr(out), _lib.stream()))
    return grad, out[kmax:kmax + int(wt.numel())]
