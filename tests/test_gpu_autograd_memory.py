"""The differentiable P0 where its kept spectra do not fit, or are not wanted: the backward pass computes the forward
pass again.  Gradients of the two ways agree to 1e-6 of their largest entry (the same kernels on the same float32 grid;
deposits differ in the order of float64 sums, so a cell may round to its neighbour)."""
import os
import subprocess
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("MAS, dims", [("CIC", 64), ("PCS", 40)])
def test_without_the_spectrum(gpu, MAS, dims):
    from pylians_amd import autograd
    x = (torch.rand((50000, 3), device="cuda", generator=torch.Generator("cuda").manual_seed(1)) * 100.0).requires_grad_(True)
    w = torch.rand(16, device="cuda", dtype=torch.float64, generator=torch.Generator("cuda").manual_seed(2))
    grads = {}
    for keep in (True, False, None):
        held = torch.cuda.memory_allocated()
        P0 = autograd.pk0(x, 100.0, dims, MAS, nbins=16, keep_spectrum=keep)
        held = torch.cuda.memory_allocated() - held
        assert (held >= 8 * dims * dims * (dims // 2 + 1)) == (keep is not False)
        grads[keep], = torch.autograd.grad((w * P0).sum(), x)
    top = grads[True].abs().max()
    for keep in (False, None):
        assert (grads[keep] - grads[True]).abs().max() <= 1e-6 * top


CHILD = """
import ctypes, sys, torch
sys.path.insert(0, %r)
from pylians_amd import autograd, _lib
x = (torch.rand((20000, 3), device="cuda") * 100.0).requires_grad_(True)
w = torch.ones(16, device="cuda", dtype=torch.float64)
def grad(many):
    g, = torch.autograd.grad(sum((w * autograd.pk0(x, 100.0, 128, nbins=16)).sum() for _ in range(many)), x)
    return g
one = grad(1)
torch.cuda.synchronize()
torch.cuda.empty_cache()
hold = torch.empty(torch.cuda.mem_get_info()[0] - (8 << 30), dtype=torch.uint8, device="cuda")
for mib in (256, 64, 16, 4, 2):   # the free memory that is reported grows at first
    while torch.cuda.mem_get_info()[0] >= (128 + mib) << 20:
        p = ctypes.c_void_p()
        _lib.check(_lib.lib().pyl_dev_alloc(ctypes.byref(p), mib << 20))
many = grad(40)
assert float((many - 40.0 * one).abs().max()) <= 1e-4 * float(many.abs().max())
print("equal")
"""


def test_many_forward_passes(gpu):
    """Forty passes of 8.5 MB of spectrum each before the first backward pass, with 128 MiB free."""
    out = subprocess.run([sys.executable, "-c", CHILD % ROOT], timeout=110, capture_output=True, text=True)
    assert out.returncode == 0 and "equal" in out.stdout, out.stderr[-2000:]
