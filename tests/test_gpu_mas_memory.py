"""Mass assignment where the device memory is nearly gone: what the routes with workspaces cannot have, the plainer
routes do without.  Each case runs in a process of its own, which takes all but some of the card's memory first.  NGP counts below 2^24 are whole
numbers in float32, so the grids are equal to the counts."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import ctypes, sys, torch
sys.path.insert(0, %r)
from pylians_amd import MAS_library, _lib
axes, dims, n, left = (int(x) for x in sys.argv[1:])
L = 100.0
pos = torch.rand((n, axes), device="cuda", generator=torch.Generator("cuda").manual_seed(1)) * L
c = torch.floor(pos.double() * (dims / L) + 0.5).long() %% dims
key = c[:, 0]
for a in range(1, axes):
    key = key * dims + c[:, a]
ref = torch.bincount(key, minlength=dims ** axes).float().reshape((dims,) * axes)
del c, key
grid = torch.zeros((dims,) * axes, device="cuda")
_lib.check(_lib.lib().pyl_mas_deposit(_lib.ptr(pos), None, 1, axes, dims, L, 1, _lib.ATOMIC, _lib.ptr(grid), _lib.stream()))
grid.zero_()
torch.cuda.synchronize()
torch.cuda.empty_cache()
hold = torch.empty(torch.cuda.mem_get_info()[0] - (8 << 30), dtype=torch.uint8, device="cuda")
for mib in (256, 64, 16, 4, 2):   # the free memory that is reported grows at first
    while torch.cuda.mem_get_info()[0] >= (left + mib) << 20:
        p = ctypes.c_void_p()
        _lib.check(_lib.lib().pyl_dev_alloc(ctypes.byref(p), mib << 20))
assert abs(torch.cuda.mem_get_info()[0] / 2.0 ** 20 - left) <= 3
MAS_library.NGP(pos, grid, L) if axes == 3 else MAS_library.NGPc2D(pos, grid, L, 1)
torch.cuda.synchronize()
assert torch.equal(grid, ref)
print("equal")
"""


# 2^24 particles: 256^3 needs 890 MiB of buckets, and 200 more for the grouped copy; the ragged grid and the map need
# hundreds and have 64
@pytest.mark.parametrize("axes, dims, left", [(3, 256, 1000), (3, 250, 64), (2, 1000, 64)])
def test_little_memory(gpu, axes, dims, left):
    out = subprocess.run([sys.executable, "-c", CHILD % ROOT, str(axes), str(dims), str(1 << 24), str(left)], timeout=110,
                         capture_output=True, text=True)
    assert out.returncode == 0 and "equal" in out.stdout, out.stderr[-2000:]
