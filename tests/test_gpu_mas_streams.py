"""2-D and ragged 3-D mass assignment on several streams and threads at once: every call's grid equals the oracle's.

Tolerance as in test_gpu_mas_map.py and test_gpu_mas_ragged.py: float64 cell sums, one rounding to the grid type (2^-24
relative), plus 1e-13 for sums in another order."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from oracle import cpu as C
from oracle import mas as M

pytestmark = pytest.mark.gpu

L = 200.0
RTOL = 2.0 ** -24 + 1e-13
PER_THREAD = 2   # hipStreamPerThread


def _case(axes, seed):
    """(device positions, edge, float64 grid): enough particles for the routes without global atomics."""
    rng = np.random.default_rng(seed)
    dims, n = (300, 600001) if axes == 2 else (61, 400001)
    pos = rng.random((n + 1000 * seed, axes), dtype=np.float32) * np.float32(L)
    if axes == 2:
        o = M.MAS_c(pos, np.zeros((dims, dims)), L, "CIC")
    else:
        o = C.deposit_f64(pos, dims, L, "CIC")
    return torch.from_numpy(pos).cuda(), dims, o


def _deposit(case, grid, stream):
    from pylians_amd import _lib
    pos, dims, _ = case
    return _lib.lib().pyl_mas_deposit(_lib.ptr(pos), None, pos.shape[0], pos.shape[1], dims, L, 2, _lib.ZERO,
                                      _lib.ptr(grid), ctypes.c_void_p(stream))


def _equal(grid, case):
    o = case[2]
    assert np.all(np.abs(grid.cpu().numpy() - o) <= RTOL * np.abs(o))


def _grids(cases):
    g = [torch.full((c[1],) * c[0].shape[1], 7.0, device="cuda") for c in cases]
    torch.cuda.synchronize()
    return g


def _runtime():
    """The HIP runtime of this process (there may be another on the disk)."""
    paths = {line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line}
    assert len(paths) == 1
    return ctypes.CDLL(paths.pop())


@pytest.mark.parametrize("axes", [2, 3])
def test_threads_with_the_per_thread_stream(gpu, axes):
    """The handle hipStreamPerThread is one value and a queue of its own in every thread."""
    from pylians_amd import _lib
    cases = [_case(axes, s) for s in range(3)]
    grids = [_grids(cases) for _ in range(8)]
    rcs, start = [], threading.Barrier(len(cases))

    def work(i):
        start.wait()
        rcs.extend(_deposit(cases[i], g[i], PER_THREAD) for g in grids)
        rcs.append(_lib.lib().pyl_stream_sync(ctypes.c_void_p(PER_THREAD)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not any(rcs)
    for g in grids:
        for i, c in enumerate(cases):
            _equal(g[i], c)


@pytest.mark.parametrize("streams", [2, 5])
def test_streams_in_turn(gpu, streams):
    """Calls of both routes go round the streams without a wait between them."""
    cases = [_case(2, 1), _case(3, 2)]
    st = [torch.cuda.Stream() for _ in range(streams)]
    grids = [_grids(cases) for _ in range(3 * streams)]
    for i, g in enumerate(grids):
        for j, c in enumerate(cases):
            assert _deposit(c, g[j], st[(i + j) % streams].cuda_stream) == 0
    torch.cuda.synchronize()
    for g in grids:
        for j, c in enumerate(cases):
            _equal(g[j], c)


def test_a_stream_that_is_gone(gpu):
    """Streams made and destroyed between the calls, whose handles come back, while earlier calls may run."""
    hip = _runtime()
    cases = [_case(2, 3), _case(3, 4)]
    grids = [_grids(cases) for _ in range(6)]
    for g in grids:
        for j, c in enumerate(cases):
            s = ctypes.c_void_p()
            assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
            assert _deposit(c, g[j], s.value) == 0
            assert hip.hipStreamDestroy(s) == 0
    torch.cuda.synchronize()
    for g in grids:
        for j, c in enumerate(cases):
            _equal(g[j], c)


def test_more_streams_than_kept_workspaces(gpu):
    """Calls that go round more streams than there are sets of workspaces do not wait for the device, and what the sets
    hold is given back on request."""
    from pylians_amd import _lib
    cases = [_case(2, 6), _case(3, 7)]
    st = [torch.cuda.Stream() for _ in range(6)]
    grids = _grids(cases)
    for _ in range(2):   # sizes every set
        for s in st:
            for j, c in enumerate(cases):
                assert _deposit(c, grids[j], s.cuda_stream) == 0
    torch.cuda.synchronize()
    a = torch.zeros(8192, 8192, device="cuda")
    torch.mm(a, a)
    turn = [_grids(cases) for _ in st]
    busy, ev = torch.cuda.Stream(), torch.cuda.Event()
    with torch.cuda.stream(busy):
        for _ in range(40):
            a = torch.mm(a, a)
        ev.record()
    for g, s in zip(turn, st):
        for j, c in enumerate(cases):
            assert _deposit(c, g[j], s.cuda_stream) == 0
    assert not ev.query()
    torch.cuda.synchronize()
    for g in turn:
        for j, c in enumerate(cases):
            _equal(g[j], c)
    held = torch.cuda.mem_get_info()[0]
    _lib.release_pool()
    assert torch.cuda.mem_get_info()[0] - held >= 4 * 60 * cases[1][0].shape[0]
    assert _deposit(cases[1], grids[1], st[0].cuda_stream) == 0
    torch.cuda.synchronize()
    _equal(grids[1], cases[1])


@pytest.mark.parametrize("axes", [2, 3])
def test_captured(gpu, axes):
    """Inside a capture the same call takes the direct kernel (float32 atomics); its replays leave the oracle's grid."""
    c = _case(axes, 5)
    g = torch.zeros((c[1],) * axes, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert _deposit(c, g, torch.cuda.current_stream().cuda_stream) == 0
    for _ in range(3):
        g.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        e = g.clone()
        assert _deposit(c, e, torch.cuda.current_stream().cuda_stream) == 0
        _equal(e, c)
        assert torch.allclose(g, e, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("axes", [2, 3])
def test_beside_a_capture(gpu, axes):
    """A call on one stream leaves a capture on another as it is, also where its workspaces are made or grow."""
    from pylians_amd import _lib
    small, large = _case(axes, 1), _case(axes, 9)
    grids = _grids([small, large])
    _lib.release_pool()
    x, side, graph = torch.zeros(4, device="cuda"), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x += 1
        for c, g in zip((small, large), grids):
            assert _deposit(c, g, side.cuda_stream) == 0
        x += 1
    side.synchronize()
    for c, g in zip((small, large), grids):
        o = c[2]
        assert np.allclose(g.cpu().numpy(), o, rtol=1e-4, atol=1e-4)   # (either route)
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, torch.full_like(x, 2.0 * (i + 1)))
