"""The binned deposit's overflow list: particles crowded into two tiles, so that the list just fits one, two or all of the
workgroups that group it or is a little longer, against the FP64 oracle (float64 cell sums, one rounding to float32: 2^-24
relative, plus 1e-13 for sums in another order)."""
import numpy as np
import pytest
import torch

from oracle import cpu as C

pytestmark = pytest.mark.gpu

L = 64.0
RTOL = 2.0 ** -24 + 1e-13
ORDER = {"NGP": 1, "CIC": 2, "PCS": 4}


def _capacity(n, dims, S):
    """Records of a tile whose stencils stay inside it that fit before they overflow."""
    nt = (dims + 15) // 16
    p0 = 1.0 - (S - 1) * nt / dims
    return (int(2.0 * n / nt ** 3 * p0 ** 3) + 32 + 15) // 16 * 16


def _crowded(records, dims, scheme, seed):
    """Particles in the middle of one tile, `records` more than fit, and a twentieth as many at another's corner."""
    S, h = ORDER[scheme], L / dims
    m = n = records
    while m - _capacity(n, dims, S) < records:
        m += 1 + (records - (m - _capacity(n, dims, S))) // 2
        n = m + m // 20
    rng = np.random.default_rng(seed)
    nt = (dims + 15) // 16
    edge = -(-3 * dims // nt)   # first cell of tile 3
    pos = np.full((n, 3), edge + 6.0) + rng.random((n, 3))
    pos[m:] = edge - 0.5 + 0.3 * rng.random((n - m, 3))
    return np.ascontiguousarray(rng.permutation(pos) * h, dtype=np.float32)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("dims, scheme, records",
                         [(d, s, r) for d, s in ((64, "CIC"), (64, "NGP"), (80, "PCS"))
                          for r in (1, 1023, 1024, 1025, 2049, 262144, 270001)] +
                         [(61, "CIC", r) for r in (262144, 270001)])   # (fewer take the direct kernel there)
def test_crowded_tiles(gpu, dims, scheme, records, weighted):
    from pylians_amd import MAS_library
    pos = _crowded(records, dims, scheme, records)
    W = np.random.default_rng(3).random(len(pos), dtype=np.float32) + np.float32(0.25) if weighted else None
    o = C.deposit_f64(pos, dims, L, scheme, W)
    for _ in range(2):
        g = np.zeros((dims,) * 3, np.float32)
        MAS_library.MA(pos, g, L, scheme, W=W)
        assert np.all(np.abs(g - o) <= RTOL * np.abs(o))


def _stage_us(pos, dims, stage, calls=20):
    """Least time of a stage of the deposit over some calls."""
    from pylians_amd import MAS_library, _lib
    p, g, t = torch.from_numpy(pos).cuda(), torch.zeros((dims,) * 3, device="cuda"), []
    try:
        for _ in range(calls):
            _lib.profile(True)
            MAS_library.MA(p, g, L, "CIC")
            torch.cuda.synchronize()
            t.append(_lib.profile_read()[stage][1] * 1e3)
    finally:
        _lib.profile(False)
    return min(t)


def test_a_short_list_costs_little(gpu):
    """Grouping 4000 records takes a few microseconds more than finding the list empty (5 measured; waiting
    workgroups that fenced wave by wave took 60)."""
    rng = np.random.default_rng(1)
    spread = np.ascontiguousarray(rng.random((70000, 3)) * L, dtype=np.float32)
    assert _stage_us(_crowded(4000, 64, "CIC", 1), 64, "deposit_overflow") <= _stage_us(spread, 64, "deposit_overflow") + 30.0


def test_long_lists_do_not_wait_for_a_counter(gpu):
    """Two million particles in one tile are put into buckets and list in no more than twice the time that spread ones
    take (one reservation a record on the list's counter took twenty times as long)."""
    n = 1 << 21
    crowded = _crowded(n, 61, "CIC", 2)
    spread = np.ascontiguousarray(np.random.default_rng(2).random((len(crowded), 3)) * L, dtype=np.float32)
    assert _stage_us(crowded, 61, "deposit_bin") <= 2.0 * _stage_us(spread, 61, "deposit_bin")
