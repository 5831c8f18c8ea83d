"""XPk in float64 at the sizes where the binning kernel's work split has edges: fewer pairs of rows than threads, a last
partial block of kz columns, lines padded to the pitch, odd numbers of pairs, one and several rounds of workgroups
(line of sight z), every instantiation by number of fields and pairs; against the float64 oracle.

Tolerance: a transform is within about 1e-15 log2 N of its rms, a mode's product and Legendre weights (factors up to 9 and
35/8) within 1e-13 of the product of the amplitudes, so every mean over modes is within 1e-12 of the largest band power."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("N,F", [(8, 1), (12, 5), (20, 2), (40, 3), (48, 4), (80, 8), (96, 3), (160, 2), (192, 2)])
def test_xpk_shapes(gpu, N, F, axis):
    from oracle import pk as P
    from pylians_amd import Pk_library
    L = 250.0
    rng = np.random.default_rng(N + axis)
    base = rng.standard_normal((N, N, N))
    fields = [base * (i + 1) + rng.standard_normal((N, N, N)) for i in range(F)]
    MAS = [("CIC", "NGP", "TSC", "PCS", "None")[i % 5] for i in range(F)]
    if F == 1:   # one field: the autos of two equal fields
        fields, MAS = fields * 2, MAS * 2
    g = Pk_library.XPk(fields, L, axis=axis, MAS=MAS)
    o = P.XPk(fields, L, axis=axis, MAS=MAS)
    for name in ("Nmodes3D", "Nmodes1D", "Nmodes2D"):
        assert np.array_equal(getattr(g, name), getattr(o, name)), name
    for name in ("Pk", "XPk", "Pk1D", "PkX1D", "Pk2D", "PkX2D"):
        a, b = getattr(g, name), getattr(o, name)
        sel = slice(1, None) if name.endswith("2D") else slice(None)   # 2-D bin 0 holds the mean
        assert np.max(np.abs(a[sel] - b[sel])) <= 1e-12 * np.max(np.abs(b[sel])), name
