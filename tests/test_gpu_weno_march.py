"""GPU: the WENO advection kernel at the edges of its blocks (rows that do not fill a
block, y remainders, short marches, both cell counts per thread) and where the common
denominator of the weights leaves the FP64 range, against the CPU oracle.

Tolerance: each face value is a convex-like combination of values of the size of x with
FP64 rounding of a few tens of operations, so an output differs by at most
200 eps |u|max |x|max (1/dx + 1/dy + 1/dz)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [5, 3, 1])
@pytest.mark.parametrize("shape,scale,zfix", [((8, 8, 8), 1.0, False), ((16, 80, 48), 1.0, True), ((80, 8, 320), 1.0, False),
                                              ((8, 48, 512), 1.0, False), ((48, 96, 512), 1.0, True), ((160, 160, 96), 1.0, False),
                                              ((16, 32, 192), 1e40, False), ((16, 32, 192), 1e-40, False)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_weno_blocks_match_oracle(shape, scale, zfix, scheme):
    from ns3dperiodic_amd import NS3D
    from oracle.oracle import Oracle
    from tests.gpu_util import to_dev, to_host
    print(f"\n[case] weno {shape} {scale} {zfix} {scheme}", flush=True)
    rng = np.random.default_rng(7)
    u = [rng.standard_normal(shape) for _ in range(3)]
    x = scale * rng.standard_normal(shape)
    g = NS3D(*shape, Re=100.0, dt=1e-3, weno_zfix=zfix)
    o = Oracle(*shape, Re=100.0, dt=1e-3, weno_zfix=zfix)
    got = to_host([g.weno_advect(scheme, to_dev(u), to_dev([x])[0])])[0]
    ref = o.weno_advect(scheme, u, x)
    umax = max(np.abs(c).max() for c in u)
    bound = 200 * np.finfo(float).eps * umax * np.abs(x).max() * sum(n / (2 * np.pi) for n in shape)
    assert np.abs(got - ref).max() <= bound
