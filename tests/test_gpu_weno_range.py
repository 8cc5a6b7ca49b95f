"""GPU: WENO advection of scalars so large that the products of the weights' common
denominator, or of the numerator over it, leave the FP64 range: every value that the
per-weight form (the oracle's) can represent stays finite and right.

Tolerance: as test_gpu_weno_march, each face value is a combination of values of the size
of x with FP64 rounding of a few tens of operations: 200 eps |u|max |x|max (1/dx + 1/dy + 1/dz)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [5, 3])
@pytest.mark.parametrize("scale", [1e32, 1e33, 3e33, 1e34, 1e36, 3e59, 1e62, 1e70])
@pytest.mark.parametrize("shape", [(16, 16, 48), (48, 160, 320)], ids=lambda v: "x".join(map(str, v)))
def test_large_scalars_stay_finite(shape, scale, scheme):
    from ns3dperiodic_amd import NS3D
    from oracle.oracle import Oracle
    from tests.gpu_util import to_dev, to_host
    print(f"\n[case] weno range {shape} {scale} {scheme}", flush=True)
    rng = np.random.default_rng(11)
    u = [rng.standard_normal(shape) for _ in range(3)]
    x = scale * rng.standard_normal(shape)
    g, o = NS3D(*shape, Re=100.0, dt=1e-3), Oracle(*shape, Re=100.0, dt=1e-3)
    got = to_host([g.weno_advect(scheme, to_dev(u), to_dev([x])[0])])[0]
    ref = o.weno_advect(scheme, u, x)
    assert np.isfinite(ref).all() and np.isfinite(got).all()
    umax = max(np.abs(c).max() for c in u)
    bound = 200 * np.finfo(float).eps * umax * np.abs(x).max() * sum(n / (2 * np.pi) for n in shape)
    assert np.abs(got - ref).max() <= bound
