"""GPU: the y-inverse pass at every y length, with y columns that the mask drops (the
alias-free mask; the reference's leaves the y axis whole): nonlinear and bilinear terms
against the oracle, whose loads of masked elements the kernel leaves out or range-checks."""
import numpy as np
import pytest

from ns3dperiodic_amd import NS3D, fields
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-5)])
@pytest.mark.parametrize("nyquist", [False, True])
@pytest.mark.parametrize("ny", [8, 16, 32, 48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512])
def test_y_lengths(ny, nyquist, precision, tol):
    """Tolerances: 1e-12 as every FP64 operator; FP32 transforms of O(1) data carry about
    eps32 * log2(N) = 1e-6, an order of magnitude is left for the products' cancellation."""
    from tests.gpu_util import to_dev, to_host
    print(f"\n[case] y loads ny={ny} nyquist={nyquist} {precision}", flush=True)
    shape = (8, ny, 32)
    g = NS3D(*shape, Re=50.0, dt=1e-3, precision=precision, mask_nyquist=nyquist)
    o = Oracle(*shape, Re=50.0, dt=1e-3, mask_nyq=nyquist)
    u, v = fields.random_solenoidal(*shape, seed=3), fields.random_solenoidal(*shape, seed=4)

    def rel(a, b):
        return float(np.sqrt(sum(np.sum(np.abs(x - y) ** 2) for x, y in zip(a, b)) / sum(np.sum(np.abs(y) ** 2) for y in b)))

    assert rel(to_host(g.calculate_convolution_2p3(to_dev(u))), o.nonlinear(u)) < tol
    assert rel(to_host(g.calculate_convolution_2p3_UV(to_dev(u), to_dev(v))), o.bilinear(u, v)) < tol
