"""GPU: the z pass at radix-3 lengths, whose pencils take a power-of-two number of
lanes (some idle in the radix-4 passes) within one wave: nonlinear and bilinear
terms against the oracle on planes that leave the last block part full."""
import numpy as np
import pytest

from ns3dperiodic_amd import NS3D, fields
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-5)])
@pytest.mark.parametrize("nz", [48, 96, 192, 384])
@pytest.mark.parametrize("ny", [8, 48])
def test_radix3_z_lengths(ny, nz, precision, tol):
    """Tolerances: 1e-12 as every FP64 operator; FP32 transforms of O(1) data carry about
    eps32 * log2(N) = 1e-6, an order of magnitude is left for the products' cancellation."""
    from tests.gpu_util import to_dev, to_host
    print(f"\n[case] z lanes ny={ny} nz={nz} {precision}", flush=True)
    shape = (8, ny, nz)
    g, o = NS3D(*shape, Re=50.0, dt=1e-3, precision=precision), Oracle(*shape, Re=50.0, dt=1e-3)
    u, v = fields.random_solenoidal(*shape, seed=3), fields.random_solenoidal(*shape, seed=4)

    def rel(a, b):
        return float(np.sqrt(sum(np.sum(np.abs(x - y) ** 2) for x, y in zip(a, b)) / sum(np.sum(np.abs(y) ** 2) for y in b)))

    assert rel(to_host(g.calculate_convolution_2p3(to_dev(u))), o.nonlinear(u)) < tol
    assert rel(to_host(g.calculate_convolution_2p3_UV(to_dev(u), to_dev(v))), o.bilinear(u, v)) < tol


@pytest.mark.parametrize("nz", [48, 96, 192, 384])
def test_radix3_standalone_transforms_and_scalar(nz):
    """The single-field z transforms and the physical velocity that the z pass writes for the
    passive scalar, whose stores leave the idle lanes out."""
    import torch
    from tests.gpu_util import to_dev, to_host
    print(f"\n[case] z transforms nz={nz}", flush=True)
    shape = (8, 16, nz)
    g, o = NS3D(*shape, Re=50.0, dt=1e-3), Oracle(*shape, Re=50.0, dt=1e-3)
    rng = np.random.default_rng(nz)
    x = rng.standard_normal(shape)
    X = to_host([g.FFTN(torch.from_numpy(x).cuda())])[0]
    ref = np.fft.rfftn(x)
    assert np.linalg.norm(X - ref) < 1e-13 * np.linalg.norm(ref)
    back = to_host([g.iFFTN(torch.from_numpy(ref).cuda())])[0]
    assert np.linalg.norm(back - x) < 1e-13 * np.linalg.norm(x)
    u, th = fields.random_solenoidal(*shape, seed=5), fields.random_scalar(*shape, seed=6)
    f = fields.kolmogorov_forcing_sin(*shape, n=2)
    ud, td = to_dev(u), torch.from_numpy(th).cuda()
    g.RK3_SSP_scalar(ud, td, to_dev(f), steps=1)
    uo, to = o.rk3_scalar(u, f, th, steps=1)
    for a, b in zip(to_host(ud) + to_host([td]), list(uo) + [to]):
        assert np.linalg.norm(a - b) < 1e-12 * np.linalg.norm(b)
