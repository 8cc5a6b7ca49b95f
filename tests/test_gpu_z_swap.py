"""GPU: the z pass at the power-of-two lengths whose first exchange goes by lane swaps:
nonlinear and bilinear terms, single transforms and the passive scalar's velocity
against the oracle, on planes that leave the last block part full."""
import numpy as np
import pytest

from ns3dperiodic_amd import NS3D, fields
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 8, 64), (8, 48, 64), (8, 8, 128), (16, 80, 128), (8, 16, 256), (8, 8, 512)],
                         ids=lambda s: "x".join(map(str, s)))
def test_swap_z_lengths(shape):
    """Tolerances: 1e-12 as every FP64 operator, 1e-13 for one transform."""
    import torch
    from tests.gpu_util import to_dev, to_host
    print(f"\n[case] z swap {shape}", flush=True)
    g, o = NS3D(*shape, Re=50.0, dt=1e-3), Oracle(*shape, Re=50.0, dt=1e-3)
    u, v = fields.random_solenoidal(*shape, seed=3), fields.random_solenoidal(*shape, seed=4)

    def rel(a, b):
        return float(np.sqrt(sum(np.sum(np.abs(x - y) ** 2) for x, y in zip(a, b)) / sum(np.sum(np.abs(y) ** 2) for y in b)))

    assert rel(to_host(g.calculate_convolution_2p3(to_dev(u))), o.nonlinear(u)) < 1e-12
    assert rel(to_host(g.calculate_convolution_2p3_UV(to_dev(u), to_dev(v))), o.bilinear(u, v)) < 1e-12
    x = np.random.default_rng(shape[2]).standard_normal(shape)
    X = to_host([g.FFTN(torch.from_numpy(x).cuda())])[0]
    ref = np.fft.rfftn(x)
    assert np.linalg.norm(X - ref) < 1e-13 * np.linalg.norm(ref)
    back = to_host([g.iFFTN(torch.from_numpy(ref).cuda())])[0]
    assert np.linalg.norm(back - x) < 1e-13 * np.linalg.norm(x)
    th, f = fields.random_scalar(*shape, seed=6), fields.kolmogorov_forcing_sin(*shape, n=2)
    ud, td = to_dev(u), torch.from_numpy(th).cuda()
    g.RK3_SSP_scalar(ud, td, to_dev(f), steps=1)
    uo, to = o.rk3_scalar(u, f, th, steps=1)
    for a, b in zip(to_host(ud) + to_host([td]), list(uo) + [to]):
        assert np.linalg.norm(a - b) < 1e-12 * np.linalg.norm(b)
