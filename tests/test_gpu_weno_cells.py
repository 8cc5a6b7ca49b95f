"""GPU: WENO advection and the scalar's stages on grids around the sizes where the launch
goes from one cell a thread to marching blocks, against the CPU oracle, in all schemes and
with both forms of the z reconstruction.

Tolerances: as test_gpu_weno_march for one application (200 eps |u|max |x|max (1/dx + 1/dy
+ 1/dz)); 1e-12 of the norm for a scalar step, as every FP64 operator."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zfix", [False, True])
@pytest.mark.parametrize("scheme", [5, 3, 1])
@pytest.mark.parametrize("shape", [(8, 16, 8), (8, 8, 512), (512, 8, 8), (48, 48, 80), (128, 64, 48), (80, 80, 80), (128, 64, 64),
                                   (96, 64, 64), (64, 96, 80)], ids=lambda s: "x".join(map(str, s)))
def test_cells_and_march(shape, scheme, zfix):
    from ns3dperiodic_amd import NS3D
    from oracle.oracle import Oracle
    from tests.gpu_util import to_dev, to_host
    print(f"\n[case] weno cells {shape} {scheme} {zfix}", flush=True)
    rng = np.random.default_rng(5)
    u = [rng.standard_normal(shape) for _ in range(3)]
    x = rng.standard_normal(shape)
    g = NS3D(*shape, Re=100.0, dt=1e-3, weno_zfix=zfix)
    o = Oracle(*shape, Re=100.0, dt=1e-3, weno_zfix=zfix)
    got = to_host([g.weno_advect(scheme, to_dev(u), to_dev([x])[0])])[0]
    umax = max(np.abs(c).max() for c in u)
    bound = 200 * np.finfo(float).eps * umax * np.abs(x).max() * sum(n / (2 * np.pi) for n in shape)
    assert np.abs(got - o.weno_advect(scheme, u, x)).max() <= bound


@pytest.mark.parametrize("scheme", [5, 3])
@pytest.mark.parametrize("shape", [(8, 8, 8), (32, 48, 32), (96, 80, 64)], ids=lambda s: "x".join(map(str, s)))
def test_scalar_steps(shape, scheme):
    import torch
    from ns3dperiodic_amd import NS3D, fields
    from oracle.oracle import Oracle
    from tests.gpu_util import to_dev, to_host
    print(f"\n[case] scalar cells {shape} {scheme}", flush=True)
    g, o = NS3D(*shape, Re=50.0, dt=1e-3), Oracle(*shape, Re=50.0, dt=1e-3)
    u, th = fields.random_solenoidal(*shape, seed=5), fields.random_scalar(*shape, seed=6)
    f = fields.kolmogorov_forcing_sin(*shape, n=2)
    ud, td = to_dev(u), torch.from_numpy(th).cuda()
    g.RK3_SSP_scalar(ud, td, to_dev(f), steps=2, scheme=scheme)
    uo, to = o.rk3_scalar(u, f, th, steps=2, scheme=scheme)
    for a, b in zip(to_host(ud) + to_host([td]), list(uo) + [to]):
        assert np.linalg.norm(a - b) < 1e-12 * np.linalg.norm(b)
