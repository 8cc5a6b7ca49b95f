"""GPU: the RK3 loops with the next stage's x-inverse transforms carried by the x-forward
pass, against the same loops with every stage's x-inverse pass on its own
(NS3D_FLAG_NO_CHAIN): bitwise the same, at every x length, in every precision, between the
stages of a step and between steps, with both masks; also batches and the passive scalar."""
import pytest
import torch

from ns3dperiodic_amd import NS3D, fields

pytestmark = pytest.mark.gpu

LENGTHS = [8, 16, 32, 48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512]


def _same(a, b):
    for x, y in zip(a, b):
        x, y = (torch.view_as_real(t) if t.is_complex() else t for t in (x, y))
        assert torch.isfinite(x).all()
        assert torch.equal(x, y)


@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("physical", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32s", "fp32i"])
@pytest.mark.parametrize("nx", LENGTHS)
def test_steps(nx, precision, physical, steps):
    from tests.gpu_util import to_dev
    print(f"\n[case] chain apart nx={nx} {precision} {physical} {steps}", flush=True)
    shape = (nx, 16, 16)
    kw = dict(Re=50.0, dt=1e-3, precision=precision, ipq=not physical, mask_nyquist=physical)
    f = to_dev(fields.kolmogorov_forcing_sin(*shape, n=2))
    a, b = to_dev(fields.random_solenoidal(*shape, seed=nx)), to_dev(fields.random_solenoidal(*shape, seed=nx))
    NS3D(*shape, **kw).RK3_SSP(a, f, steps=steps)
    NS3D(*shape, chain_stages=False, **kw).RK3_SSP(b, f, steps=steps)
    _same(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx", [16, 48, 128, 256])
def test_batch_members_and_scalar(nx, precision):
    from tests.gpu_util import to_dev
    print(f"\n[case] chain apart, batch and scalar nx={nx} {precision}", flush=True)
    shape = (nx, 8, 32)
    f = to_dev(fields.kolmogorov_forcing_sin(*shape, n=2))
    us = [to_dev(fields.random_solenoidal(*shape, seed=s)) for s in range(3)]
    th0 = torch.from_numpy(fields.random_scalar(*shape, seed=6)).cuda()
    out = []
    for chain in (True, False):
        g = NS3D(*shape, Re=50.0, dt=1e-3, precision=precision, chain_stages=chain)
        ub, um = (torch.stack([torch.stack(u) for u in us]).contiguous() for _ in range(2))
        g.RK3_SSP_batch(ub, f, steps=2)
        dt, Re = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in ([1e-3, 5e-4, 2e-3], [50.0, 70.0, 90.0]))
        n = torch.tensor([3, 0, 1], dtype=torch.int32, device="cuda")
        g.RK3_SSP_batch_members(um, f, dt, Re, n, 3)
        u, th = [c.clone() for c in us[0]], th0.clone()
        g.RK3_SSP_scalar(u, th, f, steps=2)
        out.append([ub, um, th] + u)
    _same(*out)
