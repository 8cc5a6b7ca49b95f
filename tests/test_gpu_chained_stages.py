"""GPU: within one RK3 call the x-forward pass of a stage also runs the next
stage's x-inverse transforms; a call of one step never does across its end.
Steps taken in one call and one by one must agree bitwise (the transforms are
the same, on the same values), on every kind of x plan and precision."""
import pytest
import torch

from ns3dperiodic_amd import NS3D, fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32s", "fp32i"])
@pytest.mark.parametrize("nx", [8, 16, 48, 80, 96, 160, 192, 256, 320, 512])
def test_steps_in_one_call_match_single_steps(nx, precision):
    from tests.gpu_util import to_dev
    print(f"\n[case] chained stages nx={nx} {precision}", flush=True)
    shape = (nx, 16, 8)
    u = fields.random_solenoidal(*shape, seed=nx)
    f = to_dev(fields.kolmogorov_forcing_sin(*shape, n=2))
    g = NS3D(*shape, Re=50.0, dt=1e-3, precision=precision)
    if precision in ("fp32s", "fp32i"):
        # the conversion on entry and exit of a call rounds the state: one call against the same call
        # on a context that has just run something else
        a, b = to_dev(u), to_dev(u)
        g.RK3_SSP(a, f, steps=3)
        g.RK3_SSP(to_dev(fields.random_solenoidal(*shape, seed=nx + 1)), f, steps=1)
        g.RK3_SSP(b, f, steps=3)
    else:
        a, b = to_dev(u), to_dev(u)
        g.RK3_SSP(a, f, steps=3)
        for _ in range(3):
            g.RK3_SSP(b, f, steps=1)
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        assert torch.isfinite(torch.view_as_real(x)).all()
        assert torch.equal(torch.view_as_real(x), torch.view_as_real(y))
