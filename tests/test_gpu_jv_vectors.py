"""GPU: the reduced J.v callbacks read and write the Krylov vectors in the x passes;
the same product through the unpack, bilinear right-hand side and pack entry points
is the reference.  Also the tangent step's half-sums against its stages."""
import math

import pytest
import torch

from ns3dperiodic_amd import NS3D, fields

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 2e-6)])
@pytest.mark.parametrize("shape", [(8, 8, 8), (48, 16, 32), (80, 32, 16), (256, 8, 16), (512, 8, 8)],
                         ids=lambda s: "x".join(map(str, s)))
def test_reduced_vectors(shape, precision, tol):
    """Tolerance: the FP64 arithmetic is the same up to contraction (1e-13 leaves a factor
    100 over round-off); in FP32 the transforms may round differently (eps32 * log2 N)."""
    from tests.gpu_util import to_dev
    print(f"\n[case] jv vectors {shape} {precision}", flush=True)
    g = NS3D(*shape, Re=30.0, dt=1e-3, precision=precision)
    u = to_dev(fields.random_solenoidal(*shape, seed=11))
    gen = torch.Generator().manual_seed(3)
    vec = torch.randn(g.vector_length_reduced(), generator=gen, dtype=torch.float64).cuda()
    tau = 0.7
    g.set_base_state(u, None, 1, tau)
    ref = g.pack_reduced(g.RK3_SSP_UV_RHS(u, g.unpack_reduced(vec)))
    assert _rel(g.jv_reduced(vec), ref) < tol
    assert _rel(g.jv_reduced(vec, newton=True), ref - vec / tau) < tol
    # input and output may be one vector
    both = vec.clone()
    g.lib.ns3d_jv_reduced(g.ctx, both.data_ptr(), both.data_ptr())
    torch.cuda.synchronize()
    assert torch.equal(both, g.jv_reduced(vec))


@pytest.mark.parametrize("shape", [(16, 16, 16), (96, 16, 48), (320, 8, 16)], ids=lambda s: "x".join(map(str, s)))
def test_tangent_step_is_its_stages(shape):
    """RK3_SSP_UV = half of v and half of two Euler stages about the old and the new base flow."""
    from tests.gpu_util import to_dev
    print(f"\n[case] tangent stages {shape}", flush=True)
    g = NS3D(*shape, Re=30.0, dt=1e-3)
    u, v = to_dev(fields.random_solenoidal(*shape, seed=1)), to_dev(fields.random_solenoidal(*shape, seed=2))
    u1, v1 = [c.clone() for c in u], [c.clone() for c in v]
    g.RK3_SSP_UV(u, v)
    w = [c.clone() for c in v1]
    g.single_time_step_UV(u1, w)
    g.RK3_SSP(u1)
    g.single_time_step_UV(u1, w)
    for a, b, c, d, e in zip(v, v1, w, u, u1):
        assert _rel(a, 0.5 * b + 0.5 * c) < 1e-14
        assert torch.equal(d, e)
    assert math.isfinite(float(v[0].abs().max()))
