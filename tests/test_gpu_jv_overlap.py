"""GPU: the reduced J.v callbacks on an input and an output vector that overlap without
being one vector give what they give on separate vectors (the input is a buffer of the
caller's, read in full before the output takes its place)."""
import pytest
import torch

from ns3dperiodic_amd import NS3D, fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("newton", [False, True])
@pytest.mark.parametrize("offset", [1, 7, 2048, -1, -301])
@pytest.mark.parametrize("shape", [(8, 8, 8), (32, 48, 32)], ids=lambda s: "x".join(map(str, s)))
def test_overlapping_vectors(shape, offset, newton):
    from tests.gpu_util import to_dev
    print(f"\n[case] jv overlap {shape} {offset} {newton}", flush=True)
    g = NS3D(*shape, Re=30.0, dt=1e-3)
    u = to_dev(fields.random_solenoidal(*shape, seed=11))
    g.set_base_state(u, None, 1, 0.7)
    n = g.vector_length_reduced()
    offset = max(-n + 1, min(n - 1, offset))
    vec = torch.randn(n, generator=torch.Generator().manual_seed(3), dtype=torch.float64).cuda()
    ref = g.jv_reduced(vec, newton=newton)
    buf = torch.zeros(n + abs(offset), dtype=torch.float64, device="cuda")
    i, o = (0, offset) if offset > 0 else (-offset, 0)
    buf[i:i + n] = vec
    fn = g.lib.ns3d_jv_reduced_newton if newton else g.lib.ns3d_jv_reduced
    fn(g.ctx, buf.data_ptr() + 8 * i, buf.data_ptr() + 8 * o)
    assert g.lib.ns3d_last_error(g.ctx) == 0
    torch.cuda.synchronize()
    assert torch.equal(buf[o:o + n], ref)
