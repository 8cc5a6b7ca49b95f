"""GPU: the y-inverse pass of small FP64 grids produces one output per block; larger
batches of the same grid use the pass with three outputs per block.  A batch member
must be bitwise the field advanced alone whichever form the batch takes."""
import pytest
import torch

from ns3dperiodic_amd import NS3D, fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 32, 16), (32, 48, 32), (16, 64, 64), (8, 80, 16), (16, 96, 32), (8, 128, 8),
                                   (8, 160, 8), (8, 192, 16), (8, 256, 8), (4 * 2, 320, 8), (8, 384, 8), (8, 512, 8)],
                         ids=lambda s: "x".join(map(str, s)))
def test_batch_of_many_matches_single(shape):
    from tests.gpu_util import to_dev
    print(f"\n[case] y split {shape}", flush=True)
    g = NS3D(*shape, Re=50.0, dt=1e-3)
    f = to_dev(fields.kolmogorov_forcing_sin(*shape, n=2))
    one = [to_dev(fields.random_solenoidal(*shape, seed=s)) for s in range(2)]
    many = torch.stack([torch.stack(one[i % 2]) for i in range(600)])
    g.RK3_SSP_batch(many, f, steps=2)
    for u in one:
        g.RK3_SSP(u, f, steps=2)
    torch.cuda.synchronize()
    for m in (0, 1, 598, 599):
        for c in range(3):
            assert torch.equal(torch.view_as_real(many[m, c]), torch.view_as_real(one[m % 2][c]))
