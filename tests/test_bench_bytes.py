"""bench.py's algorithmic bytes of a step: the passes that a call launches, where the
x-forward pass of a stage writes the next stage's P1 output without P1 reading the state."""
import pytest


@pytest.mark.parametrize("bulk,state", [(16, 16), (8, 16), (8, 8)])
def test_launched_bytes(bulk, state):
    import bench
    nc, steps = 256 * 256 * 129, 20
    pb = bench.pass_bytes(nc, bulk, state)
    assert bench.launched_bytes(pb, nc, bulk, steps, 3 * steps) == pytest.approx(bench.step_bytes(nc, bulk, state))
    # 59 of 60 stages read no state in P1
    chained = bench.step_bytes(nc, bulk, state) - 59 * 3 * state * nc / steps
    assert bench.launched_bytes(pb, nc, bulk, steps, 1) == pytest.approx(chained)


def test_launched_bytes_of_the_increment_loop():
    import bench
    nc = 64 * 64 * 33
    S = 8 * nc
    pb = bench.pass_bytes_incr(nc)
    assert bench.launched_bytes(pb, nc, 8, 10, 30) == pytest.approx(171 * S)
    # the first stage's P1 reads hi (3) and writes 6; the others are written (6) by the pass before
    assert bench.launched_bytes(pb, nc, 8, 10, 1, 9 * S) == pytest.approx((171 - 33 + 18) * S + 3 * S / 10)
