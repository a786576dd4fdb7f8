"""The differentiable tracker at the sizes where its launches change: slice
counts at the edges of the matrix product's 16-wide chunks and tiles and of
the range whose product runs inside the particle launch (512), odd
macroparticle counts (the arrays' pad slots), less than a pair a thread and
more than two, segments of one turn and cut short."""
import numpy as np
import pytest

from oracle import adjoint as adj

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from blond_amd.trackers.differentiable import DifferentiableTracker  # noqa: E402
from blond_amd.workloads import build_adjoint_case  # noqa: E402

KEYS = ("V", "phi", "R", "fr", "Q")


@pytest.mark.parametrize("map", ["reference", "spline"])
@pytest.mark.parametrize("n,n_slices,every,turns", [
    (5001, 15, 3, 7), (5000, 16, 1, 5), (5001, 17, 4, 5), (1, 64, 2, 4), (20001, 255, 50, 6),
    (20000, 257, 4, 9), (20001, 511, 5, 6), (20001, 512, 5, 6), (20000, 513, 5, 6),
    (20001, 1024, 3, 4), (2 * 262144 * 2 + 5, 64, 3, 4),
    # the pass's correlation over few turns: as many shares of its outputs as
    # there are 64 of them, shares cut short, and two
    (5001, 1024, 1, 1), (5001, 300, 2, 12), (5001, 100, 50, 100)])
def test_profile_and_gradient_at_size_edges(n, n_slices, every, turns, map):
    """The forward profile to 1e-8 of its peak and the gradient to 1e-6 of
    the float64 CPU map's (the bars of the full-size tests): the piecewise
    maps' rounding differences move at most single particles' weights."""
    c = build_adjoint_case(n_particles=n, n_turns=turns + 1, n_slices=n_slices, seed=5,
                           intensity=1e11)
    dtr = DifferentiableTracker(c.tracker, c.profile, checkpoint_every=every, map=map)
    m = adj.DiffMap(c.state, mode=map)
    th, ts = c.theta0, c.theta_star
    target = m.forward(c.beam.dt, c.beam.dE, ts["V"], ts["phi"], ts["R"], ts["fr"], ts["Q"], turns)
    ps = [torch.tensor(th[k], dtype=torch.float64, device="cuda", requires_grad=True)
          for k in KEYS]
    p = dtr.profile_after(*ps, turns=turns)
    want = m.forward(c.beam.dt, c.beam.dE, th["V"], th["phi"], th["R"], th["fr"], th["Q"], turns)
    got = p.detach().cpu().numpy()
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-8 * np.abs(want).max())
    torch.sum((p - torch.from_numpy(target).cuda()) ** 2).backward()
    ref = m.gradient(c.beam.dt, c.beam.dE, th["V"], th["phi"], th["R"], th["fr"], th["Q"], turns,
                     2 * (got - target))
    for k, t in zip(KEYS, ps):
        g = t.grad.cpu().numpy()[0]
        assert abs(g - ref[k][0]) <= 1e-6 * abs(ref[k][0]), (k, g, ref[k][0])
    dtr.close()
