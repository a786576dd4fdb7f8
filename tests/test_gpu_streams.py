"""Turns enqueued on a stream of the caller's that is busy and does not wait for
the default one, and what is set between them: the same bits as on the default
stream, one call after the other."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from blond_amd.trackers.differentiable import DifferentiableTracker  # noqa: E402
from blond_amd.trackers.ensemble import EnsembleTracker  # noqa: E402
from blond_amd.workloads import build_adjoint_case, build_ensemble, build_workload  # noqa: E402

BUSY = 100_000_000  # cycles of a sleep ahead of the turns: tens of ms


def _on(side, run):
    """run() on a busy stream of its own, or on the default stream."""
    if not side:
        out = run(lambda: None)
    else:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            out = run(lambda: torch.cuda._sleep(BUSY))
        stream.synchronize()
    torch.cuda.synchronize()
    return out


def _equal(run):
    for a, b in zip(_on(False, run), _on(True, run)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name,kw", [("c1", {}), ("c2", dict(n_slices=500, n_fft=1000)),
                                     ("c3", {})])
def test_program_started_again(name, kw):
    def run(busy):
        w = build_workload(name, n_particles=20001, n_turns=60, **kw)
        w.fused(1)
        busy()
        w.fused(10)
        w.rf.counter[0] = 3
        w.fused(20)
        w.rf.counter[0] = 0
        w.fused(5)
        return [w.beam.dt, w.beam.dE, w.profile.n_macroparticles]

    _equal(run)


def test_ensemble_program_started_again():
    def run(busy):
        w = build_ensemble(n_bunches=4, n_turns=60, n_slices=256, n_min=1e3, n_max=1e4)
        e = EnsembleTracker(w.trackers, w.profiles, w.tivs)
        e.track(1)
        busy()
        e.track(10)
        for tr in e.trackers:
            tr.rf_params.counter[0] = 3
        e.track(20)
        return [e.dt, e.dE, e.prof]

    _equal(run)


def test_forward_passes_one_after_the_other():
    """Each pass's profile is its own parameters', with no backward pass (whose
    gradients come back to the host) in between."""
    def run(busy):
        c = build_adjoint_case(n_particles=5001, n_turns=11, n_slices=64, seed=5, intensity=1e11)
        dtr = DifferentiableTracker(c.tracker, c.profile)
        out = []
        for scale in (1.0, 1.1, 0.9):
            busy()
            p = {k: torch.tensor(v, dtype=torch.float64) for k, v in c.theta0.items()}
            p["V"], p["R"] = p["V"] * scale, p["R"] * scale
            out.append(dtr.profile_after(p["V"], p["phi"], p["R"], p["fr"], p["Q"], turns=10))
        torch.cuda.synchronize()
        dtr.close()
        return out

    _equal(run)
