"""The intensity turn at the sizes where its launches change shape: slice
counts at the edges of the direct convolution's workgroup shapes, count copies
that are read four at a time and singly, and macroparticle counts at the edges
of the particle kernel's workgroup sizes (odd and even numbers of pairs a
thread, the last pair of an odd number, the odd macroparticle)."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from blond_amd.workloads import build_workload  # noqa: E402


def _first_turn(w, **launch):
    """The oracle's first turn: the profile exactly, the voltage to 1e-10 of
    its maximum (transform against convolution), coordinates to 1e-12."""
    ref = orc.track(w.oracle_copy(), 1)
    w.fused(1, **launch)
    assert np.array_equal(w.profile.n_macroparticles.cpu().numpy(), ref["profile"])
    v = w.tiv.induced_voltage.cpu().numpy()
    assert np.abs(v - ref["induced_voltage"]).max() <= 1e-10 * np.abs(ref["induced_voltage"]).max()
    for got, want in ((w.beam.dt, ref["dt"]), (w.beam.dE, ref["dE"])):
        assert np.abs(got.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()


@pytest.mark.parametrize("n_slices", [2, 7, 127, 500, 1023, 1024, 1025, 2047, 2049, 4096])
@pytest.mark.parametrize("groups", [1, 3, 4, 6])
def test_direct_convolution_shapes(n_slices, groups):
    w = build_workload("c2", n_particles=20001, n_turns=3, n_slices=n_slices, n_fft=2 * n_slices
                       if n_slices > 2 else 4)
    _first_turn(w, groups=groups, method="direct")


# one workgroup's transform: one wavefront a transform at both ends of its
# range and with two pairs a thread, workgroup-wide stages with their twiddles
# in LDS up to where both fit 160 KiB (n_fft 10240) and from memory above
@pytest.mark.parametrize("n_slices,n_fft", [
    (3, 6), (16, 32), (15, 30), (500, 1000), (1024, 1024), (1025, 2048), (1000, 2160),
    (2000, 8192), (2048, 10240), (2048, 10800)])
def test_one_workgroup_transform(n_slices, n_fft):
    _first_turn(build_workload("c2", n_particles=20001, n_turns=3, n_slices=n_slices, n_fft=n_fft),
                method="fft")


# pairs a thread 1 and 2 of 256, 512 and 1024 threads a workgroup on 256 CUs,
# and one macroparticle to either side
@pytest.mark.parametrize("pairs", [1, 65536, 131072, 262144, 3 * 262144])
@pytest.mark.parametrize("more", [-1, 0, 1, 3])
def test_particle_kernel_workgroup_sizes(pairs, more):
    n = 2 * pairs + more
    if n < 1:
        pytest.skip("no macroparticle")
    _first_turn(build_workload("c2", n_particles=n, n_turns=3, n_slices=300, n_fft=600))
    # plain turns, several a launch: bit for bit
    w = build_workload("c1", n_particles=n, n_turns=4)
    ref = orc.track(w.oracle_copy(), 3)
    w.fused(3)
    assert np.array_equal(w.beam.dt.cpu().numpy(), ref["dt"])
    assert np.array_equal(w.beam.dE.cpu().numpy(), ref["dE"])
    assert np.array_equal(w.profile.n_macroparticles.cpu().numpy(), ref["profile"])
