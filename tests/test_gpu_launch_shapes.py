"""Launch shapes other than the default (1024 threads, one workgroup per
CU, automatic count copies) against the oracle.  The shape sets the grid,
how many pairs a thread takes, the number of u16 partial rows that the
four-step transform's first pass sums (one per workgroup), and the number
of count copies the u32 histograms are spread over; none of it may change
a count or a coordinate.  Plain turns bit-identical; an intensity turn's
profile exact and coordinates within the first-turn bar of the large
tests."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from blond_amd.workloads import build_workload  # noqa: E402

from tests.test_gpu_tracking import host  # noqa: E402

ORC = orc.oracle_lib()
SHAPES = [(64, 1, 1), (256, 4, 2), (512, 2, 8)]


@pytest.mark.parametrize("turn_block", [25, 1])
@pytest.mark.parametrize("block,per_cu,groups", SHAPES)
def test_plain_turns_launch_shapes_bit_exact(block, per_cu, groups, turn_block):
    """c1, 11 turns as 6 + 5."""
    w = build_workload("c1", n_particles=60_001, n_turns=40)
    snap = w.snapshot()
    w.fused(6, block=block, blocks_per_cu=per_cu, groups=groups, turn_block=turn_block)
    w.fused(5)
    ref = orc.track(snap, 11, ORC)
    np.testing.assert_array_equal(host(w.beam.dt), ref["dt"])
    np.testing.assert_array_equal(host(w.beam.dE), ref["dE"])
    np.testing.assert_array_equal(host(w.profile.n_macroparticles), ref["profile"])


@pytest.mark.parametrize("name", ["c2", "c3"])
@pytest.mark.parametrize("block,per_cu,groups", SHAPES)
def test_intensity_turn_launch_shapes(name, block, per_cu, groups):
    """c2 (u32 LDS counts over `groups` copies) and c3 (u16 partial rows,
    one per workgroup: 196 to 391 rows here)."""
    w = build_workload(name, n_particles=200_001, n_turns=4)
    ref = orc.track(w.snapshot(), 1, ORC)
    w.fused(1, block=block, blocks_per_cu=per_cu, groups=groups)
    np.testing.assert_array_equal(host(w.profile.n_macroparticles), ref["profile"])
    vr = ref["induced_voltage"]
    assert np.max(np.abs(host(w.tiv.induced_voltage) - vr)) <= 1e-10 * np.abs(vr).max()
    sc = np.abs(ref["dE"]).max()
    np.testing.assert_allclose(host(w.beam.dE), ref["dE"], rtol=0, atol=1e-12 * sc)
    np.testing.assert_allclose(host(w.beam.dt), ref["dt"], rtol=1e-12, atol=0)


def test_a_given_block_is_kept():
    """5000 macroparticles on 100 slices: 256 threads where nothing was given,
    else what was, the default's value among it."""
    for given, want in (({}, 256), (dict(block=1024), 1024), (dict(block=512), 512),
                        (dict(block=64, blocks_per_cu=2), 64)):
        for name in ("c1", "c2"):
            w = build_workload(name, n_particles=5000, n_turns=4, n_slices=100,
                               **({} if name == "c1" else dict(n_fft=200)))
            assert _shape(w.fused(2, **given)) == (want, given.get("blocks_per_cu", 1))
    # many macroparticles or many slices: the default's full size
    for kw in (dict(n_particles=1_100_000, n_slices=100), dict(n_particles=5000, n_slices=2000)):
        assert _shape(build_workload("c1", n_turns=4, **kw).fused(1)) == (1024, 1)


def _shape(ft):
    import ctypes as ct

    from blond_amd import _lib

    block, per_cu = ct.c_int(), ct.c_int()
    _lib.call("blmi_engine_get_launch", ft._h, ct.byref(block), ct.byref(per_cu))
    return block.value, per_cu.value
