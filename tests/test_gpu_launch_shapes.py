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
    """5000 macroparticles on 100 slices: fewer threads where nothing was
    given, else what was, the default's value among it."""
    for given, plain, table in (({}, 256, 512), (dict(block=1024), 1024, 1024),
                                (dict(block=512), 512, 512),
                                (dict(block=64, blocks_per_cu=2), 64, 64)):
        for name, want in (("c1", plain), ("c2", table)):
            w = build_workload(name, n_particles=5000, n_turns=4, n_slices=100,
                               **({} if name == "c1" else dict(n_fft=200)))
            assert _shape(w.fused(2, **given)) == (want, given.get("blocks_per_cu", 1))
    # many macroparticles or many slices: the default's full size
    for kw in (dict(n_particles=1_100_000, n_slices=100), dict(n_particles=5000, n_slices=2000)):
        assert _shape(build_workload("c1", n_turns=4, **kw).fused(1)) == (1024, 1)


# macroparticles a CU at the edges of each form's rule, and the threads either
# side: plain turns several and one to a launch, with moments, and a table
@pytest.mark.parametrize("name,precision,launch,at,low,high", [
    ("c1", "double", {}, 1024, 256, 512), ("c1", "double", {}, 2048, 512, 1024),
    ("c1", "single", {}, 1024, 256, 512),
    ("c1", "double", dict(turn_block=1), 256, 256, 512),
    ("c1", "double", dict(turn_block=1), 1024, 512, 1024),
    ("c1", "double", dict(statistics=True), 1024, 512, 1024),
    ("c1", "single", dict(turn_block=1), 256, 512, 512),
    ("c2", "double", {}, 1024, 512, 1024), ("c2", "single", {}, 1024, 1024, 1024)])
def test_block_rule_edges(name, precision, launch, at, low, high):
    from blond_amd.utils import bm

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    bm.use_precision(precision)
    try:
        for n, want in ((cus * at, low), (cus * at + 1, high)):
            out = []
            for given in ({}, dict(block=1024)):
                w = build_workload(name, n_particles=n, n_turns=4, n_slices=300,
                                   **({} if name == "c1" else dict(n_fft=600)))
                ft = w.fused(3, **launch, **given)
                assert _shape(ft)[0] == given.get("block", want)
                out.append((w.beam.dt, w.beam.dE, w.profile.n_macroparticles))
            # counts are whole numbers and a macroparticle's arithmetic its own
            for a, b in zip(*out):
                assert torch.equal(a, b)
    finally:
        bm.use_precision("double")


def _shape(ft):
    import ctypes as ct

    from blond_amd import _lib

    block, per_cu = ct.c_int(), ct.c_int()
    _lib.call("blmi_engine_get_launch", ft._h, ct.byref(block), ct.byref(per_cu))
    return block.value, per_cu.value
