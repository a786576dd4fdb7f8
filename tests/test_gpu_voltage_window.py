"""The u16-row particle kernel with buffer descriptors and the voltage window:
the same bits as the kernel it stands in for (which merged counts still take),
and the gathered table where the bin centres are not on the cuts' line."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from blond_amd.utils import bm  # noqa: E402
from blond_amd.workloads import build_wake_workload, build_workload  # noqa: E402


def _run(name, turns, peel, launch=None, **kw):
    w = build_workload(name, n_turns=turns + 1, **kw)
    w.fused(1, max_peel=peel, **(launch or {}))
    w.fused(turns - 1)
    return [a.cpu().numpy() for a in (w.beam.dt, w.beam.dE, w.profile.n_macroparticles,
                                      w.tiv.induced_voltage)]


# u16 rows without a histogram window, with one, and a slice count whose
# transform is no power of two; one and two RF systems; odd and tiny bunches,
# an odd and an even number of pairs a thread
@pytest.mark.parametrize("name,n_slices,n_fft", [("c2", 20000, 20000), ("c2", 32768, 65536),
                                                 ("c3", 65536, 131072), ("c2", 40000, 48000)])
@pytest.mark.parametrize("n", [1, 4097, 300001, 2 * 262144 + 2, 4 * 262144 + 3])
@pytest.mark.parametrize("precision", ["double", "single"])
def test_same_bits_as_the_gathering_kernel(name, n_slices, n_fft, n, precision):
    bm.use_precision(precision)
    try:
        kw = dict(n_particles=n, n_slices=n_slices, n_fft=n_fft)
        for a, b in zip(_run(name, 4, 0, **kw), _run(name, 4, 1, **kw)):
            assert np.array_equal(a, b)
    finally:
        bm.use_precision("double")


# the other drifts, and moments (their sums run over the pairs the byte offsets
# own, and over the odd last pair and macroparticle), on the line and off it
@pytest.mark.parametrize("name,n_slices,n_fft", [("c2", 20000, 20000), ("c3", 65536, 131072)])
@pytest.mark.parametrize("n", [300001, 2 * 262144 + 2, 4 * 262144 + 3])
@pytest.mark.parametrize("solver,statistics,moved", [
    ("legacy", False, False), ("exact", False, False), ("simple", True, False),
    ("exact", True, True)])
@pytest.mark.parametrize("precision", ["double", "single"])
def test_same_bits_with_other_drifts_and_moments(name, n_slices, n_fft, n, solver, statistics,
                                                 moved, precision):
    bm.use_precision(precision)
    try:
        out = []
        for peel in (0, 1):
            w = build_workload(name, n_particles=n, n_turns=5, n_slices=n_slices, n_fft=n_fft)
            w.tracker.solver = solver
            if moved:
                w.profile.bin_centers[n_slices // 2:n_slices // 2 + 50] += \
                    0.1 * float(w.profile.bin_size)
            ft = w.fused(3, max_peel=peel, statistics=statistics)
            out.append([a.cpu().numpy() for a in (w.beam.dt, w.beam.dE,
                                                  w.profile.n_macroparticles,
                                                  w.tiv.induced_voltage)])
            if statistics:
                out[-1].append(ft.statistics(1, 3))
                assert (out[-1][-1][:, 0] == n).all()
        for a, b in zip(*out):
            assert np.array_equal(a, b)
    finally:
        bm.use_precision("double")


def test_same_bits_beyond_the_last_level_cache():
    """2^24 macroparticles and three: non-temporal coordinates, on the line
    and then off it."""
    ws = [build_workload("c3", n_particles=2 ** 24 + 3, n_turns=5, n_slices=65536, n_fft=131072)
          for _ in range(2)]
    for turns, moved in ((2, False), (1, True)):
        for peel, w in enumerate(ws):
            if moved:
                w.profile.bin_centers[32700:32800] += 0.1 * float(w.profile.bin_size)
            w.fused(turns, max_peel=peel)
        for get in (lambda w: w.beam.dt, lambda w: w.beam.dE,
                    lambda w: w.profile.n_macroparticles, lambda w: w.tiv.induced_voltage):
            assert torch.equal(get(ws[0]), get(ws[1]))


# fewer threads stage the window, in more rounds and with the last round cut
# short; at 20000 slices it starts at an odd bin
@pytest.mark.parametrize("name,n_slices,n_fft", [("c2", 20000, 20000), ("c3", 65536, 131072)])
@pytest.mark.parametrize("block,per_cu", [(64, 1), (256, 2), (512, 1)])
def test_same_bits_at_other_launch_shapes(name, n_slices, n_fft, block, per_cu):
    kw = dict(n_particles=300001, n_slices=n_slices, n_fft=n_fft,
              launch=dict(block=block, blocks_per_cu=per_cu))
    for a, b in zip(_run(name, 3, 0, **kw), _run(name, 3, 1, **kw)):
        assert np.array_equal(a, b)


# the window of entries where centres are off the line: 20000 slices (from an
# odd bin) and 65536, no pair, one and an odd number of them a thread, and
# fewer threads to stage it
@pytest.mark.parametrize("name,n_slices,n_fft", [("c2", 20000, 20000), ("c3", 65536, 131072)])
@pytest.mark.parametrize("n,block", [(1, 1024), (300001, 1024), (300001, 64),
                                     (4 * 262144 + 3, 1024)])
def test_same_bits_off_the_line(name, n_slices, n_fft, n, block):
    out = []
    for peel in (0, 1):
        w = build_workload(name, n_particles=n, n_turns=4, n_slices=n_slices, n_fft=n_fft)
        w.profile.bin_centers[n_slices // 3::2] += 0.1 * float(w.profile.bin_size)
        w.fused(3, max_peel=peel, block=block)
        out.append((w.beam.dt, w.beam.dE, w.profile.n_macroparticles, w.tiv.induced_voltage))
    for a, b in zip(*out):
        assert torch.equal(a, b)


def _turn_matches_oracle(w):
    ref = orc.track(w.oracle_copy(), 1)
    w.fused(1)
    assert np.array_equal(w.profile.n_macroparticles.cpu().numpy(), ref["profile"])
    for got, want in ((w.beam.dt, ref["dt"]), (w.beam.dE, ref["dE"])):
        assert np.abs(got.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()


def test_bin_centres_off_the_line_use_the_table():
    """Centres moved by a tenth of a bin inside the window, before the first
    turn and in place between two calls: the kick follows them."""
    w = build_workload("c3", n_particles=200001, n_turns=6, n_slices=65536, n_fft=131072,
                       intensity=1e13)
    _turn_matches_oracle(w)
    bc = w.profile.bin_centers
    step = float(w.profile.bin_size)
    line = bc.clone()
    for at in (32768, 31000):
        bc[at:at + 1000] += 0.1 * step
        _turn_matches_oracle(w)
    bc.copy_(line)
    _turn_matches_oracle(w)


def _both(build):
    """Two workloads of the same bunch, one tracked by each kernel."""
    return [(build(), dict(max_peel=peel)) for peel in (0, 1)]


def _same(pair):
    (a, _), (b, _) = pair
    for x, y in ((a.beam.dt, b.beam.dt), (a.beam.dE, b.beam.dE),
                 (a.profile.n_macroparticles, b.profile.n_macroparticles),
                 (a.tiv.induced_voltage, b.tiv.induced_voltage)):
        assert torch.equal(x, y)


def _builds():
    yield lambda: build_workload("c2", n_particles=60001, n_turns=40, n_slices=20000,
                                 n_fft=20000, intensity=1e13)
    yield lambda: build_workload("c3", n_particles=60001, n_turns=40, n_slices=65536,
                                 n_fft=131072, intensity=1e13)
    # the wake step forms the table: a multi-turn memory, an inductive source
    # alone (no transform) and beside a convolution
    for kind in ("mtw", "zovern", "mixed"):
        yield lambda kind=kind: build_wake_workload(kind, n_particles=60001, n_turns=40,
                                                    n_slices=20000, memory_turns=2)


@pytest.mark.parametrize("build", _builds(), ids=["c2", "c3", "mtw", "zovern", "mixed"])
def test_bin_centres_on_and_off_the_line(build):
    """The same bits as the gathering kernel while centres leave the line and
    come back between calls of one, two and three turns: the first, one
    inside the window and the last of the table's, and the one past it, which
    only scales the table; then the program started again."""
    pair = _both(build)
    ns = pair[0][0].profile.n_slices
    line = [w.profile.bin_centers.clone() for w, _ in pair]
    step = float(pair[0][0].profile.bin_size)
    for turns, moved in ((1, None), (2, ns // 2), (1, ns // 2 + 7), (3, None), (1, 0), (1, None),
                         (2, ns - 2), (1, None), (1, None), (3, ns - 1), (2, None)):
        for (w, kw), l in zip(pair, line):
            w.profile.bin_centers.copy_(l)
            if moved is not None:
                w.profile.bin_centers[moved] += 0.1 * step
            w.fused(turns, **kw)
        _same(pair)
    if getattr(pair[0][0].tiv.induced_voltage_list[0], "multi_turn_wake", False):
        return  # the memory belongs to the turns before
    for w, kw in pair:
        w.profile.bin_centers[ns // 2] += 0.1 * step
        w.fused(1)
        w.rf.counter[0] = 0
        w.profile.bin_centers.copy_(line[0])
        w.fused(3)
    _same(pair)
