"""Lanes of several sizes in one run: each step's launches joined over the
sizes (`Model::join_batches`). A lane's bits are those of the lane alone,
eager and replayed, and after the sizes change."""
import numpy as np
import pytest

from ppocr_native_amd import GpuModel, nets
from ppocr_native_amd.planfile import PlanBuilder

pytestmark = pytest.mark.gpu


def runs(plan, sizes, xs, times=1):
    g = GpuModel.load(plan)
    out = []
    for sz, inputs in zip(sizes, xs):
        g.set_sizes(sz)
        for _ in range(times):
            for i, x in enumerate(inputs):
                g.lane_input_mut(i)[:] = x.reshape(-1)
            g.run()
            out.append([[g.lane_output(i, k) for k in range(g.output_count())] for i in range(len(sz))])
    n = len(g.launches())
    g.close()
    return out, n


def check(plan, sizes, lane, times=3):
    xs = [[lane(s, i) for i, s in enumerate(sz)] for sz in sizes]
    got, n = runs(plan, sizes, xs, times)
    for k, sz in enumerate(sizes):
        for i, s in enumerate(sz):
            alone = runs(plan, [[s]], [[xs[k][i]]])[0][0][0]
            for t in range(times):
                for a, b in zip(got[k * times + t][i], alone):
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (s, i, t)
    return n


def line(s, i):
    return np.random.default_rng(1000 * i + s[1]).uniform(-1, 1, (*s, 3)).astype(np.float32)


# More sizes than a launch takes, several lanes of one size, lines whose
# attention runs in one launch (under 128 steps) and those whose does not, odd
# widths; then two sizes, then one.
@pytest.mark.parametrize("logits", [False, True])
def test_recogniser_widths(logits):
    plan = nets.recognizer_plan(vocab=500, init="scaled", logits=logits)
    widths = [320, 1100, 333, 401, 509, 515, 640, 801, 77, 960, 320, 355, 1201, 421, 517, 729, 865, 903, 1030, 48, 640]
    sizes = [[(48, w) for w in widths], [(48, 320), (48, 1000), (48, 320)], [(48, 320)] * 3]
    check(plan, sizes[:1] if logits else sizes, line, times=3)


def test_recogniser_widths_many_classes():
    """Joined heads of so many classes that each line's records cover runs of
    tiles, its tiles' maxima behind them, where a line alone has a record a
    tile."""
    plan = nets.recognizer_plan(vocab=18385, init="scaled")
    check(plan, [[(48, w) for w in (320, 640, 1100, 801, 960, 333)]], line, times=2)


def test_detector_sizes():
    plan = nets.detector_plan(h=64, w=64, init="scaled")
    check(plan, [[(64, 96), (160, 64), (96, 96), (64, 96)]], line)


def test_launch_count():
    plan = nets.recognizer_plan(vocab=500, init="scaled")
    one, two = (check(plan, [[(48, w) for w in ws]], line, times=1) for ws in ([320, 320], [320, 330, 340]))
    assert one == two


def test_wide_gate_of_tiny_maps():
    """A gated 1x1 layer of many channels over one large map and many maps of
    one pixel: the tile that the large map's rows ask for leaves no room for the
    gates of the 32 small maps that 32 rows span."""
    rng = np.random.default_rng(2)
    w = lambda i, o: rng.normal(0, 1 / np.sqrt(i), (1, 1, i, o)).astype(np.float32)
    b = PlanBuilder(96, 128, 8)
    x = b.conv(b.input, w(8, 800), None)
    g = b.conv(b.mean(x), w(800, 16), None, fused="relu")
    g = b.conv(g, w(16, 800), None, fused="hardsigmoid")
    plan = b.to_bytes([b.conv(b.channelmul(x, g), w(800, 96), None)])
    lane = lambda s, i: np.random.default_rng(100 * i + s[0]).uniform(-1, 1, (*s, 8)).astype(np.float32)
    check(plan, [[(96, 128)] + [(1, 1)] * 32], lane, times=2)
