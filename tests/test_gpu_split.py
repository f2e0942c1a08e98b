"""The kernels that multiply f32 on the bf16 matrix cores (csrc/split.hpp):
three bf16 parts a value, six products, at the edges of their tiles, row and
column counts and value range."""
import numpy as np
import pytest

from ppocr_native_amd import GpuModel
from ppocr_native_amd.planfile import PlanBuilder

pytestmark = pytest.mark.gpu


def gpu(plan, shape, xs):
    g = GpuModel.load(plan)
    g.set_sizes([shape[:2]] * len(xs))
    for i, x in enumerate(xs):
        g.lane_input_mut(i)[:] = x.reshape(-1)
    g.run()
    got = [g.lane_output(i) for i in range(len(xs))]
    g.close()
    return got


def ctc_plan(rng, t, c, vocab):
    w = rng.normal(0, 2 / np.sqrt(c), (c, vocab)).astype(np.float32)
    bias = rng.normal(0, 0.5, vocab).astype(np.float32)
    b = PlanBuilder(1, t, c)
    return b.to_bytes([b.ctcargmax(b.input, w, bias)])


# Rows below, at and past the 128 of a workgroup; one input group of 32 and
# four, whole and not; one column, one tile, tiles that do not fill a run;
# (4160 rows, 48 tiles) enough workgroups that each walks a whole run, (1280
# rows, 313 tiles) so many that each walks two, its last a short one; and (640
# rows, 288 tiles) few enough for single tiles, three a workgroup.
@pytest.mark.parametrize("lanes,t,c,vocab", [(1, 1, 4, 1), (1, 5, 32, 64), (3, 43, 36, 65), (1, 128, 64, 400),
                                             (2, 80, 128, 385), (26, 160, 100, 3050),
                                             (8, 160, 32, 20000), (4, 160, 64, 18385)])
def test_ctc_panel(oracle, lanes, t, c, vocab):
    rng = np.random.default_rng(c + vocab)
    plan = ctc_plan(rng, t, c, vocab)
    xs = [rng.normal(0, 1, (1, t, c)).astype(np.float32) for _ in range(lanes)]
    m = oracle.OracleModel(plan)
    for x, a in zip(xs, gpu(plan, (1, t, c), xs)):
        a, b = a.reshape(-1, 2), m.run(x)[0].reshape(-1, 2)
        assert np.array_equal(a[:, 0], b[:, 0])
        # f32 sums of `vocab` terms in another order: 1e-5, as the other CTC tests.
        np.testing.assert_allclose(a[:, 1], b[:, 1], rtol=1e-5, atol=1e-5)


def test_ctc_panel_odd_values(oracle):
    """Rows with values that have no bf16 parts leave the rows beside them
    alone, and tiny values keep their product."""
    rng = np.random.default_rng(3)
    plan = ctc_plan(rng, 40, 48, 500)
    x = rng.normal(0, 1, (1, 40, 48)).astype(np.float32)
    y = x.copy()
    y[0, 7, 5], y[0, 7, 6], y[0, 20, 0], y[0, 39, 47] = np.inf, -np.inf, np.nan, 3.4e38
    y[0, 11] *= np.float32(1e-30)
    a, b = (v.reshape(-1, 2) for v in gpu(plan, (1, 40, 48), [x, y]))
    same = [r for r in range(40) if r not in (7, 11, 20, 39)]
    assert np.array_equal(a[same].view(np.uint32), b[same].view(np.uint32))
    want = oracle.OracleModel(plan).run(y)[0].reshape(-1, 2)
    finite = [r for r in range(40) if r not in (7, 20)]  # 39 in its class alone: its logits' exponents overflow
    assert np.isfinite(want[finite]).all() and np.isnan(want[[7, 20], 1]).all()
    assert np.array_equal(b[finite, 0], want[finite, 0])
    np.testing.assert_allclose(b[finite[:-1], 1], want[finite[:-1], 1], rtol=1e-5)
    assert not (b[[7, 20], 1] <= 1).any()  # no probability where there is none


# Inputs, and then weights, so small that their last bits lie below bf16's
# smallest step: normal ones, the last normal ones, subnormal inputs.
TINY = [(2.0 ** -118, 2.0 ** 117), (2.0 ** -127, 2.0 ** 125), (2.0 ** -136, 2.0 ** 125), (2.0 ** 100, 2.0 ** -122)]


@pytest.mark.parametrize("sx,sw", TINY)
def test_ctc_panel_tiny_values(oracle, sx, sw):
    rng = np.random.default_rng(6)
    w = (rng.normal(0, 0.3, (48, 500)) * sw).astype(np.float32)
    b = PlanBuilder(1, 40, 48)
    plan = b.to_bytes([b.ctcargmax(b.input, w, rng.normal(0, 0.1 * sx * sw, 500).astype(np.float32))])
    x = (rng.normal(0, 1, (1, 40, 48)) * sx).astype(np.float32)
    got = gpu(plan, (1, 40, 48), [x])[0].reshape(-1, 2)
    want = oracle.OracleModel(plan).run(x)[0].reshape(-1, 2)
    assert np.array_equal(got[:, 0], want[:, 0])
    np.testing.assert_allclose(got[:, 1], want[:, 1], rtol=1e-5)


@pytest.mark.parametrize("sx,sw", TINY)
@pytest.mark.parametrize("s", [1, 2])
def test_conv_patch_split_tiny_values(oracle, s, sx, sw):
    rng = np.random.default_rng(7)
    b = PlanBuilder(20, 24, 40)
    wt = (rng.normal(0, 0.1, (3, 3, 40, 24)) * sw).astype(np.float32)
    plan = b.to_bytes([b.conv(b.input, wt, None, k=(3, 3), s=(s, s), pad=(1, 1, 1, 1))])
    x = (rng.uniform(-1, 1, (20, 24, 40)) * sx).astype(np.float32)
    want = oracle.OracleModel(plan).run(x)[0].reshape(-1).astype(np.float64)
    got = gpu(plan, (20, 24, 40), [x])[0]
    # The layer tests' tolerance, in the outputs' scale, and half its own step
    # (2^-149) of each subnormal input, twice.
    step = 2.0 ** -149 * np.abs(wt.astype(np.float64)).sum(axis=(0, 1, 2)).max()
    assert (np.abs(got - want) <= 1e-5 * np.abs(want) + 1e-5 * sx * sw + step).all()


# A value and a weight whose nearest bf16 values' product is past f32's largest
# while their own product is not.
NEAR_X, NEAR_W = np.float32(1.004 * 2.0 ** 127), np.float32(1.9895)


def test_ctc_panel_near_overflow(oracle):
    """A logit within 2^-7 of f32's largest value: the class holds. (The
    probability does not: past 2^128 / log2(e) the exponent overflows.)"""
    rng = np.random.default_rng(5)
    w = rng.normal(0, 0.3, (48, 500)).astype(np.float32)
    w[9, 300], w[9, 20] = NEAR_W, NEAR_W * np.float32(0.9999)
    b = PlanBuilder(1, 40, 48)
    plan = b.to_bytes([b.ctcargmax(b.input, w, rng.normal(0, 0.5, 500).astype(np.float32))])
    x = rng.normal(0, 1, (1, 40, 48)).astype(np.float32)
    x[0, 21, 9] = NEAR_X
    got = gpu(plan, (1, 40, 48), [x])[0].reshape(-1, 2)
    want = oracle.OracleModel(plan).run(x)[0].reshape(-1, 2)
    assert want[21, 0] == 300 and np.array_equal(got[:, 0], want[:, 0])
    rest = np.arange(40) != 21
    np.testing.assert_allclose(got[rest, 1], want[rest, 1], rtol=1e-5)


def conv_plan(rng, h, w, cs, n, s, act, res):
    """A 3 x 3 window over one map of cs[0] channels and, upsampled by two,
    one of cs[1]; with an Add of its output and a 1 x 1 layer's when `res`."""
    b = PlanBuilder(h, w, 8)
    x = b.conv(b.input, rng.normal(0, 0.4, (1, 1, 8, cs[0])).astype(np.float32), None)
    ctot, up = sum(cs), None
    if len(cs) > 1:
        half = b.conv(b.input, rng.normal(0, 0.2, (2, 2, 8, cs[1])).astype(np.float32), None, k=(2, 2), s=(2, 2))
        up = b.upsample(half, 2)
    wt = rng.normal(0, 1 / np.sqrt(9 * ctot), (3, 3, ctot, n)).astype(np.float32)
    y = b.conv(x, wt, rng.normal(0, 0.3, n).astype(np.float32), k=(3, 3), s=(s, s), pad=(1, 1, 1, 1), x2=up, fused=act)
    if res:
        r = b.conv(b.input, rng.normal(0, 0.4, (1, 1, 8, n)).astype(np.float32), None, s=(s, s))
        y = b.add(y, r, fused="relu")
    return b.to_bytes([y])


# Tiles of 4, 8 and 16 rows (few tiles, more, enough for 160 of 16 rows over
# the lanes), edges that cut them, channels within and past a block of 32, 17
# to 32 outputs, both strides, two sources, a folded Add; 8 channels run in f32.
@pytest.mark.parametrize("h,w,cs,n,s,act,res", [
    (1, 1, (8,), 17, 1, "none", False), (1, 1, (16,), 17, 1, "none", False), (5, 17, (40,), 24, 1, "hardswish", True), (33, 31, (96,), 32, 1, "relu", False),
    (66, 130, (32, 24), 24, 1, "relu", True), (150, 220, (24, 72), 20, 1, "none", False),
    (7, 9, (48,), 32, 2, "hardswish", False), (64, 66, (16, 16), 25, 2, "relu", True)])
def test_conv_patch_split(oracle, h, w, cs, n, s, act, res):
    rng = np.random.default_rng(h + w)
    plan = conv_plan(rng, h, w, cs, n, s, act, res)
    xs = [rng.uniform(-1, 1, (h, w, 8)).astype(np.float32) for _ in range(3)]
    m = oracle.OracleModel(plan)
    for x, got in zip(xs, gpu(plan, (h, w, 8), xs)):
        want = m.run(x)[0].reshape(-1).astype(np.float64)
        # The layer tests' tolerance for sums in another order.
        assert (np.abs(got - want) <= 1e-5 * np.abs(want) + 1e-5).all()


def test_conv_patch_split_odd_values(oracle):
    """An infinity or NaN reaches the outputs its window covers as it does in
    f32, and no others."""
    rng = np.random.default_rng(8)
    b = PlanBuilder(20, 24, 16)
    wt = rng.normal(0, 0.1, (3, 3, 16, 24)).astype(np.float32)
    plan = b.to_bytes([b.conv(b.input, wt, None, k=(3, 3), pad=(1, 1, 1, 1))])
    x = rng.uniform(-1, 1, (20, 24, 16)).astype(np.float32)
    y = x.copy()
    y[3, 4, 5], y[10, 20, 2], y[17, 1, 15], y[14, 10, 0] = np.inf, -np.inf, np.nan, 3.4e38
    a, c = (v.reshape(20, 24, 24) for v in gpu(plan, (20, 24, 16), [x, y]))
    want = oracle.OracleModel(plan).run(y)[0].reshape(20, 24, 24)
    far = np.ones((20, 24), bool)
    for py, px in ((3, 4), (10, 20), (17, 1), (14, 10)):
        far[max(py - 1, 0):py + 2, max(px - 1, 0):px + 2] = False
    assert np.array_equal(a[far].view(np.uint32), c[far].view(np.uint32))
    assert np.array_equal(np.isnan(c), np.isnan(want)) and np.array_equal(np.isinf(c), np.isinf(want))
    assert np.array_equal(c[np.isinf(c)], want[np.isinf(want)])
    fin = np.isfinite(want)
    np.testing.assert_allclose(c[fin], want[fin], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("s", [1, 2])
def test_conv_patch_split_near_overflow(oracle, s):
    """An output within 2^-7 of f32's largest value stays finite, its
    neighbours keep their bits."""
    rng = np.random.default_rng(9)
    b = PlanBuilder(20, 24, 24)
    wt = rng.normal(0, 0.1, (3, 3, 24, 24)).astype(np.float32)
    wt[1, 1, 3, 20] = NEAR_W
    plan = b.to_bytes([b.conv(b.input, wt, None, k=(3, 3), s=(s, s), pad=(1, 1, 1, 1))])
    x = rng.uniform(-1, 1, (20, 24, 24)).astype(np.float32)
    y = x.copy()
    y[8, 10, 3], y[18, 2, 3] = NEAR_X, -NEAR_X
    want = oracle.OracleModel(plan).run(y)[0].reshape(20 // s, 24 // s, 24)
    a, c = (v.reshape(want.shape) for v in gpu(plan, (20, 24, 24), [x, y]))
    assert np.isfinite(want).all() and want[8 // s, 10 // s, 20] > 3.3e38 and want[18 // s, 2 // s, 20] < -3.3e38
    # Sums in another order: 1e-5 of the largest product.
    np.testing.assert_allclose(c, want, rtol=1e-5, atol=1e-5)
    far = np.ones(want.shape[:2], bool)
    for py, px in ((8, 10), (18, 2)):
        far[(py - 1) // s:(py + 1) // s + 1, (px - 1) // s:(px + 1) // s + 1] = False
    assert np.array_equal(a[far].view(np.uint32), c[far].view(np.uint32))


@pytest.mark.parametrize("c,n,s,split", [(8, 24, 1, False), (16, 16, 1, False), (16, 17, 1, True), (24, 32, 1, True),
                                         (24, 33, 1, False), (96, 24, 1, True), (16, 24, 2, False), (24, 17, 2, True),
                                         (48, 32, 2, True)])
def test_conv_patch_split_rule(c, n, s, split):
    """Which layers run split: not channels so few that padding them to 32
    costs more than the products save."""
    b = PlanBuilder(20, 24, c)
    wt = np.zeros((3, 3, c, n), np.float32)
    g = GpuModel.load(b.to_bytes([b.conv(b.input, wt, None, k=(3, 3), s=(s, s), pad=(1, 1, 1, 1))]))
    names = [name for name, _ in g.launches()]
    g.close()
    assert names == ["conv_patch_split" if split else "conv_patch"]


@pytest.mark.parametrize("h,w,lanes,s", [(1, 352, 8, 1), (4, 352, 8, 1), (8, 300, 5, 1), (9, 150, 16, 1), (51, 130, 8, 1),
                                         (143, 254, 1, 1), (3, 5, 1, 2), (65, 31, 9, 2), (112, 160, 16, 2)])
def test_conv_patch_split_tiles(oracle, h, w, lanes, s):
    """Maps of few rows and of rows either side of a tile's, with as many tiles
    as take one round of the CUs and more: a lane's bits are those of the lane
    alone, whichever tiles each takes."""
    rng = np.random.default_rng(h)
    b = PlanBuilder(h, w, 40)
    wt = rng.normal(0, 0.06, (3, 3, 40, 24)).astype(np.float32)
    plan = b.to_bytes([b.conv(b.input, wt, None, k=(3, 3), s=(s, s), pad=(1, 1, 1, 1), fused="relu")])
    xs = [rng.uniform(-1, 1, (h, w, 40)).astype(np.float32) for _ in range(lanes)]
    got = gpu(plan, (h, w, 40), xs)
    m = oracle.OracleModel(plan)
    for i in (0, lanes - 1):
        assert np.array_equal(gpu(plan, (h, w, 40), [xs[i]])[0].view(np.uint32), got[i].view(np.uint32))
        want = m.run(xs[i])[0].reshape(-1).astype(np.float64)
        assert (np.abs(got[i] - want) <= 1e-5 * np.abs(want) + 1e-5).all()
