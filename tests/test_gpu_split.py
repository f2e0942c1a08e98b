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
# four, whole and not; one column, one tile, tiles that do not fill a run; and
# (4160 rows, 48 tiles) enough workgroups that each walks whole runs.
@pytest.mark.parametrize("lanes,t,c,vocab", [(1, 1, 4, 1), (1, 5, 32, 64), (3, 43, 36, 65), (1, 128, 64, 400),
                                             (2, 80, 128, 385), (26, 160, 100, 3050)])
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
    assert b[11, 0] == want[11, 0]
    np.testing.assert_allclose(b[11, 1], want[11, 1], rtol=1e-5)
