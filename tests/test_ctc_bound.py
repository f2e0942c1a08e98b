"""The near-tie bound of the CTC merge (ctc_merge in csrc/gemm.hip).

A column's logit is its bias plus ci products (src/engine/layers.rs:770-776:
the bias, then one fused multiply-add per input in order). Any order that
rounds once per addition lies within n u T of the exact sum, n = ci + 1,
u = 2^-24, T = |bias| + sum |w_i x_i|; so two orders lie within 2 n u T of
each other, and the merge, which needs two columns' differences (4 n u T),
tests against 8 n u T with T bounded by bias_max + wsum_max * max |x_i|.
These checks hold the error of several orders (the CPU's chain, its
reverse, random orders, and blocks of four products added together as an
MFMA step does) to n u T on inputs with heavy cancellation, against exact
sums, so a bound written too tight fails here."""
import math

import numpy as np
import pytest

U = 2.0 ** -24


def chain(bias, w, x, order):
    """One rounding per step: v = round(v + w_i x_i), the product exact."""
    v = np.float32(bias)
    for i in order:
        v = np.float32(float(v) + float(w[i]) * float(x[i]))
    return float(v)


def blocks_of_four(bias, w, x):
    """Each step adds four exact products at once (one rounding), the bias last."""
    v = 0.0
    for i in range(0, len(w), 4):
        v = float(np.float32(v + math.fsum(float(w[j]) * float(x[j]) for j in range(i, min(i + 4, len(w))))))
    return float(np.float32(v + float(bias)))


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_orders_within_bound(seed):
    rng = np.random.default_rng(seed)
    ci = 120
    n = ci + 1
    worst = 0.0
    for trial in range(60):
        x = rng.normal(0, rng.choice([0.5, 3.0]), ci).astype(np.float32)
        w = rng.normal(0, 0.05, ci).astype(np.float32)
        if trial % 3 == 0:  # heavy cancellation: the products sum to about zero
            p = w.astype(np.float64) * x.astype(np.float64)
            w[-1] = np.float32(-(p[:-1].sum()) / float(x[-1])) if x[-1] != 0 else w[-1]
        bias = np.float32(rng.normal(0, 0.5))
        exact = math.fsum([float(bias)] + [float(a) * float(b) for a, b in zip(w, x)])
        T = abs(float(bias)) + sum(abs(float(a) * float(b)) for a, b in zip(w, x))
        orders = [range(ci), range(ci - 1, -1, -1)] + [rng.permutation(ci) for _ in range(3)]
        got = [chain(bias, w, x, o) for o in orders] + [blocks_of_four(bias, w, x)]
        for g in got:
            err = abs(g - exact)
            assert err <= n * U * T * (1 + 1e-6), (trial, err, n * U * T)
            worst = max(worst, err / (n * U * T))
        # Two orders: within 2 n u T of each other, a quarter of the merge's test.
        assert max(got) - min(got) <= 2 * n * U * T * (1 + 1e-6)
    assert worst > 0.0


def test_merge_bound_covers_column_bounds():
    # T of a row's column is at most bias_max + wsum_max * max |x_i|, the
    # per-model bounds the merge is given.
    rng = np.random.default_rng(7)
    ci, vocab = 120, 300
    w = rng.normal(0, 0.05, (ci, vocab)).astype(np.float32)
    bias = rng.normal(0, 0.5, vocab).astype(np.float32)
    bias_max = float(np.abs(bias).max())
    wsum_max = float(np.abs(w.astype(np.float64)).sum(axis=0).max())
    for _ in range(20):
        x = rng.normal(0, 2.0, ci).astype(np.float32)
        T = np.abs(bias.astype(np.float64)) + np.abs(w.astype(np.float64) * x[:, None]).sum(axis=0)
        assert T.max() <= bias_max + wsum_max * float(np.abs(x).max())


def parts(v):
    """The three bf16 parts of a float32 at scales 1, 2^-8 and 2^-16, whose
    sum it is."""
    out = []
    v = np.float32(v)
    for _ in range(3):
        u = int(v.view(np.uint32))
        u = (u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000
        out.append(np.uint32(u).view(np.float32))
        v = (v - out[-1]) * np.float32(256)
    assert v == 0
    return [float(p) for p in out]


@pytest.mark.parametrize("ci", [4, 32, 120])
def test_split_order_within_bound(ci):
    """The panel kernel's order: six products of bf16 parts, an accumulator
    for each of their three scales, every addition rounded (to nearest or
    toward zero): within (1.04 ci + 4) u T, twice the first toward zero."""
    rng = np.random.default_rng(ci)
    for trial in range(20):
        x = rng.normal(0, 3, ci).astype(np.float32)
        w = rng.normal(0, 0.3, ci).astype(np.float32)
        if trial % 2:  # heavy cancellation
            w[-1] = np.float32(-(w[:-1].astype(np.float64) * x[:-1]).sum() / float(x[-1]))
        bias = np.float32(rng.normal(0, 0.5))
        exact = math.fsum([float(bias)] + [float(a) * float(b) for a, b in zip(w, x)])
        T = abs(float(bias)) + sum(abs(float(a) * float(b)) for a, b in zip(w, x))
        for toward_zero in (False, True):
            def add(v, t):
                s = np.float32(v + t)
                if toward_zero and abs(float(s)) > abs(v + t):
                    s = np.nextafter(s, np.float32(0))
                return float(s)
            acc = [0.0, 0.0, 0.0]
            for a, b in zip(w, x):
                p, q = parts(a), parts(b)
                for i, j in ((2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)):
                    acc[i + j] = add(acc[i + j], p[i] * q[j])
            low = float(np.float32(acc[1] + acc[2] / 256))
            got = float(np.float32(np.float32(acc[0] + low / 256) + bias))
            assert abs(got - exact) <= (1.04 * ci * (1 + toward_zero) + 4) * U * T


@pytest.mark.parametrize("e", [-149, -140, -134, -126, -120, -110, -60, 0, 120])
def test_split_parts_exact(e):
    """The parts are the value, down to f32's smallest."""
    rng = np.random.default_rng(e + 200)
    for v in np.float32(rng.uniform(1, 2, 200) * 2.0 ** e) * rng.choice([-1, 1], 200).astype(np.float32):
        p = parts(v)
        assert p[0] + p[1] / 256 + p[2] / 65536 == float(v)
