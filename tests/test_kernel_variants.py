"""Kernel variants that the planner chooses by size, layout or neighbouring operations, each at the sizes
where it can go wrong: compared with the CPU oracle, or with the float64 formula where stated."""
import numpy as np
import pytest

from accy_amd import hip
from accy_amd import tensor as T
from accy_amd import workloads as W
from conftest import assert_rel, hip_run, oracle_run, to_f32

F32 = T.Type("f32", ())


# ---- reductions that share a pass over their row, folds that share a launch ----

def statistics(b, a):
    """Three passes: max | two sums that read it | a sum that reads one of them; and a free sum and a
    minimum that belong to the first pass."""
    x = a[0]
    m = x.max("c")
    e = x.sub(m).exp()
    s = e.sum("c")
    p = e.div(s)
    return [m, s, x.sub(m).sum("c"), p.mul(x).sum("c"), x.mul(x).sum("c"), x.min("c"), p]


@pytest.mark.parametrize("rows,cols,passes", [(3, 16, None), (5, 64, 4), (1500, 68, 4), (7, 257, 4), (2, 9000, 4)])
def test_independent_reductions_share_a_pass(rows, cols, passes):
    src = hip.plan_source(T.define("stats", [T.spec("f32", r=rows, c=cols)], statistics))
    if passes:   # one element loop per dependency level, and one for the full row
        assert src.count("__global__") == 1 and src.count("for (int e = 0;") == passes


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("rows,cols", [(3, 16), (5, 64), (1500, 68), (7, 257), (2, 9000)])
def test_shared_passes_match_the_oracle(rows, cols, dtype):
    prog = T.define("stats", [T.spec(dtype, r=rows, c=cols)], statistics)
    # values away from zero, so that no sum cancels: per element within the reductions' 1e-5 (one
    # rounding step of the 16-bit result in those types, which an f32 sum in another order can move)
    x = W.to_dtype(1.0 + np.abs(W.normal(rows * cols, rows * cols)), dtype).reshape(rows, cols)
    tol = {"f32": 1e-5, "bf16": 2.0 ** -6, "f16": 2.0 ** -9}[dtype]
    for got, ref in zip(hip_run(prog, [x]), oracle_run(prog, [x])):
        g, r = to_f32(got, dtype).astype(np.float64), to_f32(ref, dtype).astype(np.float64)
        assert np.all(np.abs(g - r) <= tol * np.maximum(np.abs(r), np.abs(r).max() * 1e-2))


def folds(b, a):
    """Leading-axis folds: two that share a launch, one that reads a fold's result, one over another axis."""
    x = a[0]
    s = x.sum("r")
    return [s, x.mul(x).sum("r"), x.sub(s).max("r"), x.sum("c")]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "i32"])
@pytest.mark.parametrize("r,c", [(1, 1), (17, 33), (300, 77)])
def test_folds_that_share_a_launch_keep_their_order(r, c, dtype):
    prog = T.define("folds", [T.spec(dtype, r=r, c=c)], folds)
    assert "&%" in hip.plan_source(prog)
    rng = np.random.default_rng(r)
    x = (rng.standard_normal((r, c)) * 100).astype(np.float32 if dtype == "f32" else np.int32)
    got, ref = hip_run(prog, [x]), oracle_run(prog, [x])
    for g, f in list(zip(got, ref))[:3]:
        assert np.array_equal(g, f)     # serial left-to-right folds: bit for bit


@pytest.mark.gpu
def test_sine_and_cosine_of_one_value_against_float64():
    """The pair shares one reduction: each within 2 ulp of float64 below 2^17, the library's beyond,
    sin(-0) = -0, cos(0) = 1, NaN for infinities and NaN."""
    rng = np.random.default_rng(3)
    near = (np.arange(-4000, 4001) * (np.pi / 4)).astype(np.float32)
    x = np.concatenate([np.linspace(-20, 20, 20001), rng.uniform(-2.0 ** 17, 2.0 ** 17, 40000), near,
                        np.nextafter(near, np.float32(np.inf)), np.geomspace(1e-30, 1, 2000),
                        -np.geomspace(1e-30, 1, 2000), [1e6, -3.5e7, 1e30]]).astype(np.float32)
    xs = np.concatenate([x, np.array([np.inf, -np.inf, np.nan, -0.0, 0.0], np.float32)])
    prog = T.define("pair", [T.spec("f32", i=len(xs))], lambda b, a: [a[0].sin(), a[0].cos()])
    assert "sin_with_cos_f32" in hip.plan_source(prog)
    for got, f64 in zip(hip_run(prog, [xs]), (np.sin, np.cos)):
        ref = f64(x.astype(np.float64))
        ulp = np.spacing(np.abs(ref).astype(np.float32)).astype(np.float64)
        assert (np.abs(got[:len(x)].astype(np.float64) - ref) / ulp).max() <= 2.0
        assert np.isnan(got[len(x):len(x) + 3]).all()
    s, c = hip_run(prog, [xs])
    assert np.signbit(s[-2]) and s[-2] == 0 and s[-1] == 0 and not np.signbit(s[-1]) and c[-2] == c[-1] == 1.0
