"""Kernel variants that the planner chooses by size, layout or neighbouring operations, each at the sizes
where it can go wrong: compared with the CPU oracle, or with the float64 formula where stated."""
import re
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from accy_amd import hip
from accy_amd import tensor as T
from accy_amd import workloads as W
from conftest import exact_attention, hip_run, oracle_run, to_f32

F32 = T.Type("f32", ())


def work_items(prog):
    """Work items along the first grid dimension of every kernel of a plan."""
    return [int(g) * int(b) for g, b in re.findall(r"^ *// .* grid (\d+) block (\d+)$", hip.plan_source(prog), re.M)]


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
        loops = max(src.count("for (int e = 0;"), src.count("const I cr ="))   # whole iterations, the last one
        assert src.count("__global__") == 1 and loops == passes


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


def sine_or_cosine(b, a):
    """Both of every element in one kernel: [sine, cosine] along a last axis."""
    n = a[0].ty.dims[0][1]
    first = b.iota("f32", "k", ("k", 2), ("i", n)).compare("lt", b.full_float(F32, 0.5))
    return first.select(a[0].sin(), a[0].cos())


def test_sines_share_a_reduction_only_with_a_cosine_beside_them():
    """In two kernels, or two passes of one, each evaluates its own: sin_f32 is the cheaper form alone."""
    spec = [T.spec("f32", r=64, i=4096)]
    for body in (lambda b, a: [a[0].sin(), a[0].cos()], lambda b, a: [a[0].sin().sum("i"), a[0].cos()],
                 lambda b, a: [a[0].sin().sum("r"), a[0].cos().sum("i")]):
        src = hip.plan_source(T.define("pair", spec, body))
        assert "sin_with_cos_f32" not in src and "sin_f32" in src and "cos_f32" in src
    for body in (lambda b, a: [a[0].sin().sum("i"), a[0].cos().sum("i")], lambda b, a: a[0].sin().mul(a[0].cos())):
        src = hip.plan_source(T.define("pair", spec, body))
        assert "sin_with_cos_f32" in src and "accy::sin_f32" not in src


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
    prog = T.define("pair", [T.spec("f32", i=len(xs))], sine_or_cosine)
    assert "sin_with_cos_f32" in hip.plan_source(prog)
    for got, f64 in zip(hip_run(prog, [xs])[0].T, (np.sin, np.cos)):
        ref = f64(x.astype(np.float64))
        ulp = np.spacing(np.abs(ref).astype(np.float32)).astype(np.float64)
        assert (np.abs(got[:len(x)].astype(np.float64) - ref) / ulp).max() <= 2.0
        assert np.isnan(got[len(x):len(x) + 3]).all()
    s, c = hip_run(prog, [xs])[0].T
    assert np.signbit(s[-2]) and s[-2] == 0 and s[-1] == 0 and not np.signbit(s[-1]) and c[-2] == c[-1] == 1.0


# ---- scatter_add: one pass over the table ----

def scatter(dtype, pre, ext, post, n, computed=False):
    dims = lambda k, e: [d for d in (("p", pre), (k, e), ("q", post)) if d[1]]

    def body(b, a):
        table, ids, up = a
        if computed:    # table and updates that no buffer holds
            table, up = table.add(table), up.mul(up)
        return table.scatter_add(ids, up, "k")
    return T.define("scatter", [T.spec(dtype, *dims("k", ext)), T.spec("i32", j=n), T.spec(dtype, *dims("j", n))], body)


# (pre, rows, row elements, updates): a row per workgroup column tile and tails of it; one element per
# row; fewer rows than a tile; several batches of hits on one row; several row tiles per workgroup
SCATTERS = [(0, 10, 0, 5), (0, 33, 7, 64), (3, 1001, 4, 513), (0, 37, 1028, 2500), (2, 5, 2052, 40), (0, 1, 12, 3000),
            (0, 5000, 3, 60000), (0, 9000, 64, 511), (0, 40000, 0, 30000)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SCATTERS, ids=str)
@pytest.mark.parametrize("dtype", ["f32", "i32", "bf16"])
def test_scatter_add_keeps_the_order_of_the_updates(shape, dtype):
    pre, ext, post, n = shape
    rng = np.random.default_rng(ext)
    # half of the indices on a few rows, some out of range (clamped)
    ids = np.where(rng.random(n) < 0.5, rng.integers(0, min(ext, 3), n), rng.integers(-2, ext + 2, n)).astype(np.int32)
    size = lambda e: [x for x in (pre, e, post) if x]

    def values(e):
        x = rng.standard_normal(size(e)) * 8
        return x.astype(np.int32) if dtype == "i32" else W.to_dtype(x, dtype)
    ins = [values(ext), ids, values(n)]
    for computed in (False, True):
        prog = scatter(dtype, pre, ext, post, n, computed)
        got, ref = hip_run(prog, ins)[0], oracle_run(prog, ins)[0]
        assert np.array_equal(got.view(np.uint8), ref.view(np.uint8))   # every sum rounded in order: bit for bit


# (positions before the axis, rows, row elements, updates): several positions per workgroup, with one element per row
# and tails of vectors; positions in turn and several batches of hits
POSITIONS = [(70001, 8, 0, 40), (66000, 5, 3, 33), (9001, 3, 260, 17), (5001, 512, 0, 14000)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", POSITIONS, ids=str)
def test_scatter_add_over_many_leading_positions(shape):
    pre, ext, post, n = shape
    prog = scatter("f32", pre, ext, post, n)
    src = hip.plan_source(prog)
    tc, kg, loop, ploop = (int(x) for x in re.search(r"TC = (\d+), KG = (\d+), LOOP = (\d+), PLOOP = (\d+)", src).groups())
    assert tc * kg < 256 or ploop > 1
    rng = np.random.default_rng(ext)
    ids = rng.integers(-1, ext + 1, n).astype(np.int32)
    size = lambda e: [x for x in (pre, e, post) if x]
    ins = [rng.random(size(ext), np.float32), ids, rng.random(size(n), np.float32)]
    assert np.array_equal(hip_run(prog, ins)[0], oracle_run(prog, ins)[0])   # every sum rounded in order: bit for bit


def test_scatter_add_of_short_rows_shares_its_lists_between_positions():
    """A workgroup for every leading position would read and sort the index list once for each."""
    assert max(work_items(scatter("f32", 1 << 20, 8, 0, 64))) <= (1 << 20) * 8 and max(work_items(scatter("f32", 1 << 20, 2, 4, 16))) <= (1 << 20) * 8


@pytest.mark.gpu
@pytest.mark.parametrize("width", [64, 63])
def test_scatter_add_of_gathered_updates(width):
    """Updates at a gathered row: their offsets read a temporary, so no vector load is hoisted."""
    def body(b, a):
        table, ids, rows, up = a
        return [table.scatter_add(ids, up.gather(rows, "u"), "k"), up.gather(rows, "u")]
    prog = T.define("gathered", [T.spec("f32", k=50, q=width), T.spec("i32", j=200), T.spec("i32", j=200),
                                 T.spec("f32", u=30, q=width)], body)
    rng = np.random.default_rng(8)
    ins = [rng.standard_normal((50, width)).astype(np.float32), rng.integers(0, 50, 200).astype(np.int32),
           rng.integers(0, 30, 200).astype(np.int32), rng.standard_normal((30, width)).astype(np.float32)]
    for got, ref in zip(hip_run(prog, ins), oracle_run(prog, ins)):
        assert np.array_equal(got, ref)


# ---- f32 contractions in staged tiles, split along K or not ----

def contraction(dtype, m, k, n, layout="NN", batch=0, epilogue=False):
    b_ = [("b", batch)] if batch else []
    sa = b_ + ([("m", m), ("k", k)] if layout[0] == "N" else [("k", k), ("m", m)])
    sb = b_ + ([("k", k), ("n", n)] if layout[1] == "N" else [("n", n), ("k", k)])

    def body(b, a):
        c = a[0].contract(a[1], "k")
        return c.mul(b.full_float(T.Type(dtype, ()), 0.5)).add(a[2]) if epilogue else c
    specs = [T.spec(dtype, *sa), T.spec(dtype, *sb)] + ([T.spec(dtype, n=n)] if epilogue else [])
    return T.define("contraction", specs, body)


def contraction_inputs(dtype, m, k, n, layout, batch, epilogue, seed):
    rng = np.random.default_rng(seed)
    b_ = (batch,) if batch else ()
    a, b = rng.standard_normal(b_ + (m, k)), rng.standard_normal(b_ + (k, n))
    a, b = to_f32(W.to_dtype(a, dtype), dtype).astype(np.float64), to_f32(W.to_dtype(b, dtype), dtype).astype(np.float64)
    bias = to_f32(W.to_dtype(rng.standard_normal(n), dtype), dtype).astype(np.float64)
    swap = lambda x, side: x if layout[side] == "N" else np.ascontiguousarray(np.swapaxes(x, -1, -2))
    ins = [W.to_dtype(np.ascontiguousarray(swap(a, 0)), dtype), W.to_dtype(np.ascontiguousarray(swap(b, 1)), dtype)]
    return ins + ([W.to_dtype(bias, dtype)] if epilogue else []), a, b, bias


# tile remainders on both sides, rows shorter than a vector, K below a vector / a step and past it,
# one output, one row, few rows (splits), batches
F32_SHAPES = [(1, 128, 1, 0), (1, 4096, 300, 0), (3, 129, 2, 0), (31, 1023, 66, 0), (33, 130, 65, 0), (127, 131, 129, 0),
              (962, 133, 130, 0), (3000, 3, 1001, 0), (2900, 1, 2899, 0), (64, 5000, 64, 0), (300, 2050, 70, 0),
              (513, 1030, 770, 0), (5, 200, 37, 7), (130, 256, 66, 3), (3, 1129, 2, 0), (33, 1130, 65, 0),
              (127, 1131, 129, 0), (5, 1200, 37, 7)]
# of these, folded by one thread per output (serial k order, within the same bound)
F32_FOLDED = {(3, 129, 2, 0), (33, 130, 65, 0), (127, 131, 129, 0), (2900, 1, 2899, 0), (5, 200, 37, 7)}


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("shape", F32_SHAPES, ids=str)
def test_staged_f32_contractions_within_the_summation_bound(shape, layout):
    """|error| <= (K + 2) u sum|a b| for a sum of K products in any order (u = 2^-24), doubled for the
    epilogue's product and sum."""
    m, k, n, batch = shape
    for epilogue in (False, True):
        prog = contraction("f32", m, k, n, layout, batch, epilogue)
        assert ("WAVES_K" in hip.plan_source(prog)) == (shape not in F32_FOLDED)
        ins, a, b, bias = contraction_inputs("f32", m, k, n, layout, batch, epilogue, m + k)
        got = hip_run(prog, ins)[0].astype(np.float64)
        ref, size = a @ b, np.abs(a) @ np.abs(b)
        if epilogue:
            ref, size = ref * 0.5 + bias, size + 2 * np.abs(bias)
        assert np.all(np.abs(got - ref) <= 2 * (k + 2) * 2.0 ** -24 * size)


def test_f32_contractions_choose_their_kernel_by_size():
    plan = lambda m, k, n: hip.plan_source(contraction("f32", m, k, n))
    assert "WAVES_K" not in plan(8192, 8192, 8192) and "mma32f<" in plan(8192, 8192, 8192)   # whole rounds of 256-wide tiles
    assert "BM = 128" in plan(2048, 2048, 2048) and "SPLITS = 1" in plan(2048, 2048, 2048)
    assert "BM = 64" in plan(1000, 1000, 1000) and "SPLITS = 1" in plan(1000, 1000, 1000)
    assert "BM = 32" in plan(16, 4096, 4096) and "split_sum" in plan(16, 4096, 4096)
    assert "accy::gemm::" not in plan(200, 100, 200)
    for layout in ("NT", "TN", "TT"):    # the staged kernel reads every layout, the direct one needs A along K and B along N
        assert "pack" not in hip.plan_source(contraction("f32", 2048, 2048, 2048, layout))
        assert "pack" in hip.plan_source(contraction("f32", 8192, 8192, 8192, layout))
    hip.plan_source(contraction("f32", 16, 4096, 4096, epilogue=True), compile=True)


@pytest.mark.parametrize("dtype,shape,folded", [
    ("f32", (4, 128, 4, 65535), True), ("f32", (1 << 22, 4, 4, 0), True), ("f32", (1 << 20, 16, 8, 0), True),
    ("f32", (1, 256, 1, 60000), True), ("f32", (2, 130, 3, 0), True), ("f32", (128, 128, 128, 0), False),
    ("f32", (20000, 130, 9, 0), False), ("f32", (33, 130, 33, 1000), False), ("f32", (1, 1000000, 1, 0), False),
    ("bf16", (4, 128, 4, 65535), True), ("bf16", (1 << 22, 4, 4, 0), True), ("bf16", (3000000, 3, 3, 0), True),
    ("bf16", (2, 130, 3, 0), False), ("bf16", (50, 130, 50, 1000), False), ("bf16", (20000, 130, 9, 0), False)])
def test_contractions_that_leave_tiles_empty_are_folded(dtype, shape, folded):
    m, k, n, batch = shape
    assert ("accy::gemm::" not in hip.plan_source(contraction(dtype, m, k, n, "NN", batch))) == folded


def test_small_contractions_spelled_as_products_and_sums():
    """Summed over a middle axis their other form is a fold, a thread per output as for a contraction; over the last axis
    a row kernel."""
    def spelled(m, k, n, last):
        shape = [("m", m), ("n", n), ("k", k)] if last else [("m", m), ("k", k), ("n", n)]
        def body(b, a):
            return b.broadcast_in_dim(a[0], shape, [0, 2] if last else [0, 1]).mul(b.broadcast_in_dim(a[1], shape, [1, 2])).sum("k")
        return hip.plan_source(T.define("mulsum", [T.spec("f32", m=m, k=k), T.spec("f32", n=n, k=k) if last else T.spec("f32", k=k, n=n)], body))
    for m, k, n, middle, last in [(127, 131, 129, False, False), (33, 130, 65, False, False), (300, 300, 300, True, True), (64, 2000, 64, True, False)]:
        assert ("accy::gemm::" in spelled(m, k, n, False)) == middle and ("accy::gemm::" in spelled(m, k, n, True)) == last


# ---- rows whose length is no multiple of four, or that the threads' vectors do not cover exactly ----

def softmax_rows(b, a):
    x, gain, bias = a
    e = x.sub(x.max("c")).exp()
    p = e.div(e.sum("c"))
    return [p.mul(gain).add(bias), x.mul(x).sum("c"), p.max("c")]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("rows,cols", [(3, 65), (1100, 67), (1030, 258), (5, 510), (4, 513), (2, 2047), (1, 30001), (2, 50000)])
def test_ragged_rows_match_the_oracle(rows, cols, dtype):
    """A row input, a vector broadcast over the rows, a scalar broadcast over the columns, a whole-row
    output. Sums of positive terms in another order: 1e-5 of the value in f32; one rounding step of each of
    the 16-bit operations that read such a sum (division, product, sum)."""
    prog = T.define("ragged", [T.spec(dtype, r=rows, c=cols), T.spec(dtype, c=cols), T.spec(dtype, r=rows)], softmax_rows)
    assert hip.plan_source(prog).count("__global__") == 1
    rng = np.random.default_rng(cols)
    ins = [W.to_dtype(x, dtype) for x in (rng.standard_normal((rows, cols)), 1 + rng.random(cols), 1 + rng.random(rows))]
    tol = {"f32": 1e-5, "bf16": 3 * 2.0 ** -7, "f16": 3 * 2.0 ** -10}[dtype]
    for got, ref in zip(hip_run(prog, ins), oracle_run(prog, ins)):
        g, r = to_f32(got, dtype).astype(np.float64), to_f32(ref, dtype).astype(np.float64)
        assert np.all(np.abs(g - r) <= tol * np.abs(r))


def test_ragged_rows_choose_vectors_by_length():
    rows = lambda cols, body: hip.plan_source(T.define("rows", [T.spec("f32", r=5000, c=cols)], body))
    softmax = lambda b, a: a[0].sub(a[0].max("c")).exp().sum("c")
    for cols, vectors in [(255, False), (257, True), (321, False), (385, False), (511, False), (514, True)]:
        assert ("const I cr =" in rows(cols, softmax)) == vectors
    assert "const I cr =" in rows(385, lambda b, a: a[0].sum("c"))     # one pass


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,threads", [(1, 100003, 1024), (3, 80000, 1024), (256, 2050, 512), (9, 1030, 256), (257, 2050, 128)])
def test_few_rows_take_more_threads(rows, cols, threads):
    """Against float64. A thread adds at most cols / threads + 4 positive terms in a chain, the tree 10 more and the
    exponential 2 ulp: 1e-5 relative holds up to 140 roundings."""
    def body(b, a):
        x = a[0]
        m = x.max("c")
        return [x.mul(x).sum("c"), m.add(x.sub(m).exp().sum("c").log()), m]
    prog = T.define("few", [T.spec("f32", r=rows, c=cols)], body)
    assert f" block {threads}\n" in hip.plan_source(prog)
    x = (1.0 + np.abs(W.normal(cols, rows * cols))).astype(np.float32).reshape(rows, cols)
    x64 = x.astype(np.float64)
    ref = [(x64 * x64).sum(1), x64.max(1) + np.log(np.exp(x64 - x64.max(1, keepdims=True)).sum(1)), x64.max(1)]
    for got, r in zip(hip_run(prog, [x]), ref):
        assert np.all(np.abs(got - r) <= 1e-5 * r)


def norm_backward(dtype):
    """Three values of the row, the gradient and two inputs, live between its passes."""
    def body(b, a):
        x, g, w = a
        inv = b.full_float(T.Type(dtype, ()), 1.0 / 256)   # any constant does: each side computes the same
        rs = x.mul(x).sum("c").mul(inv).sqrt()
        xh, gw = x.div(rs), g.mul(w)
        return gw.sub(xh.mul(gw.mul(xh).sum("c").mul(inv))).div(rs)
    return body


def norm_backward_program(rows, cols, dtype):
    return T.define("norm", [T.spec(dtype, r=rows, c=cols)] * 2 + [T.spec(dtype, c=cols)], norm_backward(dtype))


def test_rows_of_gradients_choose_threads_and_waves_by_registers():
    """Threads per row, whether the kernel asks for four waves per SIMD, whether each pass computes its own offsets."""
    softmax = lambda rows, cols, dtype: T.define("softmax", [T.spec(dtype, r=rows, c=cols)] * 2, lambda b, a: (
        lambda p: p.mul(a[1].sub(p.mul(a[1]).sum("c"))))((lambda e: e.div(e.sum("c")))(a[0].sub(a[0].max("c")).exp())))
    moments = lambda rows, cols, dtype: T.define("moments", [T.spec(dtype, r=rows, c=cols)], lambda b, a: [
        a[0].sum("c"), a[0].mul(a[0]).sum("c"), a[0].max("c")])
    for prog, threads, waves, offsets in [
            (norm_backward_program(3000, 32000, "f32"), 512, False, True), (norm_backward_program(1500, 16384, "f32"), 256, False, False),
            (norm_backward_program(1000, 20000, "bf16"), 512, True, True), (norm_backward_program(1000, 9000, "f32"), 256, True, True),
            (softmax(1000, 12288, "f32"), 256, True, True), (softmax(1500, 16384, "f32"), 256, False, False),
            (softmax(2000, 16000, "bf16"), 256, False, True), (softmax(3000, 24000, "bf16"), 512, True, True),
            (moments(500, 32000, "f32"), 512, False, False), (moments(600, 6000, "f32"), 256, False, False),
            (moments(600, 3000, "f32"), 128, False, False), (moments(2000, 16384, "f32"), 128, False, False)]:
        src = hip.plan_source(prog)
        assert f" block {threads}\n" in src and ("amdgpu_waves_per_eu(4)" in src) == waves and ("+ t0;" in src) == offsets


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,dtype", [(3, 16384, "f32"), (3, 32000, "f32"), (300, 9000, "f32"), (300, 16000, "bf16"), (300, 20000, "bf16")])
def test_rows_of_gradients_match_float64(rows, cols, dtype):
    """Positive inputs. f32: the sums are read from 1e-5 (their order) and the result cancels to a third of its terms
    at most, six roundings of each: 4e-5 of the larger term. 16 bits: ten operations that round to 2^-8."""
    prog = norm_backward_program(rows, cols, dtype)
    ins = [W.to_dtype(1.0 + np.abs(W.normal(i, n)), dtype).reshape(s) for i, (n, s) in enumerate([(rows * cols, (rows, cols))] * 2 + [(cols, (cols,))])]
    x, g, w = (to_f32(i, dtype).astype(np.float64).reshape(i.shape) for i in ins)
    inv = 1.0 / 256
    rs = np.sqrt((x * x).sum(1, keepdims=True) * inv)
    sub = x / rs * ((g * w * x / rs).sum(1, keepdims=True) * inv)
    got = to_f32(hip_run(prog, ins)[0], dtype).astype(np.float64).reshape(rows, cols)
    bound = {"f32": 4e-5, "bf16": 10 * 2.0 ** -8}[dtype]
    assert np.all(np.abs(got - (g * w - sub) / rs) <= bound * (g * w + np.abs(sub)) / rs)


@pytest.mark.gpu
def test_ragged_rows_write_only_their_own_elements():
    """Exact integer rows of 67 and 70 next to each other: every element of the full-row output, and the
    sums, bit for bit."""
    for rows, cols in [(1, 67), (1300, 67), (9, 70), (3, 4099)]:
        prog = T.define("rows", [T.spec("i32", r=rows, c=cols)], lambda b, a: [a[0].sub(a[0].sum("c")), a[0].max("c")])
        x = np.random.default_rng(cols).integers(-1000, 1000, (rows, cols)).astype(np.int32)
        for got, ref in zip(hip_run(prog, [x]), oracle_run(prog, [x])):
            assert np.array_equal(got, ref)


# ---- 16-bit contractions straight to LDS: tiles by size, K split, K past the last whole step ----

# (m, k, n, layout, batch): K steps that K does not fill for every layout; rows of any number where the operand
# is K-contiguous; one row; splits; batches
DMA_SHAPES = [(1, 136, 8, "NN", 0), (1, 4096, 1024, "NN", 0), (3, 1000, 264, "NN", 0), (129, 1000, 135, "NT", 0),
              (136, 1001, 264, "TN", 0), (128, 129, 128, "TN", 0), (264, 159, 520, "TN", 0), (1000, 3000, 512, "NN", 0),
              (17, 2048, 8192, "NN", 0), (300, 4096, 304, "NT", 0), (256, 8192, 256, "TN", 0), (5, 264, 8, "NN", 3),
              (200, 456, 130, "NT", 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("shape", DMA_SHAPES, ids=str)
def test_direct_to_lds_contractions_within_the_summation_bound(shape, dtype):
    """|error| <= (K + 2) u sum|a b| for an f32 sum of exact products in any order (u = 2^-24), and the result's
    rounding (bf16 truncates: 2^-7; f16: 2^-11), once more per operation of the epilogue."""
    m, k, n, layout, batch = shape
    for epilogue in (False, True):
        prog = contraction(dtype, m, k, n, layout, batch, epilogue)
        assert "mma16_dma<" in hip.plan_source(prog)
        ins, a, b, bias = contraction_inputs(dtype, m, k, n, layout, batch, epilogue, m + k)
        got = to_f32(hip_run(prog, ins)[0], dtype).astype(np.float64)
        ref, size, r = a @ b, np.abs(a) @ np.abs(b), {"bf16": 2.0 ** -7, "f16": 2.0 ** -11}[dtype]
        bound = (k + 2) * 2.0 ** -24 * size + r * np.abs(ref)
        if epilogue:
            half = 0.5 * ref
            ref = half + bias
            bound = bound + r * (np.abs(half) + np.abs(ref) + bound)
        assert np.all(np.abs(got - ref) <= bound + 2.0 ** -24)


def test_partial_sums_do_not_keep_a_program_out_of_the_scratch_array():
    """A temporary of 510 MiB and a contraction that would split: 518 MiB with its partial sums, more than the
    512 MiB of accy_hip_invoke_device_scratch, so it is planned whole; half the rows split."""
    def prog(rows):
        def body(b, a):
            e = a[0].sub(a[0].max("k")).exp()
            return e.div(e.sum("k")).contract(a[1], "k")
        return T.define("wide", [T.spec("bf16", m=rows, k=32000), T.spec("bf16", k=32000, n=64)], body)
    assert "split_sum" in hip.plan_source(prog(4096)) and "split_sum" not in hip.plan_source(prog(8352))


def test_partial_folds_do_not_keep_a_program_out_of_the_scratch_array():
    """A temporary of 511.9 MiB and a fold whose chunks' partials are 256 KiB: planned in one launch; with half the
    rows, in chunks."""
    def prog(rows):
        def body(b, a):
            e = a[0].sub(a[0].max("k")).exp()
            return [e.div(e.sum("k")).contract(a[1], "k"), a[2].sum("r")]
        return T.define("wide", [T.spec("bf16", m=rows, k=32000), T.spec("bf16", k=32000, n=64), T.spec("f32", r=3000, c=2048)], body)
    assert "chunks grid" in hip.plan_source(prog(4096)) and "chunks grid" not in hip.plan_source(prog(8387))


# extents of no multiple of 8, K below one step and below a vector, shallow aligned rows, splits, batches
STAGED_SHAPES = [(1, 33, 1), (7, 65, 9), (130, 67, 131), (129, 1001, 255), (200, 64, 264), (33, 2049, 7), (1, 40, 1000),
                 (1100, 5, 1003), (16, 4097, 300), (3, 1030, 1887)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("shape", STAGED_SHAPES, ids=str)
def test_staged_16bit_contractions_within_the_summation_bound(shape, layout, dtype):
    """The bound of the direct-to-LDS contractions, for a plain and a batched contraction."""
    m, k, n = shape
    for batch in (0, 3):
        prog = contraction(dtype, m, k, n, layout, batch)
        src = hip.plan_source(prog)
        assert "mma16_staged<" in src or "mma16_dma<" in src
        ins, a, b, _ = contraction_inputs(dtype, m, k, n, layout, batch, False, m + k)
        got = to_f32(hip_run(prog, ins)[0], dtype).astype(np.float64)
        ref, r = a @ b, {"bf16": 2.0 ** -7, "f16": 2.0 ** -11}[dtype]
        assert np.all(np.abs(got - ref) <= (k + 2) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + r * np.abs(ref) + 2.0 ** -24)


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,layout", [(130, 1005, 136, "TN"), (131, 1005, 137, "NN"), (131, 1005, 137, "TT"), (9, 70, 11, "NT")])
def test_contraction_tail_ignores_what_lies_past_k(m, k, n, layout):
    """Infinities and NaN in the rows and columns that follow K in memory, or that the clamped loads
    repeat, do not reach other outputs: rows 0 and m - 1 of A and columns 0 and n - 1 of B are not finite,
    everything else is."""
    prog = contraction("bf16", m, k, n, layout)
    ins, a, b, _ = contraction_inputs("bf16", m, k, n, layout, 0, False, 4)
    clean = hip_run(prog, ins)[0]
    rows = ins[0] if layout[0] == "N" else ins[0].T
    cols = ins[1].T if layout[1] == "N" else ins[1]
    rows[0] = rows[-1] = 0x7f80      # +inf
    cols[0] = cols[-1] = 0x7fc0      # NaN
    got = hip_run(prog, ins)[0]
    assert np.array_equal(got[1:-1, 1:-1], clean[1:-1, 1:-1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,m,k,n,layout", [("bf16", 136, 1001, 264, "TN"), ("f16", 300, 1000, 264, "NN"), ("bf16", 300, 1000, 135, "NT"),
                                                ("bf16", 131, 1005, 137, "NN"), ("f16", 131, 1005, 137, "TT"), ("bf16", 9, 70, 11, "NT"),
                                                ("f32", 130, 1030, 66, "NN"), ("f32", 33, 1130, 65, "TT"), ("f32", 130, 1030, 66, "NT")])
def test_contraction_tail_repeats_nothing_that_is_infinite(dtype, m, k, n, layout):
    """The last element of K, which loads past the end repeat, is infinite in one row of A and one column of B;
    everything is positive, so those outputs are infinite (0 x inf, from an operand that is not cleared past K, would be
    NaN) and the rest as without."""
    prog = contraction(dtype, m, k, n, layout)
    ins, _, _, _ = contraction_inputs(dtype, m, k, n, layout, 0, False, 4)
    ins = [x & 0x7fff if dtype == "bf16" else np.abs(x) for x in ins]
    clean = to_f32(hip_run(prog, ins)[0], dtype)
    inf = 0x7f80 if dtype == "bf16" else np.inf
    (ins[0] if layout[0] == "N" else ins[0].T)[2, -1] = inf
    (ins[1] if layout[1] == "N" else ins[1].T)[-1, 3] = inf
    got = to_f32(hip_run(prog, ins)[0], dtype)
    hit = np.zeros((m, n), bool)
    hit[2], hit[:, 3] = True, True
    assert np.all(got[hit] == np.inf) and np.array_equal(got[~hit], clean[~hit])


def test_contractions_choose_their_tile_by_size():
    plan = lambda m, k, n, layout="NN": hip.plan_source(contraction("bf16", m, k, n, layout))
    assert "BM = 256, BN = 256" in plan(8192, 8192, 8192) and "SPLITS" not in plan(8192, 8192, 8192)
    assert "BM = 128, BN = 128" in plan(2048, 8192, 2048) and "BM = 128, BN = 128" in plan(2048, 3000, 2048, "TN")
    assert "SPLITS" in plan(256, 8192, 256) and plan(256, 8192, 256).count("__global__") == 2
    hip.plan_source(contraction("bf16", 136, 1001, 264, "TN"), compile=True)


@pytest.mark.parametrize("dtype,m,k,n", [("f32", 1 << 31, 34, 16), ("f32", 1 << 30, 2, 1), ("bf16", 1 << 31, 40, 16),
                                         ("bf16", 1 << 31, 8, 8), ("bf16", 1 << 31, 256, 8)])
def test_contractions_of_any_size_can_be_launched(dtype, m, k, n):
    """HIP refuses a launch of 2^32 work items: such a contraction runs on larger tiles or a grid-stride kernel."""
    assert max(work_items(contraction(dtype, m, k, n))) < 1 << 32
    assert max(work_items(contraction(dtype, n, k, m))) < 1 << 32


# ---- f32 attention of head dimension 64: key groups ----

# (heads, queries, keys, causal, waves, groups): fewer key blocks than groups, a last round that not every group
# takes part in, more keys than queries and fewer, every workgroup shape
F32_ATTENTION = [(1, 32, 32, False, 1, 1), (3, 32, 160, False, 1, 4), (2, 96, 96, True, 1, 4), (2, 128, 64, True, 1, 2),
                 (70, 128, 96, False, 2, 2), (72, 192, 192, True, 2, 2), (512, 128, 160, True, 4, 1), (520, 128, 32, False, 4, 1),
                 (9, 1056, 96, False, 1, 2), (513, 96, 64, True, 1, 1), (1030, 32, 288, False, 1, 2), (600, 64, 64, True, 2, 1),
                 (600, 64, 96, False, 2, 2), (70, 128, 544, True, 2, 4), (65, 192, 512, False, 2, 4), (129, 512, 544, True, 4, 2),
                 (512, 128, 512, False, 4, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", F32_ATTENTION, ids=str)
def test_f32_attention_key_groups(case):
    """Against float64, 1e-4 of the largest magnitude (as the fused f32 attention's other shapes)."""
    heads, queries, keys, causal, waves, groups = case
    specs = [T.spec("f32", head=heads, query=queries, dim=64)] + [T.spec("f32", head=heads, key=keys, dim=64)] * 2
    def body(b, a):
        q, k, v = a
        s = q.contract(k, "dim").mul(b.full_float(F32, 0.125))
        if causal:
            dims = [d for d in s.ty.dims if d[0] in ("query", "key")]
            s = b.iota("i32", "query", *dims).compare("ge", b.iota("i32", "key", *dims)).select(s, b.full_float(F32, -np.inf))
        e = s.sub(s.max("key")).exp()
        return e.div(e.sum("key")).contract(v, "key")
    prog = T.define("attention", specs, body)
    assert f"WAVES = {waves}, GROUPS = {groups};" in hip.plan_source(prog)
    rng = np.random.default_rng(queries + keys)
    ins = [rng.standard_normal((heads, n, 64)).astype(np.float32) for n in (queries, keys, keys)]
    exact = exact_attention(*ins, 0.125, causal, "f32")
    assert np.abs(hip_run(prog, ins)[0] - exact).max() <= 1e-4 * np.abs(exact).max()


# ---- folds of a long leading range: chunks over workgroups and waves ----

# (reduced, kept, and a kept axis before the reduced one): vectors of four outputs and single ones, one chunk,
# quarters that the chunk does not fill, a last chunk shorter than a quarter, one output
FOLDS = [(256, 512, 0), (257, 1110, 0), (1142, 1110, 0), (3000, 2048, 0), (131072, 1, 0), (40000, 4, 0), (300, 128, 5),
         (16387, 12, 2), (999, 6, 30), (513, 8193, 0), (1100, 8199, 0), (700, 2741, 3)]


def test_folds_choose_their_split_by_size():
    plan = lambda r, c: hip.plan_source(T.define("fold", [T.spec("f32", r=r, c=c)], lambda b, a: a[0].sum("r")))
    for r, c in [(300, 262143), (300, 262144), (600, 100000), (255, 4096)]:     # a thread per output
        assert "parts[" not in plan(r, c) and plan(r, c).count("__global__") == 1 and "unroll" not in plan(r, c)
    for r, c in [(256, 512), (260, 5001), (512, 256)]:                           # one launch of workgroups
        assert "parts[4]" in plan(r, c) and plan(r, c).count("__global__") == 1
    sines = hip.plan_source(T.define("fold", [T.spec("f32", r=300, c=30000)], lambda b, a: a[0].sin().sum("r")))
    assert sines.count("__global__") == 2                                        # a transcendental per element: more waves
    for r, c, parts in [(100000, 64, 4), (1142, 1110, 4), (4000, 30001, 1), (1000, 9001, 1), (1000, 5001, 4)]:
        assert f"parts[{parts}]" in plan(r, c) and plan(r, c).count("__global__") == 2
    assert "s < (I)256" in plan(100000, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", FOLDS, ids=str)
@pytest.mark.parametrize("dtype", ["f32", "bf16", "i32"])
def test_chunked_folds_of_a_leading_axis(shape, dtype):
    """A computed operand. Integers, max and min bit for bit; a float sum within (n - 1) u sum|x| of float64
    and the result's rounding (bf16 truncates: 2^-7)."""
    r, c, p = shape
    dims = ([("p", p)] if p else []) + [("r", r), ("c", c)]
    prog = T.define("folds", [T.spec(dtype, *dims)], lambda b, a: [a[0].neg().sum("r"), a[0].max("r"), a[0].neg().min("r")])
    assert f"parts[{1 if c * max(p, 1) > 8192 and r > 512 else 4}]" in hip.plan_source(prog)
    rng = np.random.default_rng(r)
    x = rng.standard_normal([e for _, e in dims]) * 100
    x = x.astype(np.int32) if dtype == "i32" else W.to_dtype(x, dtype)
    got, ref = hip_run(prog, [x]), oracle_run(prog, [x])
    assert np.array_equal(got[1], ref[1]) and np.array_equal(got[2], ref[2])
    if dtype == "i32":
        assert np.array_equal(got[0], ref[0])
        return
    x64 = to_f32(x, dtype).astype(np.float64)
    exact, size = -x64.sum(-2), np.abs(x64).sum(-2)
    bound = (r - 1) * 2.0 ** -24 * size
    assert np.all(np.abs(to_f32(got[0], dtype) - exact) <= bound + (2.0 ** -7 * (np.abs(exact) + bound) if dtype == "bf16" else 2.0 ** -24 * np.abs(exact)))


# ---- attention of one query per batch index ----

# (heads, keys, dim, dtype): fewer keys than a step and than a lane group's rows, steps that the keys do not fill,
# one workgroup per head and several, every number of lanes per row
DECODES = [(3, 1, 128, "bf16"), (2, 37, 64, "f16"), (5, 128, 128, "bf16"), (600, 300, 64, "bf16"), (2, 5000, 128, "f16"),
           (3, 1029, 64, "f32"), (2, 700, 128, "f32"), (2, 300, 256, "f32"), (4, 513, 256, "bf16"), (2, 999, 8, "f16"),
           (1, 20000, 16, "bf16")]


def decode(heads, keys, dim, dtype, query_axis, computed=False):
    def body(b, a):
        q, k, v = (x.add(x) for x in a) if computed else a
        s = q.contract(k, "dim").mul(b.full_float(T.Type(dtype, ()), 0.125))
        e = s.sub(s.max("key")).exp()
        return e.div(e.sum("key")).contract(v, "key")
    one = [("query", 1)] if query_axis else []
    return T.define("decode", [T.spec(dtype, ("head", heads), *one, ("dim", dim))]
                    + [T.spec(dtype, head=heads, key=keys, dim=dim)] * 2, body)


@pytest.mark.gpu
@pytest.mark.parametrize("query_axis", [False, True])
@pytest.mark.parametrize("case", DECODES, ids=str)
def test_single_query_attention(case, query_axis):
    """Against float64: f32 scores and sums (1e-5 of the largest magnitude), then the result's rounding (bf16
    truncates: 2^-7; f16: 2^-11)."""
    heads, keys, dim, dtype = case
    prog = decode(heads, keys, dim, dtype, query_axis)
    assert "accy::decode::attend<" in hip.plan_source(prog)
    rng = np.random.default_rng(keys)
    shapes = [(heads, 1, dim) if query_axis else (heads, dim), (heads, keys, dim), (heads, keys, dim)]
    ins = [W.to_dtype(rng.standard_normal(sh), dtype) for sh in shapes]
    exact = exact_attention(ins[0].reshape(heads, 1, dim), ins[1], ins[2], 0.125, False, dtype).reshape(shapes[0])
    got = to_f32(hip_run(prog, ins)[0], dtype).astype(np.float64)
    r = {"bf16": 2.0 ** -7, "f16": 2.0 ** -11, "f32": 2.0 ** -24}[dtype]
    assert np.all(np.abs(got - exact) <= 1e-5 * np.abs(exact).max() + r * np.abs(exact))


@pytest.mark.gpu
@pytest.mark.parametrize("heads,keys,dim", [(128, 1030, 128), (3, 700, 64), (5, 520, 96)])
def test_single_query_attention_of_computed_operands(heads, keys, dim):
    """Queries, keys and values that no buffer holds: computed once, and no contraction is folded serially. No further
    from float64 than 1.5x the oracle's own error and one bf16 rounding of the largest value."""
    prog = decode(heads, keys, dim, "bf16", False, computed=True)
    assert "// dot:" not in hip.plan_source(prog)
    rng = np.random.default_rng(dim)
    ins = [W.to_dtype(rng.standard_normal(s) / 2, "bf16") for s in ((heads, dim), (heads, keys, dim), (heads, keys, dim))]
    q, k, v = (W.to_dtype(2 * to_f32(x, "bf16"), "bf16") for x in ins)
    exact = exact_attention(q.reshape(heads, 1, dim), k, v, 0.125, False, "bf16").reshape(heads, dim)
    got, ref = (to_f32(r[0], "bf16").astype(np.float64) for r in (hip_run(prog, ins), oracle_run(prog, ins)))
    assert np.abs(got - exact).max() <= 1.5 * np.abs(ref - exact).max() + 2.0 ** -7 * np.abs(exact).max()


@pytest.mark.parametrize("heads,keys,dim,dtype,fused", [
    (200000, 4, 64, "f32", False), (200000, 16, 64, "f32", True), (60000, 64, 8, "f32", False), (60000, 128, 8, "f32", True),
    (200000, 8, 128, "bf16", True), (200000, 128, 16, "bf16", False),
    (6000, 4, 64, "f32", True), (200000, 8, 64, "bf16", False), (200000, 32, 64, "bf16", True), (60000, 4, 64, "bf16", True),
    (1 << 20, 2, 8, "bf16", False), (300, 1, 8, "f16", True)])
def test_single_query_attention_of_a_few_keys(heads, keys, dim, dtype, fused):
    """A workgroup loads a whole step of keys: very many heads of a small part of one run unfused."""
    assert ("accy::decode::" in hip.plan_source(decode(heads, keys, dim, dtype, False))) == fused


def test_single_query_attention_of_any_number_of_heads_can_be_launched():
    """HIP refuses a launch of 2^32 work items: 2^24 heads of a workgroup each run as separate kernels."""
    assert "accy::decode::" in hip.plan_source(decode((1 << 24) - 1, 4096, 8, "f16", False))
    prog = decode(1 << 24, 4096, 8, "f16", False)
    assert "accy::decode::" not in hip.plan_source(prog) and max(work_items(prog)) < 1 << 32


@pytest.mark.gpu
def test_single_query_attention_special_values():
    """The row past the last key in memory (the next head's first) and the last row, which clamped loads
    repeat, are not finite: heads 0 and 2 stay exact, as does head 1 with a score of -inf."""
    heads, keys, dim = 4, 131, 64
    prog = decode(heads, keys, dim, "f32", False)
    rng = np.random.default_rng(5)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((heads, dim), (heads, keys, dim), (heads, keys, dim)))
    clean = hip_run(prog, [q, k, v])[0]
    k[3, 0], v[3, 0] = np.nan, np.inf
    q[1], k[1, 7] = np.abs(q[1]), -np.inf
    got, ref = hip_run(prog, [q, k, v])[0], oracle_run(prog, [q, k, v])[0]
    assert np.array_equal(got[0], clean[0]) and np.array_equal(got[2], clean[2])
    assert np.allclose(got[1], ref[1], rtol=1e-4, atol=1e-5) and np.isnan(got[3]).all() and np.isnan(ref[3]).all()
    v[2, -1] = np.inf              # the last key's own value: inf in the sum, in every dimension
    assert np.array_equal(np.isinf(hip_run(prog, [q, k, v])[0][2]), np.isinf(oracle_run(prog, [q, k, v])[0][2]))


@pytest.mark.gpu
def test_grouped_projections_with_a_k_tail():
    """Three contractions of one activation in one launch whose K is no multiple of 32, against separate float64
    products (the direct-to-LDS contractions' bound)."""
    m, k, n = 256, 1000, 256
    prog = T.define("qkv", [T.spec("bf16", m=m, k=k)] + [T.spec("bf16", k=k, n=n)] * 3,
                    lambda b, a: [a[0].contract(w, "k") for w in a[1:]])
    assert "mma16_dma_group<" in hip.plan_source(prog)
    rng = np.random.default_rng(6)
    ins = [W.to_dtype(rng.standard_normal(s), "bf16") for s in ((m, k), (k, n), (k, n), (k, n))]
    x, *ws = (to_f32(i, "bf16").astype(np.float64) for i in ins)
    for got, w in zip(hip_run(prog, ins), ws):
        ref = x @ w
        assert np.all(np.abs(to_f32(got, "bf16") - ref) <= (k + 2) * 2.0 ** -24 * (np.abs(x) @ np.abs(w)) + 2.0 ** -7 * np.abs(ref))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,model,ffn", [(130, 264, 520), (3, 67, 131), (257, 1000, 3001)])
def test_mlp_block_of_odd_sizes(tokens, model, ffn):
    """RMS norm, two contractions, GELU and a residual at sizes that take every contraction kernel's edges; no
    further from float64 than 1.5x the oracle's own error and one bf16 rounding of the largest value."""
    def body(b, a):
        x, g, w1, w2 = a
        return x.add(W.gelu(b, W.rms_norm(b, x, g, "model", "bf16").contract(w1, "model"), "bf16").contract(w2, "ffn"))
    prog = T.define("mlp", [T.spec("bf16", token=tokens, model=model), T.spec("bf16", model=model),
                            T.spec("bf16", model=model, ffn=ffn), T.spec("bf16", ffn=ffn, model=model)], body)
    rng = np.random.default_rng(tokens)
    ins = [W.to_dtype(v, "bf16") for v in (rng.standard_normal((tokens, model)), 0.5 + rng.random(model),
                                           rng.standard_normal((model, ffn)) / np.sqrt(model),
                                           rng.standard_normal((ffn, model)) / np.sqrt(ffn))]
    x, g, w1, w2 = (to_f32(i, "bf16").astype(np.float64) for i in ins)
    h = x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5) * g @ w1
    exact = x + 0.5 * h * (1 + np.tanh(0.7978845608028654 * (h + 0.044715 * h ** 3))) @ w2
    got, ref = (to_f32(r[0], "bf16").astype(np.float64) for r in (hip_run(prog, ins), oracle_run(prog, ins)))
    assert np.abs(got - exact).max() <= 1.5 * np.abs(ref - exact).max() + 2.0 ** -7 * np.abs(exact).max()


# ---- a process that loaded PyTorch, whose wheel brings another ROCm's compiler, before the library ----

AFTER_TORCH = """
import sys
import torch
import numpy as np
sys.path[:0] = [{root!r}, {tests!r}]
from accy_amd import hip, workloads as W
from conftest import exact_attention, hip_run, to_f32
for dtype, dim, seq, causal in [("f16", 64, 96, True), ("bf16", 128, 128, True), ("f16", 128, 192, False)]:
    print(dtype, dim, seq, causal, flush=True)
    prog = W.attention_program(2, seq, dim, dtype, causal)
    assert "accy::attn::flash<" in hip.plan_source(prog, compile=True)
    if {run}:
        ins = W.attention_inputs(2, seq, dim, dtype, seed=dim)
        exact = exact_attention(*ins, 1.0 / np.sqrt(dim), causal, dtype)
        got = to_f32(hip_run(prog, ins)[0], dtype)
        assert np.linalg.norm(got - exact) <= 1e-2 * np.linalg.norm(exact)
print("all ran")
"""


def after_torch(run):
    tests = Path(__file__).resolve().parent
    done = subprocess.run([sys.executable, "-c", AFTER_TORCH.format(root=str(tests.parent), tests=str(tests), run=run)],
                          capture_output=True, text=True, timeout=110)
    assert done.returncode == 0 and "all ran" in done.stdout, done.stdout + done.stderr


def test_16bit_attention_compiles_in_a_process_that_loaded_torch():
    """That compiler ends the process at an option it does not know."""
    after_torch(False)


@pytest.mark.gpu
def test_16bit_attention_runs_in_a_process_that_loaded_torch():
    """1e-2 normwise of float64, the bound of 16-bit attention everywhere."""
    after_torch(True)
