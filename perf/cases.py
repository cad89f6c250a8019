"""The work that programs built on this target have it do, as measured cases.

A case is one traced program at one size, run as a serving or training loop runs it: compiled once
(``hip.Hip``), inputs and outputs resident in HBM as torch tensors, one ``launch_device`` per pass on
torch's current stream. The kinds, and what they stand for:

* ``tone``       the consumer example's fit step: mismatch of every guess and its slope;
* ``logsumexp``  row-wise logsumexp, the row reduction of the benchmark;
* ``loss``       sparse cross-entropy of a language-model head with its logits gradient;
* ``linear``     one projection, from a decode step's few tokens to the benchmark's 8192^3;
* ``backward``   the gradients of a projection with a bias: input, weight and bias;
* ``mlp``        a decoder block's RMS norm -> W1 -> GELU -> W2 -> residual;
* ``attention``  softmax attention over whole sequences in f32 (prefill), causal or not;
* ``decode``     one query per head against a cache of keys and values;
* ``embedding``  the update of an embedding table: the gradients of a batch's tokens added to their rows.

16-bit attention over whole sequences is left to bench.py: its kernel needs a compiler option that the
hiprtc in torch's own wheel does not know, and a process that loads torch first compiles with that one.
Sizes are the benchmark programs' (accy_amd/workloads.py) or generic ones, odd ones among them.
"""
import math

import torch

from accy_amd import hip
from accy_amd import tensor as T
from accy_amd import workloads as W

TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "i32": torch.int32}
SIZE = {"f32": 4, "bf16": 2, "f16": 2, "i32": 4}


def listed():
    return [
        # The README's tone fit: eight guesses over sixteen points. Nothing but launch latency.
        {"name": "tone-readme", "kind": "tone", "guesses": 8, "points": 16},
        # The benchmark's tone workload, every guess with its slope.
        {"name": "tone-8192x16384", "kind": "tone", "guesses": 8192, "points": 16384},
        # The benchmark's logsumexp: 1 GiB streamed once.
        {"name": "lse-32768x8192-f32", "kind": "logsumexp", "rows": 32768, "features": 8192, "dtype": "f32"},
        # A training batch's loss over an odd-sized vocabulary, with the gradient of its logits.
        {"name": "loss-2048x50257-bf16", "kind": "loss", "tokens": 2048, "vocab": 50257, "dtype": "bf16"},
        # The benchmark's contraction, the largest piece of work here.
        {"name": "linear-8192-bf16", "kind": "linear", "tokens": 8192, "inner": 8192, "out": 8192, "dtype": "bf16"},
        # A decode step's MLP-up projection for sixteen sequences: the weights are read for few rows.
        {"name": "linear-decode16-bf16", "kind": "linear", "tokens": 16, "inner": 2048, "out": 8192, "dtype": "bf16"},
        # A general f32 contraction off every tile grid.
        {"name": "linear-1000-f32", "kind": "linear", "tokens": 1000, "inner": 1000, "out": 1000, "dtype": "f32"},
        # Gradients of a projection for a packed batch of sequences of uneven lengths.
        {"name": "backward-3000-bf16", "kind": "backward", "tokens": 3000, "inner": 2048, "out": 2048, "dtype": "bf16"},
        # The decoder block's MLP half for one sequence of the benchmark's length.
        {"name": "mlp-2048-bf16", "kind": "mlp", "tokens": 2048, "model": 2048, "ffn": 8192, "dtype": "bf16"},
        # Causal f32 attention of head dimension 64 over whole sequences.
        {"name": "attention-16x2048-f32", "kind": "attention", "heads": 16, "seq": 2048, "dim": 64, "causal": True,
         "dtype": "f32"},
        # A decode step's attention: eight sequences of sixteen heads against 4096 cached keys.
        {"name": "decode-128x4096-bf16", "kind": "decode", "heads": 128, "keys": 4096, "dim": 128, "dtype": "bf16"},
        # An embedding table's update for a batch of 4096 tokens.
        {"name": "embedding-32000x1024-f32", "kind": "embedding", "vocab": 32000, "model": 1024, "tokens": 4096,
         "dtype": "f32"},
    ]


# ---- drawn cases: the same kinds over the ranges their listed cases stand for ----

def _spread(rng, lo, hi):
    """A whole number of [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A model dimension: mostly multiples of 64, sometimes any number."""
    n = _spread(rng, lo, hi)
    return n if rng.random() < 0.3 else max(64, n // 64 * 64)


def draw(rng):
    kind = rng.choice(["tone", "logsumexp", "loss", "linear", "linear", "backward", "mlp", "attention", "decode",
                       "embedding"])
    if kind == "tone":
        return {"kind": kind, "guesses": _spread(rng, 1, 8192), "points": _spread(rng, 16, 16384)}
    if kind == "logsumexp":
        features = _spread(rng, 64, 131072)
        return {"kind": kind, "rows": _spread(rng, 1, min(32768, (1 << 28) // features)), "features": features,
                "dtype": rng.choice(["f32", "bf16", "f16"])}
    if kind == "loss":
        vocab = _spread(rng, 1000, 131072)
        return {"kind": kind, "tokens": _spread(rng, 16, min(8192, (1 << 27) // vocab)), "vocab": vocab,
                "dtype": rng.choice(["f32", "bf16"])}
    if kind == "linear":
        dtype = rng.choice(["bf16", "f16", "f32"])
        inner, out = _width(rng, 64, 8192), _width(rng, 64, 8192)
        most = (1 << 34 if dtype == "f32" else 1 << 39) // (inner * out)
        return {"kind": kind, "tokens": _spread(rng, 1, max(1, min(8192, most))), "inner": inner, "out": out,
                "dtype": dtype}
    if kind == "backward":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        inner, out = _width(rng, 64, 4096), _width(rng, 64, 4096)
        most = (1 << 33 if dtype == "f32" else 1 << 36) // (inner * out)
        return {"kind": kind, "tokens": _spread(rng, 16, max(16, min(8192, most))), "inner": inner, "out": out,
                "dtype": dtype}
    if kind == "mlp":
        model = _spread(rng, 4, 32) * 64
        return {"kind": kind, "tokens": _spread(rng, 1, 8192), "model": model, "ffn": 4 * model,
                "dtype": rng.choice(["bf16", "f16"])}
    if kind == "attention":
        seq = _spread(rng, 32, 4096)
        seq = seq if rng.random() < 0.3 else max(32, seq // 32 * 32)
        return {"kind": kind, "heads": _spread(rng, 1, min(64, max(1, (1 << 27) // (seq * seq)))), "seq": seq,
                "dim": 64, "causal": rng.random() < 0.5, "dtype": "f32"}
    if kind == "decode":
        dim, keys = rng.choice([64, 128]), _spread(rng, 16, 32768)
        return {"kind": kind, "heads": _spread(rng, 8, min(512, (1 << 27) // (keys * dim))), "keys": keys, "dim": dim,
                "dtype": rng.choice(["bf16", "f16", "f32"])}
    model, vocab = _width(rng, 64, 2048), _spread(rng, 1000, 131072)
    return {"kind": "embedding", "vocab": min(vocab, (1 << 27) // model), "model": model,
            "tokens": _spread(rng, 16, 8192), "dtype": "f32"}


# ---- programs, as a user traces them ----

def _scalar(b, dtype, v):
    return b.full_float(T.Type(dtype, ()), v)


def _loss(case):
    n, vocab, dtype = case["tokens"], case["vocab"], case["dtype"]

    def body(b, a):
        x, target = a
        e = x.sub(x.max("vocab")).exp()
        p = e.div(e.sum("vocab"))
        classes = b.iota("i32", "vocab", ("token", n), ("vocab", vocab))
        hot = classes.compare("eq", target).select(_scalar(b, dtype, 1.0), _scalar(b, dtype, 0.0))
        return [x.sparse_cross_entropy_loss(target, "vocab"), p.sub(hot).mul(_scalar(b, dtype, 1.0 / n))]
    return T.define("loss", [T.spec(dtype, token=n, vocab=vocab), T.spec("i32", token=n)], body)


def _linear(case):
    return W.gemm_program(case["tokens"], case["inner"], case["out"], case["dtype"])


def _backward(case):
    n, i, o, dtype = case["tokens"], case["inner"], case["out"], case["dtype"]

    def body(b, a):
        x, w, dy = a
        return [dy.contract(w, "out"), x.contract(dy, "token"), dy.sum("token")]
    return T.define("backward", [T.spec(dtype, token=n, inner=i), T.spec(dtype, inner=i, out=o),
                                 T.spec(dtype, token=n, out=o)], body)


def _mlp(case):
    n, m, f, dtype = case["tokens"], case["model"], case["ffn"], case["dtype"]

    def body(b, a):
        x, g, w1, w2 = a
        h = W.rms_norm(b, x, g, "model", dtype)
        return x.add(W.gelu(b, h.contract(w1, "model"), dtype).contract(w2, "ffn"))
    return T.define("mlp", [T.spec(dtype, token=n, model=m), T.spec(dtype, model=m), T.spec(dtype, model=m, ffn=f),
                            T.spec(dtype, ffn=f, model=m)], body)


def _decode(case):
    h, n, d, dtype = case["heads"], case["keys"], case["dim"], case["dtype"]

    def body(b, a):
        q, k, v = a
        s = q.contract(k, "dim").mul(_scalar(b, dtype, 1.0 / math.sqrt(d)))
        e = s.sub(s.max("key")).exp()
        return e.div(e.sum("key")).contract(v, "key")
    return T.define("decode", [T.spec(dtype, head=h, dim=d), T.spec(dtype, head=h, key=n, dim=d),
                               T.spec(dtype, head=h, key=n, dim=d)], body)


def _embedding(case):
    def body(b, a):
        table, ids, grad = a
        return table.scatter_add(ids, grad.mul(_scalar(b, case["dtype"], -0.01)), "vocab")
    return T.define("embedding", [T.spec(case["dtype"], vocab=case["vocab"], model=case["model"]),
                                  T.spec("i32", token=case["tokens"]),
                                  T.spec(case["dtype"], token=case["tokens"], model=case["model"])], body)


def _program(case):
    kind = case["kind"]
    if kind == "tone":
        return W.tone_value_and_slope_program(case["guesses"], case["points"])
    if kind == "logsumexp":
        return W.logsumexp_program(case["rows"], case["features"], case["dtype"])
    if kind == "attention":
        return W.attention_program(case["heads"], case["seq"], case["dim"], case["dtype"], case["causal"])
    return {"loss": _loss, "linear": _linear, "backward": _backward, "mlp": _mlp, "decode": _decode,
            "embedding": _embedding}[kind](case)


# ---- inputs, in the programs' parameter order ----

def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype = case["kind"], TORCH[case.get("dtype", "f32")]

    def normal(*shape, std=1.0):
        return torch.randn(shape, generator=gen, device="cuda").mul_(std).to(dtype)

    def uniform(*shape, lo, hi):
        return torch.rand(shape, generator=gen, device="cuda").mul_(hi - lo).add_(lo).to(dtype)

    if kind == "tone":
        # time[i] = 0.25 i and a sampled tone of frequency 3 with a little noise
        time = torch.arange(case["points"], device="cuda", dtype=torch.float32) * 0.25
        sample = torch.sin(3.0 * time) + normal(case["points"], std=0.01)
        return [uniform(case["guesses"], lo=0.5, hi=5.0), time, sample]
    if kind == "logsumexp":
        return [normal(case["rows"], case["features"])]
    if kind == "loss":
        logits = normal(case["tokens"], case["vocab"], std=3.0)
        target = torch.randint(0, case["vocab"], (case["tokens"],), generator=gen, device="cuda", dtype=torch.int32)
        return [logits, target]
    if kind == "linear":
        return [uniform(case["tokens"], case["inner"], lo=-1.0, hi=1.0), uniform(case["inner"], case["out"], lo=-1.0, hi=1.0)]
    if kind == "backward":
        return [normal(case["tokens"], case["inner"]), normal(case["inner"], case["out"], std=0.02),
                normal(case["tokens"], case["out"])]
    if kind == "mlp":
        return [normal(case["tokens"], case["model"]), uniform(case["model"], lo=0.5, hi=1.5),
                normal(case["model"], case["ffn"], std=0.02), normal(case["ffn"], case["model"], std=0.02)]
    if kind == "attention":
        return [normal(case["heads"], case["seq"], case["dim"]) for _ in range(3)]
    if kind == "decode":
        return [normal(case["heads"], case["dim"])] + [normal(case["heads"], case["keys"], case["dim"]) for _ in range(2)]
    # token frequencies fall about as 1 / rank: the logarithm of the rank is uniform
    u = torch.rand(case["tokens"], generator=gen, device="cuda", dtype=torch.float64)
    ids = torch.exp(u * math.log(case["vocab"] + 1)).to(torch.int32) - 1
    return [normal(case["vocab"], case["model"], std=0.02), ids.clamp_(0, case["vocab"] - 1),
            normal(case["tokens"], case["model"])]


def prepare(case, seed):
    executor = hip.Hip(_program(case))
    inputs = _inputs(case, seed)
    names = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
    outputs = [torch.empty(tuple(e for _, e in d.dims), dtype=names[d.dtype], device="cuda") for d in executor.outputs]
    return {"executor": executor, "inputs": inputs, "outputs": outputs}


def run(state):
    state["executor"].launch_device([t.data_ptr() for t in state["inputs"]], [t.data_ptr() for t in state["outputs"]],
                                    torch.cuda.current_stream().cuda_stream)
    return state["outputs"]


# ---- the work, what results may differ by, and the results in 64 bits ----

def work(case):
    kind, size = case["kind"], SIZE[case.get("dtype", "f32")]
    if kind == "tone":
        g, p = case["guesses"], case["points"]
        # phase, sin, difference, square, sum; twice the difference, cos, two products, sum
        return {"bytes": 4 * (3 * g + 2 * p), "flops": 11 * g * p}
    if kind == "logsumexp":
        n = case["rows"] * case["features"]
        return {"bytes": size * (n + case["rows"]), "flops": 4 * n}
    if kind == "loss":
        n = case["tokens"] * case["vocab"]
        return {"bytes": 2 * size * n + (4 + size) * case["tokens"], "flops": 7 * n}
    if kind == "linear":
        m, k, n = case["tokens"], case["inner"], case["out"]
        return {"bytes": size * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "backward":
        m, k, n = case["tokens"], case["inner"], case["out"]
        return {"bytes": size * (2 * (m * k + k * n) + m * n + n), "flops": 4 * m * k * n + m * n}
    if kind == "mlp":
        m, k, n = case["tokens"], case["model"], case["ffn"]
        return {"bytes": size * (2 * m * k + k + 2 * k * n), "flops": 4 * m * k * n}
    if kind == "attention":
        h, s, d = case["heads"], case["seq"], case["dim"]
        pairs = h * (s * (s + 1) // 2 if case["causal"] else s * s)
        return {"bytes": 4 * size * h * s * d, "flops": 4 * d * pairs}
    if kind == "decode":
        h, n, d = case["heads"], case["keys"], case["dim"]
        return {"bytes": 2 * size * h * d * (n + 1), "flops": 4 * h * n * d}
    v, m, n = case["vocab"], case["model"], case["tokens"]
    return {"bytes": size * (2 * v * m + n * m) + 4 * n, "flops": 2 * n * m}


def tolerance(case):
    if case.get("dtype", "f32") == "f32":
        # sums in another order differ by about 1e-6 of the result here
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] in ("decode", "mlp"):
        # Programs that round every operation to 16 bits: their results are 1.1e-2 (mlp) and 1.6e-2
        # (decode, whose scores, exponentials and quotients each lose bits) from the same in 64 bits.
        return {"rel": 3e-2, "max": 0.4}
    return {"rel": 1e-2, "max": 0.2}


def exact(case, seed):
    kind = case["kind"]
    args = [t.double() if t.is_floating_point() else t.long() for t in _inputs(case, seed)]
    if kind == "tone":
        frequency, time, sample = args
        value, slope = [], []
        for f in frequency.split(1024):
            phase = f[:, None] * time
            difference = torch.sin(phase) - sample
            value.append((difference * difference).sum(1))
            slope.append((2.0 * difference * torch.cos(phase) * time).sum(1))
        return [torch.cat(value), torch.cat(slope)]
    if kind == "logsumexp":
        return [torch.cat([torch.logsumexp(x, 1) for x in args[0].split(1024)])]
    if kind == "loss":
        x, target = args
        p = torch.log_softmax(x, 1)
        loss = -p.gather(1, target[:, None])[:, 0]
        grad = p.exp_()
        grad[torch.arange(case["tokens"], device="cuda"), target] -= 1.0
        return [loss, grad / case["tokens"]]
    if kind == "linear":
        return [args[0] @ args[1]]
    if kind == "backward":
        x, w, dy = args
        return [dy @ w.t(), x.t() @ dy, dy.sum(0)]
    if kind == "mlp":
        x, g, w1, w2 = args
        h = x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-5) * g
        return [x + torch.nn.functional.gelu(h @ w1, approximate="tanh") @ w2]
    if kind == "attention":
        q, k, v = args
        out = []
        for i in range(case["heads"]):
            s = (q[i] @ k[i].t()) / math.sqrt(case["dim"])
            if case["causal"]:
                s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(1), -math.inf)
            out.append(torch.softmax(s, 1) @ v[i])
        return [torch.stack(out)]
    if kind == "decode":
        q, k, v = args
        p = torch.softmax((k * q[:, None, :]).sum(2) / math.sqrt(case["dim"]), 1)
        return [(v * p[:, :, None]).sum(1)]
    table, ids, grad = args
    return [table.index_add(0, ids, grad * -0.01)]
