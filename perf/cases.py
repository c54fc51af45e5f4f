"""The work that programs have polytensors_amd do, as cases that can be timed and checked.

A program of this framework carries degree-K Taylor series (one tensor per order) through the
layers of a network: matrix products, attention, norms, activations and losses, forward and in
reverse mode. The listed cases are those layers at the sizes of the repository's benchmark
configurations, at generic layer sizes and at ragged ones; ``draw`` gives others of the same
ranges. Every case goes through ``PolyTensor`` and ``torch.nn.functional`` as a program calls them.

``exact`` restates each path in 64-bit plain torch on lists of coefficients; gradients come from
torch's own autograd of that restatement.
"""

import math

import torch
import torch.nn.functional as F

from polytensors_amd import PolyTensor

DEV = "cuda"
DTYPES = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZES = {"f64": 8, "f32": 4, "bf16": 2, "f16": 2}
# matrix-product rates used to bound a drawn case's cost (operations per second)
RATES = {"f64": 60e12, "f32": 120e12, "bf16": 1200e12, "f16": 1200e12}


def listed():
    return [
        # the launch-bound end: the whole of benchmark config 1 (a single-head float64 attention, a
        # projection and a mean loss), where the host path and the small launches are what counts
        dict(name="pipeline_f64", kind="pipeline", dtype="f64", degree=3, length=128, head=64, classes=256),
        # one layer on few rows (step-by-step evaluation, a small batch): little work per launch
        dict(name="linear_rows32_bf16", kind="linear", dtype="bf16", degree=2, rows=32, inner=1024, outer=4096),
        # the first MLP layer of the benchmark decoder: 8 x 1024 tokens, 768 -> 3072, with its bias
        dict(name="linear_decoder_f32", kind="linear", dtype="f32", degree=3, rows=8192, inner=768, outer=3072),
        # a training step's MLP block (no biases) in bfloat16: forward, and the gradients of every
        # coefficient and weight (coefficient autograd)
        dict(name="mlp_train_bf16", kind="mlp_train", dtype="bf16", degree=3, rows=4096, inner=1024, outer=4096),
        # series times series at benchmark config 2's size
        dict(name="matmul_4096_f32", kind="matmul", dtype="f32", degree=4, batch=1, m=4096, k=4096, n=4096),
        # the same product batched, in bfloat16, with sides that no tile divides
        dict(name="matmul_ragged_bf16", kind="matmul", dtype="bf16", degree=4, batch=4, m=511, k=1023, n=769),
        # causal prefill attention of benchmark config 3
        dict(name="attention_2048_f32", kind="attention", dtype="f32", degree=4, batch=4, heads=16, queries=2048,
             keys=2048, head=128, mask="causal"),
        # a padded batch with a length off the tiles, a mask per batch entry, the decoder's heads
        dict(name="attention_padded_bf16", kind="attention", dtype="bf16", degree=3, batch=4, heads=12, queries=1000,
             keys=1000, head=64, mask="padding"),
        # attention in a training step: forward and the gradient series of q, k and v
        dict(name="attention_grad_bf16", kind="attention_grad", dtype="bf16", degree=3, batch=2, heads=16,
             queries=1024, keys=1024, head=128, mask="causal"),
        # RMSNorm with its weight in a training step, on benchmark config 4's activations
        dict(name="rms_norm_grad_bf16", kind="norm_grad", dtype="bf16", degree=4, norm="rms", rows=8192, width=4096),
        # the loss of a training step over a vocabulary that is not a multiple of a vector
        dict(name="loss_grad_bf16", kind="loss_grad", dtype="bf16", degree=3, rows=4096, classes=32001),
        # one whole block of the benchmark decoder (config 5) along a complex direction
        dict(name="block_complex_f32", kind="block", dtype="f32", degree=3, batch=2, length=512, width=768, heads=12),
    ]


def _log(rng, low, high, multiple=1):
    """A size between low and high, even over its logarithm; odd ones among them."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(1, int(round(v / multiple))) * multiple


def _drawn(rng):
    kind = rng.choice(["pipeline", "linear", "linear", "mlp_train", "matmul", "matmul", "attention", "attention",
                       "attention_grad", "norm", "norm_grad", "loss", "loss_grad", "activation", "block"])
    dtype = rng.choice(["f32", "f32", "bf16", "bf16", "f16", "f64"])
    degree = rng.choice([1, 2, 2, 3, 3, 4, 4, 5])
    # sizes: whole vectors of 8 mostly, any size otherwise
    step = rng.choice([8, 8, 64, 1])
    c = dict(kind=kind, dtype=dtype, degree=degree)
    if kind == "pipeline":
        return dict(c, dtype=rng.choice(["f32", "f64"]), length=_log(rng, 16, 256), head=rng.choice([16, 32, 64, 128]),
                    classes=_log(rng, 16, 1024))
    if kind in ("linear", "mlp_train"):
        return dict(c, rows=_log(rng, 8, 8192), inner=_log(rng, 64, 4096, step), outer=_log(rng, 64, 4096, step))
    if kind == "matmul":
        return dict(c, batch=rng.choice([1, 1, 2, 4, 8]), m=_log(rng, 16, 4096, step), k=_log(rng, 16, 4096, step),
                    n=_log(rng, 16, 4096, step))
    if kind in ("attention", "attention_grad"):
        queries = _log(rng, 32, 2048)
        keys = queries if rng.random() < 0.7 else _log(rng, 32, 2048)
        if kind == "attention" and rng.random() < 0.25:   # a step of generation: few queries, all the keys
            queries, keys = rng.choice([1, 4, 16]), _log(rng, 128, 4096)
        mask = rng.choice(["causal", "padding", "none"]) if queries == keys else rng.choice(["padding", "none"])
        return dict(c, batch=rng.choice([1, 2, 4]), heads=rng.choice([4, 8, 12, 16]), queries=queries, keys=keys,
                    head=rng.choice([32, 64, 64, 128]), mask=mask)
    if kind in ("norm", "norm_grad"):
        return dict(c, norm=rng.choice(["rms", "layer"]), rows=_log(rng, 16, 16384), width=_log(rng, 64, 8192, step))
    if kind in ("loss", "loss_grad"):
        return dict(c, rows=_log(rng, 16, 8192), classes=_log(rng, 256, 65536, step))
    if kind == "activation":
        return dict(c, function=rng.choice(["gelu", "gelu_tanh", "silu", "tanh"]), rows=_log(rng, 16, 16384),
                    width=_log(rng, 64, 8192, step))
    heads = rng.choice([4, 8, 12])
    return dict(c, dtype=rng.choice(["f32", "f64"]), degree=rng.choice([1, 2, 3]), batch=rng.choice([1, 2, 4]),
                length=_log(rng, 32, 512), width=64 * heads, heads=heads)


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 4e12, w["flops"] / RATES[case["dtype"]])


def draw(rng):
    top = max(_cost(c) for c in listed())
    while True:
        c = _drawn(rng)
        if _cost(c) <= 0.6 * top:
            return c


# ---------------------------------------------------------------------------
# Inputs: normal values, coefficient k scaled by 0.5^k (the repository's benchmark and tests); the
# activations of a network between norms are of order one, weights of order 1 / sqrt(inner).

def _inputs(case, seed):
    """The plain tensors of a case: a dict of coefficient lists and tensors."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    dtype, K, kind = DTYPES[case["dtype"]], case["degree"], case["kind"]

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)

    def series(*shape, scale=1.0):
        return [normal(*shape, scale=scale * 0.5 ** k) for k in range(K + 1)]

    def classes(rows, n):
        return torch.randint(0, n, (rows,), generator=g, device=DEV)

    if kind == "pipeline":
        L, d, C = case["length"], case["head"], case["classes"]
        lines = [[normal(1, 1, L, d, scale=0.125), normal(1, 1, L, d, scale=0.125)] for _ in range(3)]
        return dict(q=lines[0], k=lines[1], v=lines[2], w=normal(d, C, scale=0.125), target=classes(L, C))
    if kind == "linear":
        return dict(x=series(case["rows"], case["inner"]),
                    w=normal(case["outer"], case["inner"], scale=case["inner"] ** -0.5), b=normal(case["outer"], scale=0.1))
    if kind == "mlp_train":
        r, i, o = case["rows"], case["inner"], case["outer"]
        return dict(x=series(r, i), w1=normal(o, i, scale=i ** -0.5), w2=normal(i, o, scale=o ** -0.5),
                    cot=series(r, i))
    if kind == "matmul":
        lead = () if case["batch"] == 1 else (case["batch"],)
        return dict(a=series(*lead, case["m"], case["k"], scale=case["k"] ** -0.5), b=series(*lead, case["k"], case["n"]))
    if kind in ("attention", "attention_grad"):
        B, H, L, S, d = (case[k] for k in ("batch", "heads", "queries", "keys", "head"))
        out = dict(q=series(B, H, L, d, scale=0.5), k=series(B, H, S, d, scale=0.5), v=series(B, H, S, d), mask=None)
        if case["mask"] == "padding":   # batch entry b admits all but the last b / (2 B) of its keys
            lengths = torch.tensor([max(1, S - b * S // (2 * B)) for b in range(B)], device=DEV)
            keep = torch.arange(S, device=DEV)[None, :] < lengths[:, None]
            out["mask"] = keep[:, None, None, :].expand(B, 1, L, S).contiguous()
        if kind == "attention_grad":
            out["cot"] = series(B, H, L, d)
        return out
    if kind in ("norm", "norm_grad"):
        r, n = case["rows"], case["width"]
        out = dict(x=series(r, n), w=1 + normal(n, scale=0.02), b=None)
        if case["norm"] == "layer":
            out["b"] = normal(n, scale=0.02)
        if kind == "norm_grad":
            out["cot"] = series(r, n)
        return out
    if kind in ("loss", "loss_grad"):
        return dict(z=series(case["rows"], case["classes"], scale=2.0), target=classes(case["rows"], case["classes"]))
    if kind == "activation":
        return dict(x=series(case["rows"], case["width"]))
    # block: weights N(0, 0.02), a complex direction N(0, 1) + i N(0, 1), as the benchmark decoder's
    B, T, d = case["batch"], case["length"], case["width"]
    p = dict(ln1_w=1 + normal(d, scale=0.02), ln1_b=normal(d, scale=0.02), attn_w=normal(3 * d, d, scale=0.02),
             attn_b=normal(3 * d, scale=0.02), proj_w=normal(d, d, scale=0.02), proj_b=normal(d, scale=0.02),
             ln2_w=1 + normal(d, scale=0.02), ln2_b=normal(d, scale=0.02), fc_w=normal(4 * d, d, scale=0.02),
             fc_b=normal(4 * d, scale=0.02), fc2_w=normal(d, 4 * d, scale=0.02), fc2_b=normal(d, scale=0.02))
    # the hidden state between blocks is of order one, the direction perturbs a part of it
    return dict(p=p, x=[normal(B, T, d), torch.complex(normal(B, T, d, scale=0.5), normal(B, T, d, scale=0.5))])


# ---------------------------------------------------------------------------
# The calls

def prepare(case, seed):
    t = _inputs(case, seed)
    kind, K = case["kind"], case["degree"]
    s = dict(t, case=case)
    if kind == "pipeline":
        for n in "qkv":
            s[n] = PolyTensor(tuple(t[n]), degree=K)
    elif kind in ("linear", "norm", "activation"):
        s["x"] = PolyTensor(tuple(t["x"]))
    elif kind == "block":
        s["x"] = PolyTensor(tuple(t["x"]), degree=K)
    elif kind == "matmul":
        s["a"], s["b"] = PolyTensor(tuple(t["a"])), PolyTensor(tuple(t["b"]))
    elif kind == "attention":
        for n in "qkv":
            s[n] = PolyTensor(tuple(t[n]))
    elif kind == "attention_grad":
        for n in "qkv":
            s[n] = PolyTensor(tuple(t[n]), requires_grad=True)
        s["cot"] = PolyTensor(tuple(t["cot"]))
    elif kind == "norm_grad":
        s["x"], s["cot"] = PolyTensor(tuple(t["x"]), requires_grad=True), PolyTensor(tuple(t["cot"]))
    elif kind in ("loss", "loss_grad"):
        s["z"] = PolyTensor(tuple(t["z"]), requires_grad=kind == "loss_grad")
    elif kind == "mlp_train":   # coefficients and weights are ordinary autograd leaves
        for n in ("w1", "w2"):
            s[n] = t[n].requires_grad_()
        s["leaves"] = [c.requires_grad_() for c in t["x"]]
        s["x"] = PolyTensor(tuple(s["leaves"]))
    return s


def _norm(s, x):
    n = (s["case"]["width"],)
    if s["case"]["norm"] == "rms":
        return F.rms_norm(x, n, s["w"], 1e-6)
    return F.layer_norm(x, n, s["w"], s["b"], 1e-5)


def _block(p, x, heads):
    B, T, d = x.shape
    h = F.layer_norm(x, (d,), p["ln1_w"], p["ln1_b"])
    q, k, v = F.linear(h, p["attn_w"], p["attn_b"]).split(d, dim=-1)
    q, k, v = (t.reshape(B, T, heads, d // heads).transpose(1, 2) for t in (q, k, v))
    y = F.scaled_dot_product_attention(q, k, v, is_causal=True)
    x = x + F.linear(y.transpose(1, 2).reshape(B, T, d), p["proj_w"], p["proj_b"])
    h = F.layer_norm(x, (d,), p["ln2_w"], p["ln2_b"])
    h = F.gelu(F.linear(h, p["fc_w"], p["fc_b"]), approximate="tanh")
    return x + F.linear(h, p["fc2_w"], p["fc2_b"])


_FUNCTIONS = {"gelu": F.gelu, "gelu_tanh": lambda x: F.gelu(x, approximate="tanh"), "silu": F.silu, "tanh": torch.tanh}


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind.endswith("_grad"):   # reverse mode through the series: one step's gradients
        with PolyTensor.plain_range(), PolyTensor.retain_wrappers():
            if kind == "attention_grad":
                ins = (s["q"], s["k"], s["v"])
            else:
                ins = (s["z"],) if kind == "loss_grad" else (s["x"],)
            for x in ins:
                x.grad = None
            if kind == "attention_grad":
                y = F.scaled_dot_product_attention(*ins, attn_mask=s["mask"], is_causal=case["mask"] == "causal")
                y.backward(s["cot"])
            elif kind == "norm_grad":
                y = _norm(s, s["x"])
                y.backward(s["cot"])
            else:
                y = PolyTensor.cross_entropy(s["z"], s["target"])
                y.backward()
            return dict(y=[c.detach() for c in y.coeffs], grads=[list(x.grad.coeffs) for x in ins])
    if kind == "mlp_train":
        with PolyTensor.plain_range(), PolyTensor.coefficient_autograd():
            y = F.linear(F.gelu(F.linear(s["x"], s["w1"])), s["w2"])
        grads = torch.autograd.grad(y.coeffs, s["leaves"] + [s["w1"], s["w2"]], s["cot"])
        return dict(y=[c.detach() for c in y.coeffs], grads=list(grads))
    with torch.no_grad(), PolyTensor.plain_range():
        if kind == "pipeline":
            out = F.scaled_dot_product_attention(s["q"], s["k"], s["v"], is_causal=True)
            logits = out.reshape(case["length"], case["head"]) @ s["w"]
            loss = F.cross_entropy(logits, s["target"])
            return dict(loss=list(loss.coeffs), logits=list(logits.coeffs))
        if kind == "linear":
            y = F.linear(s["x"], s["w"], s["b"])
        elif kind == "matmul":
            y = s["a"] @ s["b"]
        elif kind == "attention":
            y = F.scaled_dot_product_attention(s["q"], s["k"], s["v"], attn_mask=s["mask"],
                                               is_causal=case["mask"] == "causal")
        elif kind == "norm":
            y = _norm(s, s["x"])
        elif kind == "loss":
            y = PolyTensor.cross_entropy(s["z"], s["target"])
        elif kind == "activation":
            y = _FUNCTIONS[case["function"]](s["x"])
        else:
            y = _block(s["p"], s["x"], case["heads"])
        return list(y.coeffs)


# ---------------------------------------------------------------------------
# Work: each input read once, each output written once; the products of the series rules

def work(case):
    K, e, kind = case["degree"], SIZES[case["dtype"]], case["kind"]
    n, pairs = K + 1, (K + 1) * (K + 2) // 2
    if kind == "pipeline":
        L, d, C = case["length"], case["head"], case["classes"]
        return dict(bytes=e * (6 * L * d + d * C + n * L * C), flops=2 * pairs * 2 * d * L * (L + 1) / 2 + 2 * n * L * d * C)
    if kind == "linear":
        r, i, o = case["rows"], case["inner"], case["outer"]
        return dict(bytes=e * (n * r * (i + o) + i * o), flops=2 * n * r * i * o)
    if kind == "mlp_train":
        r, i, o = case["rows"], case["inner"], case["outer"]
        # x, cotangents and y, dx once; the hidden series and its gradient written and read once; weights, gradients
        return dict(bytes=e * (n * r * (4 * i + 4 * o) + 4 * i * o), flops=3 * 2 * 2 * n * r * i * o)
    if kind == "matmul":
        b, m, k, c = (case[x] for x in ("batch", "m", "k", "n"))
        return dict(bytes=e * n * b * (m * k + k * c + m * c), flops=2 * pairs * b * m * k * c)
    if kind in ("attention", "attention_grad"):
        B, H, L, S, d = (case[k] for k in ("batch", "heads", "queries", "keys", "head"))
        seen = L * (L + 1) / 2 if case["mask"] == "causal" else L * S
        if case["mask"] == "padding":
            seen = L * sum(max(1, S - b * S // (2 * B)) for b in range(B)) / B
        forward = 2 * 2 * pairs * d * B * H * seen
        once = e * n * B * H * d * (2 * L + 2 * S)
        if kind == "attention":
            return dict(bytes=once, flops=forward)
        # gradient: the scores again and four more products
        return dict(bytes=once + e * n * B * H * d * (4 * L + 4 * S), flops=forward * 3.5)
    if kind in ("norm", "norm_grad", "activation"):
        one = e * n * case["rows"] * case["width"]
        # forward: x and y; gradient: x, the cotangent and dx besides
        return dict(bytes=one * (5 if kind == "norm_grad" else 2), flops=4 * pairs * case["rows"] * case["width"])
    if kind in ("loss", "loss_grad"):
        one = e * n * case["rows"] * case["classes"]
        return dict(bytes=one * (3 if kind == "loss_grad" else 1), flops=2 * pairs * case["rows"] * case["classes"])
    # block: 2 K + 1 real planes a series; a product of two complex orders takes three real ones
    B, T, d = case["batch"], case["length"], case["width"]
    planes = 2 * K + 1
    products = 1 + 2 * (2 * K) + 3 * (K * (K - 1) // 2)
    flops = 2 * planes * B * T * 12 * d * d + 2 * 2 * products * d * B * T * (T + 1) / 2
    return dict(bytes=e * (planes * B * T * d * 2 + 12 * d * d), flops=flops)


# ---------------------------------------------------------------------------
# Tolerances: relative 2-norm error of each output order, four times the errors measured against
# ``exact`` over the listed and drawn cases. float32 sums over 4096 terms 2.6e-6, layers' outputs
# 3.5e-3 in bfloat16 and 4.3e-4 in float16 (a few roundings of sums held in float32).

def tolerance(case):
    return dict(rel={"f64": 1e-12, "f32": 1e-5, "f16": 1.7e-3, "bf16": 1.4e-2}[case["dtype"]])


# ---------------------------------------------------------------------------
# The same paths in 64-bit plain torch on coefficient lists

def _mul(a, b, product=torch.mul):
    """Cauchy product of two coefficient lists, to the longer one's length (a list of one: a constant)."""
    out = []
    for k in range(max(len(a), len(b))):
        terms = [product(a[i], b[k - i]) for i in range(k + 1) if i < len(a) and k - i < len(b)]
        out.append(sum(terms[1:], terms[0]))
    return out


def _ode(u, d0, step):
    """y' = d u' order by order: ``step(k, y)`` gives coefficient k of d from y's coefficients to k."""
    y = [d0]
    d = [step(0, y)]
    for k in range(1, len(u)):
        y.append(sum(j * u[j] * d[k - j] for j in range(1, k + 1)) / k)
        d.append(step(k, y))
    return y


def _exp(u):
    return _ode(u, u[0].exp(), lambda k, y: y[k])


def _rsqrt(s):
    r = [s[0].rsqrt()]
    for k in range(1, len(s)):
        r.append(-sum((2 * k - i) / (2 * k) * s[i] * r[k - i] for i in range(1, k + 1)) / s[0])
    return r


def _divide(a, b):
    y = []
    for k in range(len(a)):
        y.append((a[k] - sum(b[i] * y[k - i] for i in range(1, k + 1))) / b[0])
    return y


def _log_series(s):
    n = [c / s[0] for c in s]
    y = [s[0].log()]
    for k in range(1, len(s)):
        y.append(n[k] - sum(i / k * y[i] * n[k - i] for i in range(1, k)))
    return y


def _tanh(u):
    return _ode(u, u[0].tanh(), lambda k, y: (1 if k == 0 else 0) - sum(y[i] * y[k - i] for i in range(k + 1)))


def _gelu_tanh(u):
    c, a = math.sqrt(2 / math.pi), 0.044715
    cube = _mul(_mul(u, u), u)
    t = _tanh([c * (x + a * y) for x, y in zip(u, cube)])
    return [0.5 * x for x in _mul(u, [t[0] + 1] + t[1:])]


def _gelu(u):
    half = [-0.5 * c for c in _mul(u, u)]
    density = [c / math.sqrt(2 * math.pi) for c in _exp(half)]
    cdf = [0.5 * (1 + torch.erf(u[0] / math.sqrt(2)))]
    for k in range(1, len(u)):
        cdf.append(sum(j * u[j] * density[k - j] for j in range(1, k + 1)) / k)
    return _mul(u, cdf)


def _silu(u):
    return _mul(u, _ode(u, torch.sigmoid(u[0]), lambda k, y: y[k] - sum(y[i] * y[k - i] for i in range(k + 1))))


_EXACT_FUNCTIONS = {"gelu": _gelu, "gelu_tanh": _gelu_tanh, "silu": _silu, "tanh": _tanh}


def _normalise(x, w, b, eps, layer):
    if layer:
        x = [c - c.mean(-1, keepdim=True) for c in x]
    s = [c.mean(-1, keepdim=True) for c in _mul(x, x)]
    y = [c * w for c in _mul(x, _rsqrt([s[0] + eps] + s[1:]))]
    return y if b is None else [y[0] + b] + y[1:]


def _attend(q, k, v, keep):
    """Attention of one head's [L, d], [S, d] series; ``keep``: admissible pairs or None."""
    s = _mul(q, [c.transpose(-1, -2) for c in k], torch.matmul)
    s = [c / math.sqrt(q[0].shape[-1]) for c in s]
    if keep is not None:
        s = [c.masked_fill(~keep, float("-inf") if i == 0 else 0.0) for i, c in enumerate(s)]
    e = _exp([s[0] - s[0].detach().amax(-1, keepdim=True)] + s[1:])
    return _divide(_mul(e, v, torch.matmul), [c.sum(-1, keepdim=True) for c in e])


def _exact_attention(case, t):
    B, H, L, S = (case[k] for k in ("batch", "heads", "queries", "keys"))
    K = case["degree"]
    causal = torch.ones(L, S, dtype=torch.bool, device=DEV).tril() if case["mask"] == "causal" else None
    grad = case["kind"] == "attention_grad"
    y = [torch.empty(B, H, L, case["head"], dtype=torch.float64, device=DEV) for _ in range(K + 1)]
    grads = [[torch.empty(c.shape, dtype=torch.float64, device=DEV) for c in t[n]] for n in "qkv"]
    for b in range(B):
        keep = causal if t["mask"] is None else t["mask"][b, 0]
        for h in range(H):
            ins = [[c[b, h].double().requires_grad_(grad) for c in t[n]] for n in "qkv"]
            out = _attend(*ins, keep)
            for k in range(K + 1):
                y[k][b, h] = out[k].detach()
            if grad:
                # gradient series j is the gradient of coefficient K - j for the cotangents reversed
                cots = [t["cot"][K - k][b, h].double() for k in range(K + 1)]
                got = torch.autograd.grad(out, [c for x in ins for c in x], cots)
                for n in range(3):
                    for j in range(K + 1):
                        grads[n][j][b, h] = got[n * (K + 1) + K - j]
    return dict(y=y, grads=grads) if grad else y


def _log_sum_exp(z):
    top = z[0].amax(-1, keepdim=True)
    e = _exp([z[0] - top] + z[1:])
    s = [c.sum(-1) for c in e]
    lse = _log_series(s)
    return [lse[0] + top.squeeze(-1)] + lse[1:], e, s


def _exact_loss(case, t):
    rows, K = case["rows"], case["degree"]
    total = [torch.zeros((), dtype=torch.float64, device=DEV) for _ in range(K + 1)]
    grad = case["kind"] == "loss_grad"
    dz = [torch.empty(c.shape, dtype=torch.float64, device=DEV) for c in t["z"]] if grad else None
    for r in range(0, rows, 1024):
        z, y = [c[r:r + 1024].double() for c in t["z"]], t["target"][r:r + 1024]
        lse, e, s = _log_sum_exp(z)
        for k in range(K + 1):
            total[k] += (lse[k] - z[k].gather(1, y[:, None])[:, 0]).sum()
        if grad:   # the softmax series less one at the target
            p = _divide(e, [c[:, None] for c in s])
            p[0].scatter_add_(1, y[:, None], -torch.ones_like(y, dtype=torch.float64)[:, None])
            for k in range(K + 1):
                dz[k][r:r + 1024] = p[k] / rows
    loss = [c / rows for c in total]
    return dict(y=loss, grads=[dz]) if grad else loss


def _exact_block(case, t):
    heads, K, wide = case["heads"], case["degree"], torch.complex128
    p = {n: v.to(wide) for n, v in t["p"].items()}
    x = [t["x"][0].to(wide), t["x"][1].to(wide)] + [torch.zeros_like(t["x"][1], dtype=wide) for _ in range(K - 1)]
    B, T, d = x[0].shape

    def linear(u, w, b):
        y = [c @ p[w].T for c in u]
        return [y[0] + p[b]] + y[1:]

    def split(u):
        return [c.reshape(B, T, heads, d // heads).transpose(1, 2) for c in u]

    def attend(q, k, v):   # as _attend, with the real maximum of a complex constant order
        s = _mul(split(q), [c.transpose(-1, -2) for c in split(k)], torch.matmul)
        s = [c / math.sqrt(d // heads) for c in s]
        keep = torch.ones(T, T, dtype=torch.bool, device=DEV).tril()
        top = s[0].real.masked_fill(~keep, float("-inf")).amax(-1, keepdim=True)
        e0 = (s[0].real - top).exp().masked_fill(~keep, 0.0).to(wide)
        e = _ode(s, e0, lambda k, y: y[k])
        o = _divide(_mul(e, split(v), torch.matmul), [c.sum(-1, keepdim=True) for c in e])
        return [c.transpose(1, 2).reshape(B, T, d) for c in o]

    h = linear(_normalise(x, p["ln1_w"], p["ln1_b"], 1e-5, True), "attn_w", "attn_b")
    y = attend(*([c[..., i * d:(i + 1) * d] for c in h] for i in range(3)))
    x = [u + v for u, v in zip(x, linear(y, "proj_w", "proj_b"))]
    h = linear(_normalise(x, p["ln2_w"], p["ln2_b"], 1e-5, True), "fc_w", "fc_b")
    x = [u + v for u, v in zip(x, linear(_gelu_tanh(h), "fc2_w", "fc2_b"))]
    return [x[0].real] + x[1:]


def exact(case, seed):
    t, kind, K = _inputs(case, seed), case["kind"], case["degree"]

    def wide(xs):
        return [c.double() for c in xs]

    if kind in ("attention", "attention_grad"):
        return _exact_attention(case, t)
    if kind in ("loss", "loss_grad"):
        return _exact_loss(case, t)
    if kind == "block":
        return _exact_block(case, t)
    if kind == "pipeline":
        q, k, v = (wide(t[n]) + [torch.zeros_like(t[n][0], dtype=torch.float64) for _ in range(K - 1)] for n in "qkv")
        L = case["length"]
        out = _attend(q, k, v, torch.ones(L, L, dtype=torch.bool, device=DEV).tril())
        logits = [c.reshape(L, -1) @ t["w"].double() for c in out]
        lse, _, _ = _log_sum_exp(logits)
        loss = [(a - z.gather(1, t["target"][:, None])[:, 0]).mean() for a, z in zip(lse, logits)]
        return dict(loss=loss, logits=logits)
    if kind == "linear":
        y = [c @ t["w"].double().T for c in wide(t["x"])]
        return [y[0] + t["b"].double()] + y[1:]
    if kind == "matmul":
        return _mul(wide(t["a"]), wide(t["b"]), torch.matmul)
    if kind == "activation":
        return _EXACT_FUNCTIONS[case["function"]](wide(t["x"]))
    eps = 1e-6 if case.get("norm") == "rms" else 1e-5
    if kind in ("norm", "norm_grad"):
        x = [c.requires_grad_(kind == "norm_grad") for c in wide(t["x"])]
        y = _normalise(x, t["w"].double(), None if t["b"] is None else t["b"].double(), eps, case["norm"] == "layer")
        if kind == "norm":
            return y
        got = torch.autograd.grad(y, x, wide(t["cot"])[::-1])
        return dict(y=[c.detach() for c in y], grads=[list(got)[::-1]])
    # mlp_train
    x = [c.requires_grad_() for c in wide(t["x"])]
    w1, w2 = (t[n].double().requires_grad_() for n in ("w1", "w2"))
    y = [c @ w2.T for c in _gelu([c @ w1.T for c in x])]
    got = torch.autograd.grad(y, x + [w1, w2], wide(t["cot"]))
    return dict(y=[c.detach() for c in y], grads=list(got))
