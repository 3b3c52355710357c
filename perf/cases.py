"""The work that the performance of this package is judged by.

A case is a plain dict: what kind of call it is, the shapes of the parameter set, the element types and
the options.  ``prepare`` makes what a training program holds when it reaches the call (parameters,
gradients, an optimizer in the middle of its run), ``run`` makes the call once, ``work`` says what
the call has to move and compute at the least, ``tolerance`` how far two correct results may lie apart.

Values follow ``bench.py``: parameters N(0, 0.02), gradients N(0, 1e-3), ema N(0, 1e-4), ema_squared
N(0, 1e-3)^2.
"""
import math
import random

import torch

from ramtorch_amd import AdamW, copy_stochastic_

BF16, F16, F32, F64 = "bfloat16", "float16", "float32", "float64"
_ESIZE = {BF16: 2, F16: 2, F32: 4, F64: 8}
_FIRST_STEP = 100   # steps behind the optimizer when the case begins: bias corrections and noise of a run under way


def _case(name, path, shapes, p=BF16, g=BF16, m=BF16, v=BF16, **more):
    case = {"path": path, "shapes": shapes, "p": p, "g": g, "m": m, "v": v}
    if name:
        case["name"] = name
    case.update(more)
    return case


def listed():
    return [
        # The smallest step anyone takes: a toy network, or one adapter.  Host time and launches.
        _case("mlp_bf16", "step", "mlp", width=129, depth=3, inputs=77, outputs=10),
        # An ordinary small model: 305 tensors of all lengths, decayed and undecayed parameters in two groups.
        _case("groups_305", "step", "spread", tensors=305, longest=262144, layout=3, groups=2),
        # A model of tens of thousands of short tensors (bench.py's "small" set).
        _case("short_20064", "step", "spread", tensors=20000, longest=4096, layout=1234, squares=64),
        # One layer of the Llama-3-8B-shaped set: a shard, an adapted model, a pipeline stage.
        _case("layer_bf16", "step", "layers", hidden=4096, kv=1024, ffn=14336, layers=1, vocab=0),
        # The embeddings and two layers of that set: large enough for the optimizer to place its states.
        _case("embeddings_bf16", "step", "layers", hidden=4096, kv=1024, ffn=14336, layers=2, vocab=128256),
        # fp32 gradients under a loss scale, a global-norm clip, an fp32 second moment (bench.py's "mixed").
        _case("layer_mixed_clip", "step", "layers", g=F32, v=F32, hidden=4096, kv=1024, ffn=14336, layers=1, vocab=0,
              scale=1024.0, clip=1.0),
        # fp32 parameters and gradients with the default bf16 states, lengths that divide by nothing, clipped.
        _case("fp32_ragged_clip", "step", "spread", p=F32, g=F32, tensors=160, longest=1500000, layout=7, clip=1.0),
        # Gradient centralization over convolutions and a classifier: rows from 27 to 4608 elements, biases.
        _case("central_conv", "step", "conv", width=64, stages=4, blocks=2, classes=1000, central=1.0),
        # Gradients that are views of one communication bucket: a learnable scalar in front puts every other
        # gradient off by one element from any vector boundary.
        _case("bucket_gradients", "step", "layers", hidden=2048, kv=512, ffn=8192, layers=2, vocab=0, scalar=True,
              grads="bucket"),
        # The offload flow of step(): parameters, gradients and states all in pinned CPU memory.
        _case("offload_step", "offload", "layers", hidden=1024, kv=256, ffn=4096, layers=1, vocab=0, grads="cpu",
              pinned=True),
        # The offload flow of the backward hook: one layer in pinned CPU memory, updated parameter by
        # parameter from GPU gradients, last parameter first, and a closing step().
        _case("offload_hook", "hook", "layers", hidden=4096, kv=1024, ffn=14336, layers=1, vocab=0, grads="gpu",
              pinned=True),
        # copy_stochastic_ on its own: a master weight rounded into its bf16 copy.
        _case("round_weights", "copy", "one", p=BF16, g=F32, elements=67_108_867),
    ]


_MIXES = [  # (weight, p, g, m, v): what training programs hold
    (8, BF16, BF16, BF16, BF16), (3, BF16, F32, BF16, F32), (3, F32, F32, BF16, BF16), (2, F32, F32, F32, F32),
    (2, BF16, BF16, F32, F32), (2, F16, F16, F32, F32), (1, F16, F16, F16, F16), (1, F32, BF16, BF16, BF16),
    (1, BF16, BF16, F64, F64),
]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: every path, set shape, element type and option above, sizes
    spread over their logarithm.  At most the work of ``embeddings_bf16`` on the GPU and of
    ``offload_hook`` over the host link."""
    path = rng.choice(["step"] * 6 + ["offload", "hook", "copy"])
    if path == "copy":
        return _case(None, "copy", "one", p=BF16, g=F32, elements=_log(rng, 500, 300_000_000))
    on_gpu = path == "step"
    weights = [w for w, *_ in _MIXES]
    _, p, g, m, v = rng.choices(_MIXES, weights)[0]
    options = {}
    family = rng.choice(["mlp", "spread", "spread", "layers", "layers", "conv"])
    if family == "mlp":
        options.update(width=_log(rng, 16, 2000), depth=rng.randint(1, 6), inputs=_log(rng, 8, 1000), outputs=_log(rng, 1, 1000))
    elif family == "spread":
        options.update(tensors=_log(rng, 3, 8000 if on_gpu else 300), layout=rng.randrange(1 << 20))
        options["longest"] = min(_log(rng, 500, 3_000_000), 200_000_000 // options["tensors"] if on_gpu else 1_000_000)
        options["longest"] = max(options["longest"], 64)
    elif family == "layers":
        hidden = 8 * _log(rng, 24, 400 if on_gpu else 200) + rng.choice([0, 0, 0, 4, 1])
        options.update(hidden=hidden, kv=max(1, hidden // rng.choice([1, 4, 8])), ffn=int(hidden * rng.choice([2.7, 3.5, 4])),
                       layers=rng.randint(1, 3 if on_gpu else 2), vocab=rng.choice([0, 0, _log(rng, 100, 20_000)]))
        options["scalar"] = rng.random() < 0.3
    else:
        options.update(width=rng.choice([16, 24, 30, 32, 48, 64, 100]), stages=rng.randint(1, 4), blocks=rng.randint(1, 3),
                       classes=_log(rng, 2, 1000))
    if not on_gpu:
        options.update(grads="gpu" if path == "hook" else rng.choice(["cpu", "cpu", "gpu"]), pinned=rng.random() < 0.75)
        if F64 in (m, v):
            m = v = F32
    else:
        options["grads"] = rng.choice(["own", "own", "bucket"])
    if rng.random() < 0.3:
        options["scale"] = rng.choice([1024.0, 65536.0])
    if path != "hook" and rng.random() < 0.3:
        options["clip"] = rng.choice([1.0, 0.1])
    elif rng.random() < 0.3:
        options["central"] = rng.choice([1.0, 0.5])
    if rng.random() < 0.3:
        options["groups"] = 2
    return _case(None, path, family, p, g, m, v, **options)


# ---- the parameter sets --------------------------------------------------------------------------
def _shapes(case):
    family, shapes = case["shapes"], []
    if family == "one":
        return [(case["elements"],)]
    if family == "mlp":
        wide = [case["inputs"]] + [case["width"]] * case["depth"] + [case["outputs"]]
        for a, b in zip(wide, wide[1:]):
            shapes += [(b, a), (b,)]
    elif family == "layers":
        h, kv, f = case["hidden"], case["kv"], case["ffn"]
        if case.get("scalar"):
            shapes.append((1,))
        if case["vocab"]:
            shapes.append((case["vocab"], h))
        for _ in range(case["layers"]):
            shapes += [(h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f), (h,), (h,)]
        if case["vocab"]:
            shapes.append((case["vocab"], h))
    elif family == "conv":
        c = case["width"]
        shapes += [(c, 3, 3, 3), (c,)]
        for s in range(case["stages"]):
            out = case["width"] << s
            for _ in range(case["blocks"]):
                shapes += [(out, c, 3, 3), (out,), (out, out, 3, 3), (out,)]
                c = out
        shapes += [(case["classes"], c), (case["classes"],)]
    else:   # spread: lengths uniform in their logarithm; the longer half of the range are matrices
        rng = random.Random(case["layout"])
        for _ in range(case["tensors"]):
            n = min(case["longest"], max(1, _log(rng, 1, case["longest"])))
            cols = rng.randint(17, 700)
            shapes.append((n,) if n < math.sqrt(case["longest"]) * 8 else (max(1, n // cols), cols))
        shapes += [(1024, 1024)] * case.get("squares", 0)
    return shapes


def _numel(shape):
    return math.prod(shape)


def _elements(case):
    return sum(_numel(s) for s in _shapes(case))


_SCALES = {"p": 0.02, "g": 1e-3, "m": 1e-4, "v": 1e-3}
_PIECE = 1 << 26   # values drawn at a time: bounds the fp32 temporary


def _values(n, kind, dtype, gen, factor=1.0):
    """``n`` values of one array on the GPU."""
    out = torch.empty(n, dtype=dtype, device="cuda")
    for lo in range(0, n, _PIECE):
        x = torch.empty(min(_PIECE, n - lo), dtype=torch.float32, device="cuda").normal_(generator=gen).mul_(_SCALES[kind] * factor)
        out[lo:lo + x.numel()] = x.square_() if kind == "v" else x
    return out


def _carve(buf, shapes, step):
    """Views of ``shapes`` in one buffer; each begins at a multiple of ``step`` elements."""
    views, at = [], 0
    for s in shapes:
        views.append(buf[at:at + _numel(s)].view(s))
        at += (_numel(s) + step - 1) // step * step
    return views


def _room(shapes, step):
    return sum((_numel(s) + step - 1) // step * step for s in shapes)


# A set of up to this many tensors has a storage per tensor, and its results are handed back tensor by
# tensor.  Larger sets lie in a few flat buffers, at the 512-byte steps at which torch's allocator packs short tensors.
_APART = 20


# ---- what the program holds ----------------------------------------------------------------------
def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["path"] == "copy":
        n = case["elements"]
        return {"case": case, "source": _values(n, "p", torch.float32, gen), "seed": seed,
                "target": torch.zeros(n, dtype=torch.bfloat16, device="cuda")}
    shapes = _shapes(case)
    dtypes = {k: getattr(torch, case[k]) for k in "pgmv"}
    host = case["path"] != "step"
    apart = len(shapes) <= _APART

    def arrays(kind, where, factor=1.0):
        """(tensors, what holds their values)"""
        if kind == "g" and case.get("grads") == "bucket":
            buf = _values(_room(shapes, 1), kind, dtypes[kind], gen, factor)
            return _carve(buf, shapes, 1), [buf]
        if apart:
            flat = [_values(_numel(s), kind, dtypes[kind], gen, factor) for s in shapes]
        else:
            flat = [_values(_room(shapes, 256), kind, dtypes[kind], gen, factor)]
        if where != "cuda":
            flat = [t.cpu() for t in flat]
            if case.get("pinned"):
                flat = [t.pin_memory() for t in flat]
        return ([t.view(s) for t, s in zip(flat, shapes)] if apart else _carve(flat[0], shapes, 256)), flat

    where = "cpu" if host else "cuda"
    values, p_flat = arrays("p", where)
    params = [torch.nn.Parameter(t, requires_grad=False) for t in values]
    grads, _ = arrays("g", "cpu" if case.get("grads") == "cpu" else "cuda", case.get("scale", 1.0))
    options = dict(lr=1e-4, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01, dtype=dtypes["m"], ema_squared_dtype=dtypes["v"],
                   storage_device=where, seed=1234, loss_scale=case.get("scale", 1.0), max_grad_norm=case.get("clip"),
                   centralization=case.get("central", 0))
    if case.get("groups") == 2:   # matrices decay, vectors do not
        groups = [{"params": [p for p in params if p.dim() > 1]}, {"params": [p for p in params if p.dim() <= 1], "weight_decay": 0.0}]
        opt = AdamW([g for g in groups if g["params"]], **options)
    else:
        opt = AdamW(params, **options)
    if apart:   # the optimizer's own state tensors, where it placed them
        for p in params:
            st = opt.state[p]
            st["step"] = _FIRST_STEP
            st["ema"].copy_(_values(p.numel(), "m", dtypes["m"], gen).view(p.shape))
            st["ema_squared"].copy_(_values(p.numel(), "v", dtypes["v"], gen).view(p.shape))
        held = [opt.state[p][k] for k in ("ema", "ema_squared") for p in params]
    else:       # states as a flat checkpoint left them
        m, m_flat = arrays("m", where)
        v, v_flat = arrays("v", where)
        for p, a, b in zip(params, m, v):
            opt.state[p].update(step=_FIRST_STEP, ema=a, ema_squared=b)
        held = m_flat + v_flat
    given = None
    if all(g.dtype == p.dtype and g.device == p.device for p, g in zip(params, grads)):
        for p, g in zip(params, grads):
            p.grad = g
    else:       # torch does not store such gradients in .grad
        given = dict(zip(params, grads))
    return {"case": case, "params": params, "grads": grads, "given": given, "opt": opt, "outputs": p_flat + held}


def run(state):
    case = state["case"]
    if case["path"] == "copy":
        return copy_stochastic_(state["target"], state["source"], seed=state["seed"])
    opt = state["opt"]
    if case["path"] == "hook":
        for p, g in zip(reversed(state["params"]), reversed(state["grads"])):
            opt.step_param(p, g)
        opt.step()
    else:
        opt.step(grads=state["given"])
    return state["outputs"]


def work(case):
    n = _elements(case)
    if case["path"] == "copy":
        return {"bytes": 6 * n, "flops": 2 * n}
    size = {k: _ESIZE[case[k]] for k in "pgmv"}
    return {"bytes": n * (2 * (size["p"] + size["m"] + size["v"]) + size["g"]), "flops": 25 * n}


def tolerance(case):
    # The noise is a function of seed, tensor, element and step, and every rounding of the update is fixed:
    # the same bits come out.  A clip coefficient and a row mean are sums whose order is free, though: they
    # may differ in the last bits, and then now and then a bf16 value is rounded the other way, by one step of
    # 2^-8 to 2^-7 of its size.  Two passes with these sums in float64 instead lay up to 1.2e-5 (2-norm) and
    # 0.0103 (one value) from the path as it is.
    if case.get("clip") or case.get("central"):
        return {"rel": 5e-5, "max": 0.03}
    return "exact"
