"""Workloads of the optimizer path, as a training program runs them: what is timed when a change is judged.

Every case goes through the package's public entry points: the Newton-Schulz hooks of ``archscale_amd.optim``, whole
``step()`` calls of the three matrix optimizers, the groups for vectors and vocabulary matrices, the symmetric products
and the power iteration.  Sizes are those of this repository's configurations and tests, or generic ones between them.

Families (the ``what`` field of a case):

``hook``      one Newton-Schulz call on a gradient or momentum tensor (``Muon(newton_schulz_func=...)`` users, evaluation
              scripts): coefficient tables ``quintic`` (production), ``constant`` (the older five-step row) and ``polar``
              (matrix sign, fp32 input)
``dense``     ``optim.muon.Muon.step()`` of a decoder: attention and MLP matrices under Muon or MuonH; with a vocabulary,
              embedding, output head and norm vectors under AdamW in the same optimizer
``experts``   the same for stacks of routed experts, renormalised per expert
``emerging``  ``emerging.Muon.step()``: EMA momentum in fp32, matrix sign, decoupled decay
``ball``      ``emerging.MuonBall.step()``: fused QKV and gate|up parameters split into pieces, power iteration,
              retraction to the spectral sphere
``vocab``     the groups without matrices of their own kind: AdamW, hyperball AdamW or Lion over vocabulary matrices and
              norm vectors
``syrk``      one symmetric product (``ns_line_1``, ``tsyrk_ex``), with or without an addend
``sigma``     power iteration on a stack of weights: spectral norms, with or without the singular vectors

Gradients are N(0, 1e-3^2), weights N(0, 0.02^2), optimizer state is that of the middle of a run; a single large matrix
gets heavy-tailed entries with a few empty rows, as embedding-like gradients have them.
"""
import math

import torch

from archscale_amd.emerging import Muon as EmergingMuon
from archscale_amd.emerging import MuonBall, power_iteration, spectral_norm
from archscale_amd.emerging.spectral_ball_utils import msign
from archscale_amd.optim.muon import Muon
from archscale_amd.optim import newton_schulz_hip as hooks

DEVICE = "cuda"
ALIGN = 256          # elements: parameters start at aligned places of the flat buffers that hold them
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}


# ---------------------------------------------------------------------------------------------------------------------
# which cases
# ---------------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # smallest call of the hook: a per-head or adapter-sized matrix; latency and launches count
        dict(name="hook_128x384", what="hook", batch=1, rows=128, cols=384, table="quintic", dtype="bfloat16"),
        # one projection of a small model through the five-step hook of the older optimizer
        dict(name="hook_512x2048", what="hook", batch=1, rows=512, cols=2048, table="constant", dtype="bfloat16"),
        # a ragged fp32 gradient (vocabulary-like long side), tall
        dict(name="hook_3001x1023_fp32", what="hook", batch=1, rows=3001, cols=1023, table="quintic", dtype="float32"),
        # one MLP matrix of a 7B-class model, heavy-tailed
        dict(name="hook_4096x14336", what="hook", batch=1, rows=4096, cols=14336, table="quintic", dtype="bfloat16"),
        # whole optimizer of a small research model in fp32: cautious decay, AdamW for embedding, head and norms
        dict(name="dense_384_fp32", what="dense", hidden=384, kv=96, ffn=1032, layers=4, vocab=5003, dtype="float32",
             muonh=False, cautious=True),
        # the depth-16 decoder, bf16 MuonH: the repository's headline workload
        dict(name="dense_2048_d16", what="dense", hidden=2048, kv=512, ffn=5632, layers=16, vocab=0, dtype="bfloat16",
             muonh=True, cautious=False),
        # 64 routed experts of one layer, norms per expert
        dict(name="experts_64", what="experts", experts=64, hidden=2048, up=512, down=256, layers=1, dtype="bfloat16"),
        # fp32 EMA momentum and matrix sign for a mid-sized decoder
        dict(name="emerging_1024_fp32", what="emerging", hidden=1024, kv=256, ffn=2816, layers=4, nesterov=True),
        # fused QKV (one piece per group and component) and gate|up parameters on the spectral sphere
        dict(name="ball_1024_fused", what="ball", hidden=1024, groups=4, kv=64, ffn=2816, layers=4, split="group",
             rounds=10, dtype="bfloat16"),
        # vocabulary matrices of the depth-16 decoder kept on the sphere, its norm vectors under plain AdamW
        dict(name="vocab_hyperball", what="vocab", vocab=50304, hidden=2048, norms=33, algorithm="hyperball", dtype="bfloat16"),
        # a Gram matrix through the single-product entry point
        dict(name="syrk_2048x5632", what="syrk", batch=1, n=2048, k=5632, addend=False),
        # spectral norms and vectors of one shape class of a mid-sized model, default number of rounds
        dict(name="sigma_16x1024x2816", what="sigma", batch=16, rows=1024, cols=2816, rounds=50, vectors=True, dtype="bfloat16"),
    ]


def _log(rng, lo, hi):
    """A size between lo and hi, even over the logarithm: half of them multiples of 8, the others as they come."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, v // 8 * 8) if rng.random() < 0.5 else v


def _sides(rng, lo, hi, most):
    """Two sides whose product stays below `most`, in either order."""
    a = _log(rng, lo, hi)
    b = min(_log(rng, lo, hi), max(lo, most // a))
    return (a, b) if rng.random() < 0.5 else (b, a)


def draw(rng):
    what = rng.choice(["hook", "hook", "dense", "experts", "emerging", "ball", "vocab", "syrk", "sigma"])
    if what == "hook":
        table = rng.choice(["quintic", "quintic", "constant", "polar"])
        rows, cols = _sides(rng, 33, 8192, 16 << 20)
        batch = rng.choice([1, 1, 1, 2, 3, 8]) if rows * cols < 1 << 20 else 1
        dtype = "float32" if table == "polar" else rng.choice(["bfloat16", "float32"])
        return dict(what=what, batch=batch, rows=rows, cols=cols, table=table, dtype=dtype)
    if what == "dense":
        hidden = _log(rng, 128, 2048)
        layers = rng.randint(1, 8 if hidden < 1024 else 4)
        return dict(what=what, hidden=hidden, kv=max(16, hidden // 4), ffn=max(64, int(hidden * rng.uniform(1.5, 3.0))),
                    layers=layers, vocab=rng.choice([0, _log(rng, 1000, 50304)]), dtype=rng.choice(["bfloat16", "float32"]),
                    muonh=rng.random() < 0.5, cautious=rng.random() < 0.5)
    if what == "experts":
        hidden = _log(rng, 256, 2048)
        return dict(what=what, experts=rng.choice([4, 8, 16, 32, 64]), hidden=hidden, up=_log(rng, 64, 768),
                    down=_log(rng, 64, 768), layers=rng.randint(1, 2), dtype=rng.choice(["bfloat16", "float32"]))
    if what == "emerging":
        hidden = _log(rng, 128, 2048)
        return dict(what=what, hidden=hidden, kv=max(16, hidden // 4), ffn=max(64, int(hidden * rng.uniform(1.5, 3.0))),
                    layers=rng.randint(1, 4), nesterov=rng.random() < 0.5)
    if what == "ball":
        kv, groups = rng.choice([32, 64, 96, 128]), rng.choice([2, 4, 8])
        hidden = _log(rng, 256, 1536)
        return dict(what=what, hidden=hidden, groups=groups, kv=kv, ffn=max(64, int(hidden * rng.uniform(1.5, 3.0))),
                    layers=rng.randint(1, 4), split=rng.choice(["component", "group", "head"]), rounds=rng.choice([5, 10, 50]),
                    dtype=rng.choice(["bfloat16", "float32"]))
    if what == "vocab":
        return dict(what=what, vocab=_log(rng, 1000, 50304), hidden=_log(rng, 128, 2048), norms=rng.randint(1, 65),
                    algorithm=rng.choice(["adamw", "hyperball", "lion"]), dtype=rng.choice(["bfloat16", "float32"]))
    if what == "syrk":
        n, k = _sides(rng, 64, 8192, 16 << 20)
        n = min(n, 6144)
        return dict(what=what, batch=rng.choice([1, 1, 4]) if n * max(n, k) < 4 << 20 else 1, n=n, k=k, addend=rng.random() < 0.5)
    rows, cols = _sides(rng, 64, 6144, 8 << 20)
    return dict(what="sigma", batch=rng.randint(1, 16), rows=rows, cols=cols, rounds=rng.choice([5, 10, 50]),
                vectors=rng.random() < 0.5, dtype=rng.choice(["bfloat16", "float32"]))


# ---------------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------------
class _Random:
    """Normal tensors on the device from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(int(seed))

    def normal(self, shape, scale, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.gen, device=DEVICE) * scale).to(dtype)

    def heavy(self, rows, cols, dtype):
        """Student-t with three degrees of freedom, standard deviation 1e-3, one row in a hundred empty."""
        z = self.normal((rows, cols), 1.0)
        chi = torch.zeros_like(z)
        for _ in range(3):
            chi += self.normal((rows, cols), 1.0).square_()
        z /= (chi / 3).sqrt_() * (math.sqrt(3.0) / 1e-3)
        z[torch.randperm(rows, generator=self.gen, device=DEVICE)[: rows // 100]] = 0
        return z.to(dtype)


def _flat(rnd, shapes, scale, dtype, positive=False):
    """One flat buffer and the tensors in it, as a program with flat parameter storage keeps them."""
    starts, total = [], 0
    for s in shapes:
        starts.append(total)
        total += (math.prod(s) + ALIGN - 1) // ALIGN * ALIGN
    flat = torch.zeros(total, dtype=dtype, device=DEVICE)
    views = [flat[a:a + math.prod(s)].view(s) for a, s in zip(starts, shapes)]
    for v in views:
        x = rnd.normal(v.shape, scale)
        v.copy_(x.square_() if positive else x)
    return flat, views


def _layer(hidden, kv, ffn):
    return [(hidden, hidden), (kv, hidden), (kv, hidden), (hidden, hidden), (ffn, hidden), (ffn, hidden), (hidden, ffn)]


def _matrix_shapes(c):
    if c["what"] in ("dense", "emerging"):
        return _layer(c["hidden"], c["kv"], c["ffn"]) * c["layers"]
    if c["what"] == "experts":
        return [(c["experts"], c["up"], c["hidden"]), (c["experts"], c["hidden"], c["down"])] * c["layers"]
    if c["what"] == "ball":
        h, f = c["hidden"], c["ffn"]
        return [(c["groups"] * _qkv_rows(c), h), (h, h), (2 * f, h), (h, f)] * c["layers"]
    return []


def _qkv_rows(c):
    return 6 * c["kv"]   # per group: four query heads, one key head, one value head


def _other_shapes(c):
    if c["what"] == "vocab":
        return [(c["vocab"], c["hidden"])] * 2 + [(c["hidden"],)] * c["norms"]
    if c["what"] == "dense" and c["vocab"]:
        return [(c["vocab"], c["hidden"])] * 2 + [(c["hidden"],)] * (2 * c["layers"] + 1)
    return []


def _step_state(c, seed):
    rnd = _Random(seed)
    dtype = torch.float32 if c["what"] == "emerging" else DTYPES[c["dtype"]]
    matrices, others = _matrix_shapes(c), _other_shapes(c)
    shapes = matrices + others
    weights, w = _flat(rnd, shapes, 0.02, dtype)
    _, g = _flat(rnd, shapes, 1e-3, dtype)
    # momentum of a run under way: the sum (or mean) of many gradients
    momentum, m = _flat(rnd, shapes, 3e-3 if c["what"] in ("dense", "experts") else 3e-4, dtype)
    params = [torch.nn.Parameter(t) for t in w]
    for p, t in zip(params, g):
        p.grad = t
    out = {"weights": weights, "momentum": momentum}
    mats, rest = params[:len(matrices)], params[len(matrices):]
    if c["what"] == "emerging":
        opt = EmergingMuon(params, lr=0.02, momentum_beta=0.95, weight_decay=0.01, use_nesterov=c["nesterov"], num_ns_steps=5)
    elif c["what"] == "ball":
        f = c["ffn"]
        for i in range(0, len(params), 4):
            params[i].is_qkv, params[i + 2].is_fc1 = True, True
        opt = MuonBall(params, lr=0.02, momentum_beta=0.9, weight_decay=0.01, power_iteration_steps=c["rounds"],
                       split_qkv=True, is_qkv_fn=lambda p: getattr(p, "is_qkv", False),
                       qkv_split_shapes=(4 * c["kv"], c["kv"], c["kv"]), qkv_split_mode=c["split"],
                       split_fc1=True, is_fc1_fn=lambda p: getattr(p, "is_fc1", False), fc1_split_shapes=(f, f))
    else:
        variance, v = _flat(rnd, others, 1e-3, dtype, positive=True) if others else (None, [])
        algorithm = c.get("algorithm", "adamw")
        groups = []
        if mats:
            groups.append(dict(params=mats))
        if rest:
            groups.append(dict(params=rest, algorithm="lion" if algorithm == "lion" else "adamw", lr=1e-3, weight_decay=0.1))
        opt = Muon(groups, lr=0.02, weight_decay=0.1 if c.get("cautious") else 0.0, nesterov=True,
                   cautious_wd=bool(c.get("cautious")), use_muonh=bool(c.get("muonh")) or c["what"] == "experts" or algorithm == "hyperball",
                   muonh_per_matrix=c["what"] == "experts")
        if variance is not None and algorithm != "lion":
            out["variance"] = variance
            for p, t in zip(rest, v):
                opt.state[p]["variance"] = t
    key = "momentum_buffer" if c["what"] in ("emerging", "ball") else "momentum"
    for p, t in zip(params, m):
        opt.state[p][key] = t
    return dict(what="step", opt=opt, out=out)


def prepare(case, seed):
    c = case
    if c["what"] == "hook":
        rnd, dtype = _Random(seed), DTYPES[c["dtype"]]
        if c["batch"] == 1 and c["rows"] * c["cols"] >= 16 << 20:
            x = rnd.heavy(c["rows"], c["cols"], dtype)
        else:
            lead = (c["batch"],) if c["batch"] > 1 else ()
            x = rnd.normal((*lead, c["rows"], c["cols"]), 1e-3, dtype)
        return dict(what="hook", table=c["table"], x=x)
    if c["what"] == "syrk":
        rnd = _Random(seed)
        lead = (c["batch"],) if c["batch"] > 1 else ()
        a = rnd.normal((*lead, c["n"], c["k"]), 1.0 / math.sqrt(c["k"]), torch.bfloat16)
        s = None
        if c["addend"]:
            s = rnd.normal((c["n"], c["n"]), 0.1)
            s = (s + s.t()).to(torch.bfloat16)
            a = a if a.dim() == 2 else a[0]   # the entry point with an addend takes one matrix
        return dict(what="syrk", a=a, c=s)
    if c["what"] == "sigma":
        w = _Random(seed).normal((c["batch"], c["rows"], c["cols"]), 0.02, DTYPES[c["dtype"]])
        return dict(what="sigma", w=w, rounds=c["rounds"], vectors=c["vectors"])
    return _step_state(c, seed)


# ---------------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------------
def run(state):
    what = state["what"]
    if what == "hook":
        x = state["x"]
        if state["table"] == "quintic":
            return hooks.zeropower_via_newtonschulz5(x, 1e-7)
        if state["table"] == "constant":
            return hooks.zeropower_via_newtonschulz5_legacy(x, steps=5)
        return msign(x, 5)
    if what == "syrk":
        if state["c"] is None:
            return hooks.ns_line_1(state["a"])
        return hooks.tsyrk_ex(state["a"], state["c"], alpha=1.2, beta=-0.7)
    if what == "sigma":
        return (power_iteration if state["vectors"] else spectral_norm)(state["w"], state["rounds"])
    state["opt"].step()
    return state["out"]


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct passes may be apart
# ---------------------------------------------------------------------------------------------------------------------
def _ns_flops(rows, cols, table):
    """Five iterations with the symmetric products taken once; the production table may finish its last two iterations
    on the short side (three more short-side products instead of two long ones)."""
    m, n = min(rows, cols), max(rows, cols)
    f = 5.0 * (3.0 * m * m * n + float(m) ** 3)
    return f - 3.0 * m * m * (n - m) if table == "quintic" else f


def _pieces(c):
    """(rows, cols) of every matrix that is orthogonalised on its own."""
    if c["what"] != "ball":
        return [s[-2:] for s in _matrix_shapes(c) for _ in range(s[0] if len(s) == 3 else 1)]
    h, f, kv, g = c["hidden"], c["ffn"], c["kv"], c["groups"]
    qkv = {"component": [(g * 4 * kv, h), (g * kv, h), (g * kv, h)],
           "group": [(4 * kv, h), (kv, h), (kv, h)] * g,
           "head": [(kv, h)] * (6 * g)}[c["split"]]
    return (qkv + [(h, h), (f, h), (f, h), (h, f)]) * c["layers"]


def _sigma_flops(rows, cols, rounds):
    m, n = min(rows, cols), max(rows, cols)
    return min(4.0 * m * n * rounds, 1.0 * m * m * n + 2.0 * m * m * rounds)


def work(case):
    c = case
    size = 4 if c.get("dtype") == "float32" or c["what"] == "emerging" else 2
    if c["what"] == "hook":
        elems = c["batch"] * c["rows"] * c["cols"]
        return {"bytes": elems * (size + 2.0), "flops": c["batch"] * _ns_flops(c["rows"], c["cols"], c["table"])}
    if c["what"] == "syrk":
        batch = 1 if c["addend"] else c["batch"]
        return {"bytes": 2.0 * batch * (c["n"] * c["k"] + c["n"] * c["n"] * (2 if c["addend"] else 1)),
                "flops": 1.0 * batch * c["n"] * c["n"] * c["k"]}
    if c["what"] == "sigma":
        return {"bytes": 1.0 * c["batch"] * c["rows"] * c["cols"] * size,
                "flops": c["batch"] * _sigma_flops(c["rows"], c["cols"], c["rounds"])}
    elems = sum(math.prod(s) for s in _matrix_shapes(c))
    rest = sum(math.prod(s) for s in _other_shapes(c))
    # weight read and written, gradient read, momentum read and written; AdamW: the variance too
    bytes_ = size * (5.0 * elems + (5.0 if c.get("algorithm") == "lion" else 7.0) * rest)
    table = "quintic" if c["what"] in ("dense", "experts") else "polar"
    flops = sum(_ns_flops(r, k, table) for r, k in _pieces(c)) + 12.0 * (elems + rest)
    if c["what"] == "ball":
        flops += sum(_sigma_flops(r, k, c["rounds"]) for r, k in _pieces(c))
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times what was measured against the same path with its products in fp64 (hooks: 3.3e-3 to 4.7e-3 for the
    production table, 1.9e-3 to 2.3e-3 for the two others; weights after a step: 5e-4 in bf16, 1e-4 in fp32, 6e-4 with
    the matrix sign) or against the same step in the package's other precision mode (spherical weights: 2.1e-3 to 3.4e-3);
    a product rounded to bf16 is off by 1.7e-3.  Singular vectors before convergence of a spectrum without gaps follow
    every rounding of the powers of the Gram matrix (1e-2), the norms do not (1e-4)."""
    c = case
    half = c.get("dtype") == "bfloat16"
    if c["what"] == "hook":
        return {"rel": 1.4e-2 if c["table"] == "quintic" else 9e-3}
    if c["what"] == "syrk":
        return {"rel": 7e-3}
    if c["what"] == "sigma":
        return {"rel": 3e-2 if c["vectors"] else 1e-3}
    if c["what"] == "vocab":
        return {"rel": 2e-3 if half else 1e-5}
    if c["what"] == "emerging":
        return {"rel": 2.5e-3}
    if c["what"] == "ball":
        return {"rel": 1e-2}
    return {"rel": 2e-3 if half else 4e-4}
