"""The work that a user of this framework has it do, as cases to time and compare.

Two kinds of entry points are used, as programs use them: pico's C API through
``pico_amd.pico`` (ops, ``pico_backward``, optimizers; tensors live in the
library's own device memory) and the launchers over torch tensors in
``pico_amd.kernels``.  Sizes are those of this repository's benchmark
configurations, or generic ones around them.

Inputs are drawn with torch's seeded device generator.  ``exact`` computes the
same outputs in float64 with torch alone.
"""
import ctypes
import math

import torch

from pico_amd import kernels as K
from pico_amd.pico import GPT_KEYS, TP, Pico

DEV = "cuda:0"
PRECISION = {"fp32": 0, "bf16": 1, "bf16x3": 2, "fp8": 3}
EPS = 1e-6


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one SGD step of a 784-128-10 ReLU classifier,
        # where latency and the number of launches count
        {"name": "mlp_step", "kind": "mlp", "batch": 64, "d_in": 784, "hidden": 128,
         "classes": 10},
        # a layer whose sizes are no multiple of anything: forward and both
        # backward products
        {"name": "matmul_ragged", "kind": "matmul", "m": 2000, "n": 1503, "k": 1001,
         "precision": "fp32"},
        # the headline product: a square matmul and its backward
        {"name": "matmul_square", "kind": "matmul", "m": 4096, "n": 4096, "k": 4096,
         "precision": "fp32"},
        # the fused row kernels on a large model's activations, forward and backward
        {"name": "rmsnorm_rows", "kind": "rmsnorm", "rows": 8192, "cols": 4096},
        {"name": "swiglu_rows", "kind": "swiglu", "rows": 8192, "cols": 11008},
        {"name": "xent_rows", "kind": "xent", "rows": 8192, "cols": 32000},
        # pre-norm attention layer of the 12-layer model (head size 64)
        {"name": "attention_64", "kind": "attention", "batch": 8, "seq": 1024, "heads": 12,
         "head": 64, "precision": "fp32"},
        # the same layer with larger heads and a sequence that is no multiple
        # of a tile
        {"name": "attention_128", "kind": "attention", "batch": 4, "seq": 1000, "heads": 8,
         "head": 128, "precision": "fp32"},
        # SwiGLU feed-forward layer of the 12-layer model with bf16 products
        {"name": "ffn_bf16", "kind": "ffn", "tokens": 8192, "d": 768, "ff": 2048,
         "precision": "bf16"},
        # pico's own op set: a broadcast expression and its gradients
        {"name": "broadcast_ops", "kind": "broadcast", "rows": 4096, "cols": 2048},
        # the optimizer step of a small transformer's parameters
        {"name": "adamw_step", "kind": "adamw", "layers": 4, "d": 512, "ff": 1376,
         "vocab": 8192},
        # a whole training step's forward and backward: the 1-layer model
        {"name": "gpt_step", "kind": "gpt", "batch": 16, "seq": 256, "d": 512, "heads": 8,
         "ff": 1376, "vocab": 8192, "layers": 1, "precision": "fp32"},
    ]


def _log(rng, lo, hi):
    """a size between lo and hi, spread over the logarithm; odd as often as even"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _precision(rng):
    return rng.choice(["fp32", "fp32", "fp32", "bf16", "bf16x3", "fp8"])


def draw(rng):
    kind = rng.choice(["mlp", "matmul", "matmul", "matmul", "rmsnorm", "swiglu", "xent",
                       "attention", "attention", "attention", "ffn", "broadcast", "adamw", "gpt"])
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 16, 1024), "d_in": _log(rng, 64, 1024),
                "hidden": _log(rng, 32, 512), "classes": _log(rng, 2, 128)}
    if kind == "matmul":
        step = rng.choice([1, 1, 4, 64])
        m, n, k = (max(step, _log(rng, 64, 4096) // step * step) for _ in range(3))
        return {"kind": kind, "m": m, "n": n, "k": k,
                "precision": rng.choice(["fp32", "fp32", "fp32", "bf16", "bf16x3"])}
    if kind in ("rmsnorm", "swiglu", "xent"):
        lo, hi = {"rmsnorm": (64, 8192), "swiglu": (64, 11008), "xent": (64, 32000)}[kind]
        step = rng.choice([1, 4, 64])
        return {"kind": kind, "rows": _log(rng, 32, 8192),
                "cols": max(step, _log(rng, lo, hi) // step * step)}
    if kind == "attention":
        head = rng.choice([32, 64, 64, 64, 96, 128])
        seq = _log(rng, 32, 2048)
        heads = rng.randint(2, max(2, 768 // head))
        batch = rng.randint(1, max(1, min(32, 8192 // seq)))
        return {"kind": kind, "batch": batch, "seq": seq, "heads": heads, "head": head,
                "precision": _precision(rng)}
    if kind == "ffn":
        d = 4 * _log(rng, 32, 256)
        return {"kind": kind, "tokens": _log(rng, 32, 8192), "d": d,
                "ff": rng.choice([32, 4]) * _log(rng, 8, 64), "precision": _precision(rng)}
    if kind == "broadcast":
        return {"kind": kind, "rows": _log(rng, 16, 4096), "cols": _log(rng, 16, 2048)}
    if kind == "adamw":
        d = 64 * rng.randint(1, 8)
        return {"kind": kind, "layers": rng.randint(1, 4), "d": d, "ff": _log(rng, d, 3 * d),
                "vocab": _log(rng, 64, 8192)}
    head = rng.choice([32, 64, 64])
    heads = rng.randint(2, 8)
    seq = _log(rng, 32, 512)
    return {"kind": kind, "batch": rng.randint(1, max(1, 4096 // seq)), "seq": seq,
            "d": head * heads, "heads": heads, "ff": 32 * rng.randint(4, 43),
            "vocab": _log(rng, 100, 8192), "layers": rng.randint(1, 2), "precision": "fp32"}


# ------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _inputs(c, seed):
    """the tensors a user's program has in hand, fp32 (ids int32) on the GPU"""
    g = _gen(seed)

    def normal(*shape, std=1.0, mean=0.0):
        return torch.randn(*shape, device=DEV, generator=g) * std + mean

    def uniform(*shape):
        return torch.rand(*shape, device=DEV, generator=g) * 2 - 1

    def ids(n, vocab):
        return torch.randint(0, vocab, (n,), device=DEV, generator=g, dtype=torch.int32)

    kind = c["kind"]
    if kind == "mlp":
        b, i, h, o = c["batch"], c["d_in"], c["hidden"], c["classes"]
        return {"x": normal(b, i), "w1": uniform(i, h) * i ** -0.5, "b1": uniform(h) * i ** -0.5,
                "w2": uniform(h, o) * h ** -0.5, "b2": uniform(o) * h ** -0.5, "labels": ids(b, o)}
    if kind == "matmul":
        m, n, k = c["m"], c["n"], c["k"]
        return {"a": uniform(m, k), "b": uniform(k, n), "dc": uniform(m, n)}
    if kind == "rmsnorm":
        r, n = c["rows"], c["cols"]
        return {"x": normal(r, n), "g": normal(n, std=0.02, mean=1.0), "dy": normal(r, n)}
    if kind == "swiglu":
        r, n = c["rows"], c["cols"]
        return {"a": normal(r, n), "u": normal(r, n), "dh": normal(r, n)}
    if kind == "xent":
        return {"z": normal(c["rows"], c["cols"], std=2.0), "labels": ids(c["rows"], c["cols"])}
    if kind == "attention":
        n, d = c["batch"] * c["seq"], c["heads"] * c["head"]
        return {"x": normal(n, d), "g": normal(d, std=0.02, mean=1.0),
                "wqkv": normal(d, 3 * d, std=d ** -0.5), "wo": normal(d, d, std=d ** -0.5)}
    if kind == "ffn":
        n, d, f = c["tokens"], c["d"], c["ff"]
        return {"x": normal(n, d), "g": normal(d, std=0.02, mean=1.0),
                "w13": normal(d, 2 * f, std=d ** -0.5), "w2": normal(f, d, std=f ** -0.5)}
    if kind == "broadcast":
        r, n = c["rows"], c["cols"]
        return {"x": normal(r, n), "scale": normal(n, std=0.1, mean=1.0), "bias": normal(n),
                "mean": normal(r, 1, std=0.3)}
    d, f, v = c["d"], c["ff"], c["vocab"]
    weights = [normal(v, d, std=0.02)]
    for _ in range(c["layers"]):
        weights += [normal(d, std=0.02, mean=1.0), normal(d, 3 * d, std=0.02),
                    normal(d, d, std=0.02), normal(d, std=0.02, mean=1.0),
                    normal(d, 2 * f, std=0.02), normal(f, d, std=0.02)]
    weights += [normal(d, std=0.02, mean=1.0), normal(d, v, std=0.02)]
    if kind == "adamw":
        return {"params": weights, "grads": [normal(*w.shape, std=1e-2) for w in weights]}
    n = c["batch"] * c["seq"]
    return {"params": weights, "tokens": ids(n, v), "targets": ids(n, v)}


# --------------------------------------------------- pico tensors and views
_pico = None


def _api():
    global _pico
    if _pico is None:
        _pico = Pico()
    return _pico


class _Memory:
    """device memory of the library as torch sees it; keeps its owner alive"""

    def __init__(self, ptr, shape, owner, typestr="<f4"):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 2}


class _Session:
    """the parameters, arenas and optimizers of one pico program"""

    def __init__(self, work_bytes):
        self.P = _api()
        self.lib = self.P.lib
        self.params, self.linears, self.optims = [], [], []
        self.model = None
        self.data = self.lib.arena_init(1 << 20)
        self.work = self.lib.arena_init(int(work_bytes))

    def view(self, t, grad=False):
        ptr = t.contents.grad if grad else t.contents.data
        return torch.as_tensor(_Memory(ptr, self.P.shape(t), self), device=DEV)

    def fill(self, t, values):
        self.lib.pico_gpu_synchronize()
        self.view(t).copy_(values.reshape(self.P.shape(t)))
        torch.cuda.synchronize()
        return t

    def param(self, values):
        t = self.P.param(list(values.shape))
        self.params.append(t)
        return self.fill(t, values)

    def ids(self, values):
        host = values.cpu().numpy()
        self.lib.arena_ctx_push(self.data)
        try:
            p = self.lib.pico_ids_to_device(host.ctypes.data_as(ctypes.c_void_p), host.size)
        finally:
            self.lib.arena_ctx_pop()
        if not p:
            raise RuntimeError("pico_ids_to_device failed")
        return p

    def sgd(self, lr, params):
        o = self.lib.pico_optim_sgd_init(lr)
        for p in params:
            self.lib.pico_optim_sgd_add(o, p)
        self.optims.append((o, self.lib.pico_optim_sgd_free))
        return o

    def begin(self, precision="fp32"):
        lib = self.lib
        if lib.pico_set_matmul_precision(PRECISION[precision]):
            raise RuntimeError("pico_set_matmul_precision failed")
        lib.arena_ctx_push(self.work)
        lib.arena_reset(self.work)

    def end(self):
        self.lib.arena_ctx_pop()
        self.lib.pico_set_matmul_precision(0)
        err = self.lib.pico_gpu_last_error()
        if err:
            self.lib.pico_gpu_clear_error()
            raise RuntimeError(err.decode(errors="replace"))

    def __del__(self):
        lib = self.lib
        lib.pico_gpu_synchronize()
        for o, free in self.optims:
            free(o)
        for fc in self.linears:
            lib.pico_nn_linear_free(fc)
        for p in self.params:
            lib.pico_free(p)
        if self.model:
            lib.pico_gpt_free(self.model)
        lib.arena_destroy(self.work)
        lib.arena_destroy(self.data)


def _linear(s, fan_in, fan_out, w, b):
    s.lib.arena_ctx_push(s.work)
    fc = s.lib.pico_nn_linear_init(fan_in, fan_out, True)
    s.lib.arena_ctx_pop()
    if not fc:
        raise RuntimeError("pico_nn_linear_init failed")
    s.linears.append(fc)
    wt = ctypes.cast(fc + 8, ctypes.POINTER(TP)).contents
    bt = ctypes.cast(fc + 16, ctypes.POINTER(TP)).contents
    s.fill(wt, w)
    s.fill(bt, b)
    return fc, wt, bt


def prepare(case, seed):
    c, x = case, _inputs(case, seed)
    kind = c["kind"]
    st = {"case": c, "x": x}
    if kind == "matmul":
        m, n, k = c["m"], c["n"], c["k"]
        need = max(K.gemm_workspace(m, n, k), K.gemm_workspace(m, k, n), K.gemm_workspace(k, n, m))
        st.update(c=torch.empty(m, n, device=DEV), da=torch.empty(m, k, device=DEV),
                  db=torch.empty(k, n, device=DEV), ws=torch.empty(max(1, need // 4), device=DEV))
    elif kind == "rmsnorm":
        r, n = c["rows"], c["cols"]
        st.update(y=torch.empty(r, n, device=DEV), rstd=torch.empty(r, device=DEV),
                  dx=torch.empty(r, n, device=DEV), dg=torch.empty(n, device=DEV),
                  ws=torch.empty(max(1, K.rmsnorm_bwd_workspace(r, n) // 4), device=DEV))
    elif kind == "swiglu":
        r, n = c["rows"], c["cols"]
        st.update({k: torch.empty(r, n, device=DEV) for k in ("h", "da", "du")})
    elif kind == "xent":
        st.update(rows=torch.empty(c["rows"], device=DEV), loss=torch.empty(1, device=DEV),
                  dz=torch.empty_like(x["z"]))
    else:
        sizes = {"mlp": 1 << 24, "broadcast": 1 << 28, "adamw": 1 << 20}
        s = _Session(sizes.get(kind, 1 << 30))
        st["s"] = s
        if kind == "mlp":
            st["fc1"], w1, b1 = _linear(s, c["d_in"], c["hidden"], x["w1"], x["b1"])
            st["fc2"], w2, b2 = _linear(s, c["hidden"], c["classes"], x["w2"], x["b2"])
            st["weights"] = [w1, b1, w2, b2]
            st["input"] = s.param(x["x"])
            st["labels"] = s.ids(x["labels"])
            st["opt"] = s.sgd(0.01, st["weights"])
        elif kind in ("attention", "ffn", "broadcast"):
            st["leaves"] = {k: s.param(v) for k, v in x.items()}
            st["opt"] = s.sgd(0.01, list(st["leaves"].values()))
        elif kind == "adamw":
            st["weights"] = [s.param(w) for w in x["params"]]
            opt = s.lib.pico_optim_adamw_init(3e-4, 0.9, 0.95, 1e-8, 0.1)
            s.optims.append((opt, s.lib.pico_optim_adamw_free))
            for t, gr in zip(st["weights"], x["grads"]):
                s.lib.pico_optim_adamw_add(opt, t)
                s.P.set_grad(t, gr.cpu().numpy())
            st["opt"] = opt
        else:
            cfg = dict(zip(GPT_KEYS, (c["vocab"], c["d"], c["layers"], c["heads"], c["ff"],
                                      c["batch"], c["seq"])))
            s.model = s.P.gpt_init(cfg, 1, norm_eps=EPS)
            st["weights"] = s.P.gpt_params(s.model)
            for t, w in zip(st["weights"], x["params"]):
                s.fill(t, w)
            st["tokens"], st["targets"] = s.ids(x["tokens"]), s.ids(x["targets"])
            st["opt"] = s.sgd(0.01, st["weights"])
        del st["x"]
    torch.cuda.synchronize()
    return st


# --------------------------------------------------------------------- runs
def _run_matmul(st):
    c, x = st["case"], st["x"]
    a, b, dc, ws = x["a"], x["b"], x["dc"], st["ws"]
    if c["precision"] == "fp32":
        product = K.gemm_ex
    elif c["precision"] == "bf16":
        product = K.gemm_bf16
    else:
        product = K.gemm_bf16x3
    product("N", "N", a, b, st["c"], ws=ws)
    product("N", "T", dc, b, st["da"], ws=ws)
    product("T", "N", a, dc, st["db"], ws=ws)
    return {"c": st["c"], "da": st["da"], "db": st["db"]}


def _run_attention(st):
    c, s, v = st["case"], st["s"], st["leaves"]
    lib, P = s.lib, s.P
    s.begin(c["precision"])
    lib.pico_optim_sgd_zero_grad(st["opt"])
    h = P.rmsnorm(v["x"], v["g"], EPS)
    q, k, w = P.split_cols(P.matmul(h, v["wqkv"]), 3)
    y = P.matmul_add(P.attention_causal(q, k, w, c["batch"], c["heads"]), v["wo"], v["x"])
    lib.pico_backward(s.work, y)
    s.end()
    return dict({"d" + n: s.view(t, grad=True) for n, t in v.items()}, y=s.view(y))


def _run_ffn(st):
    c, s, v = st["case"], st["s"], st["leaves"]
    lib, P = s.lib, s.P
    s.begin(c["precision"])
    lib.pico_optim_sgd_zero_grad(st["opt"])
    gate, up = P.split_cols(P.matmul_gate_up(P.rmsnorm(v["x"], v["g"], EPS), v["w13"]), 2)
    y = P.swiglu_matmul_add(gate, up, v["w2"], v["x"])
    lib.pico_backward(s.work, y)
    s.end()
    return dict({"d" + n: s.view(t, grad=True) for n, t in v.items()}, y=s.view(y))


def _run_broadcast(st):
    s, v = st["s"], st["leaves"]
    lib, P = s.lib, s.P
    s.begin()
    lib.pico_optim_sgd_zero_grad(st["opt"])
    t = P.tanh(P.add(P.mul(v["x"], v["scale"]), v["bias"]))
    y = P.mul(P.relu(P.sub(t, v["mean"])), v["x"])
    lib.pico_backward(s.work, y)
    s.end()
    return dict({"d" + n: s.view(p, grad=True) for n, p in v.items()}, y=s.view(y))


def run(state):
    st, kind = state, state["case"]["kind"]
    if kind == "matmul":
        return _run_matmul(st)
    if kind == "attention":
        return _run_attention(st)
    if kind == "ffn":
        return _run_ffn(st)
    if kind == "broadcast":
        return _run_broadcast(st)
    if kind == "rmsnorm":
        x = st["x"]
        K.rmsnorm_fwd(x["x"], x["g"], st["y"], st["rstd"], EPS)
        K.rmsnorm_bwd(x["x"], x["g"], st["rstd"], x["dy"], st["dx"], st["dg"], st["ws"])
        return {n: st[n] for n in ("y", "dx", "dg")}
    if kind == "swiglu":
        x = st["x"]
        K.swiglu_fwd(x["a"], x["u"], st["h"])
        K.swiglu_bwd(x["a"], x["u"], x["dh"], st["da"], st["du"])
        return {n: st[n] for n in ("h", "da", "du")}
    if kind == "xent":
        x, r = st["x"], st["case"]["rows"]
        K.xent_mean(x["z"], x["labels"], st["loss"], loss_rows=st["rows"], dlogits=st["dz"],
                    scale=1.0 / r, mean_scale=1.0 / r)
        return {n: st[n] for n in ("loss", "rows", "dz")}
    s = st["s"]
    lib, P = s.lib, s.P
    if kind == "adamw":
        lib.pico_optim_adamw_step(st["opt"])
        return [s.view(t) for t in st["weights"]]
    if kind == "mlp":
        s.begin()
        lib.pico_optim_sgd_zero_grad(st["opt"])
        h = P.relu(P.nn_linear_forward(st["fc1"], st["input"]))
        logits = P.nn_linear_forward(st["fc2"], h)
        loss = P.softmax_xent(logits, st["labels"])
        lib.pico_backward(s.work, loss)
        lib.pico_optim_sgd_step(st["opt"])
        s.end()
        return {"loss": s.view(loss), "logits": s.view(logits),
                "weights": [s.view(t) for t in st["weights"]],
                "grads": [s.view(t, grad=True) for t in st["weights"]]}
    s.begin(st["case"]["precision"])
    lib.pico_optim_sgd_zero_grad(st["opt"])
    loss = P.gpt_loss(s.model, st["tokens"], st["targets"])
    lib.pico_backward(s.work, loss)
    s.end()
    return {"loss": s.view(loss), "grads": [s.view(t, grad=True) for t in st["weights"]]}


# ---------------------------------------------------- work, tolerance, exact
def _attention_flops(c):
    # scores and their product with v over the causal pairs: 4 flops a head
    # value forward, 10 backward
    return 14.0 * c["batch"] * c["heads"] * c["head"] * c["seq"] * (c["seq"] + 1) / 2


def work(case):
    c, kind = case, case["kind"]
    if kind == "mlp":
        b, i, h, o = c["batch"], c["d_in"], c["hidden"], c["classes"]
        w = i * h + h + h * o + o
        return {"bytes": 4 * (b * (i + 1 + o) + 3 * w), "flops": 6 * b * (i * h + h * o)}
    if kind == "matmul":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4 * 2 * (m * k + k * n + m * n), "flops": 6 * m * n * k}
    if kind == "rmsnorm":
        return {"bytes": 4 * 4 * c["rows"] * c["cols"], "flops": 10 * c["rows"] * c["cols"]}
    if kind == "swiglu":
        return {"bytes": 4 * 6 * c["rows"] * c["cols"], "flops": 20 * c["rows"] * c["cols"]}
    if kind == "xent":
        return {"bytes": 4 * 2 * c["rows"] * c["cols"], "flops": 5 * c["rows"] * c["cols"]}
    if kind == "attention":
        n, d = c["batch"] * c["seq"], c["heads"] * c["head"]
        return {"bytes": 4 * (3 * n * d + 2 * 4 * d * d),
                "flops": 6 * n * 4 * d * d + _attention_flops(c)}
    if kind == "ffn":
        n, d, f = c["tokens"], c["d"], c["ff"]
        return {"bytes": 4 * (3 * n * d + 2 * 3 * d * f), "flops": 6 * n * 3 * d * f}
    if kind == "broadcast":
        r, n = c["rows"], c["cols"]
        return {"bytes": 4 * (3 * r * n + 4 * n + 2 * r), "flops": 12 * r * n}
    d, f, v = c["d"], c["ff"], c["vocab"]
    layer = 4 * d * d + 3 * d * f
    count = 2 * v * d + c["layers"] * (layer + 2 * d) + d
    if kind == "adamw":
        return {"bytes": 4 * 7 * count, "flops": 12 * count}
    n = c["batch"] * c["seq"]
    heads = dict(c, head=d // c["heads"])
    return {"bytes": 4 * (2 * count + 2 * n),
            "flops": 6 * n * (c["layers"] * layer + d * v) + c["layers"] * _attention_flops(heads)}


def tolerance(case):
    kind, p = case["kind"], case.get("precision", "fp32")
    if kind == "broadcast":
        return {"rel": 1e-5, "max": 1e-2}
    if kind in ("mlp", "rmsnorm", "swiglu", "xent", "adamw"):
        return {"rel": 1e-5}
    layered = kind != "matmul"
    rel = {"fp32": 1e-5, "bf16x3": 5e-5, "bf16": 1.5e-2, "fp8": 3e-2}[p]
    return {"rel": rel, "max": min(0.9, (200 if layered else 40) * rel)}


def _rms(x, g):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * g


def _causal(q, k, v, b, h):
    n, d = q.shape
    t, hd = n // b, d // h
    out = []
    keep = torch.ones(t, t, dtype=torch.bool, device=q.device).tril()
    for i in range(b):  # one sequence at a time: [h, t, t] scores
        qi, ki, vi = (x[i * t:(i + 1) * t].reshape(t, h, hd).transpose(0, 1).contiguous()
                      for x in (q, k, v))
        sc = torch.bmm(qi, ki.transpose(1, 2).contiguous()) * hd ** -0.5
        p = torch.softmax(sc.masked_fill(~keep, float("-inf")), -1)
        out.append(torch.bmm(p, vi).transpose(0, 1).reshape(t, d))
    return torch.cat(out)


def _swiglu(a, u):
    return torch.nn.functional.silu(a) * u


class _PicoTanh(torch.autograd.Function):
    """pico's tanh: its gradient is g - y*y, as the C expression has it"""

    @staticmethod
    def forward(ctx, x):
        y = torch.tanh(x)
        ctx.save_for_backward(y)
        return y

    @staticmethod
    def backward(ctx, g):
        y, = ctx.saved_tensors
        return g - y * y


def _leaves(x):
    return {k: v.double().requires_grad_() for k, v in x.items()}


def _graded(y, v):
    y.backward(torch.ones_like(y))
    return dict({"d" + n: t.grad for n, t in v.items()}, y=y.detach())


def exact(case, seed):
    c, x, kind = case, _inputs(case, seed), case["kind"]
    if kind == "matmul":
        a, b, dc = (x[n].double() for n in ("a", "b", "dc"))
        return {"c": a @ b, "da": dc @ b.t().contiguous(), "db": a.t().contiguous() @ dc}
    if kind == "rmsnorm":
        xs, g = x["x"].double().requires_grad_(), x["g"].double().requires_grad_()
        y = _rms(xs, g)
        y.backward(x["dy"].double())
        return {"y": y.detach(), "dx": xs.grad, "dg": g.grad}
    if kind == "swiglu":
        a, u = x["a"].double().requires_grad_(), x["u"].double().requires_grad_()
        h = _swiglu(a, u)
        h.backward(x["dh"].double())
        return {"h": h.detach(), "da": a.grad, "du": u.grad}
    if kind == "xent":
        z = x["z"].double().requires_grad_()
        rows = torch.nn.functional.cross_entropy(z, x["labels"].long(), reduction="none")
        loss = rows.mean()
        loss.backward()
        return {"loss": loss.detach().reshape(1), "rows": rows.detach(), "dz": z.grad}
    if kind == "mlp":
        w = [x[n].double().requires_grad_() for n in ("w1", "b1", "w2", "b2")]
        logits = torch.relu(x["x"].double() @ w[0] + w[1]) @ w[2] + w[3]
        loss = torch.nn.functional.cross_entropy(logits, x["labels"].long())
        loss.backward()
        return {"loss": loss.detach().reshape(1), "logits": logits.detach(),
                "weights": [t.detach() - 0.01 * t.grad for t in w], "grads": [t.grad for t in w]}
    if kind == "attention":
        v = _leaves(x)
        qkv = _rms(v["x"], v["g"]) @ v["wqkv"]
        q, k, w = qkv.chunk(3, -1)
        return _graded(v["x"] + _causal(q, k, w, c["batch"], c["heads"]) @ v["wo"], v)
    if kind == "ffn":
        v = _leaves(x)
        a, u = (_rms(v["x"], v["g"]) @ v["w13"]).chunk(2, -1)
        return _graded(v["x"] + _swiglu(a, u) @ v["w2"], v)
    if kind == "broadcast":
        v = _leaves(x)
        t = _PicoTanh.apply(v["x"] * v["scale"] + v["bias"])
        return _graded(torch.relu(t - v["mean"]) * v["x"], v)
    if kind == "adamw":
        out = []
        for w, g in zip(x["params"], x["grads"]):
            g = g.double()
            m, v = 0.1 * g, 0.05 * g * g
            step = 3e-4 / 0.1 * m / (v.sqrt() / 0.05 ** 0.5 + 1e-8)
            out.append(w.double() * (1 - 3e-4 * 0.1) - step)
        return out
    w = [t.double().requires_grad_() for t in x["params"]]
    h = w[0][x["tokens"].long()]
    for i in range(c["layers"]):
        g1, wqkv, wo, g2, w13, w2 = w[1 + 6 * i:7 + 6 * i]
        q, k, v = (_rms(h, g1) @ wqkv).chunk(3, -1)
        h = h + _causal(q, k, v, c["batch"], c["heads"]) @ wo
        a, u = (_rms(h, g2) @ w13).chunk(2, -1)
        h = h + _swiglu(a, u) @ w2
    logits = _rms(h, w[-2]) @ w[-1]
    loss = torch.nn.functional.cross_entropy(logits, x["targets"].long())
    loss.backward()
    return {"loss": loss.detach().reshape(1), "grads": [t.grad for t in w]}
