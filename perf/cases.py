"""Performance cases of the fused softplus-MLP library: the calls a user's
program makes, through the public entry points (``kernel._fused_mlp_fwd``, the
modules of ``fused_mlp`` / ``fused_mlp5``), over the ranges they are used in.

A case is a dict:

* ``mode``: ``"infer"`` (no autograd) or ``"train"`` (forward, loss gradient,
  backward: the output and every gradient are returned);
* ``api``: ``"launcher"`` (three weight tensors in hand), ``"module"`` or
  ``"wn"`` (the weight-normalised module);
* ``d_in``, ``hidden``, ``d_out``, ``layers``, ``rows``: the network and batch;
* ``dtype``: element type of the tensors, or with ``amp`` the autocast type
  around an fp32 module and an fp32 input; the weight-normalised module keeps
  its parameters in fp32, whatever the input's type;
* ``x_grad``: the input needs a gradient too;
* ``loss``: ``"dense"`` (an upstream gradient per output element) or ``"sum"``
  (``out.sum()``);
* ``graph``: the step was captured as a HIP graph once and is replayed, which
  is how a program with small fixed batches runs it;
* ``uniform``: inputs are coordinates in (-1, 1) instead of N(0, 1) features.

Weights are N(0, 1/in), the modules' own initialisation.
"""
import math

import torch
import torch.nn.functional as F

import fused_mlp
import fused_mlp5
import kernel

_DTYPE = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, mode, api, widths, layers, dtype, rows, **options):
    d_in, hidden, d_out = widths
    case = {"mode": mode, "api": api, "d_in": d_in, "hidden": hidden, "d_out": d_out, "layers": layers,
            "dtype": dtype, "rows": rows, "amp": False, "x_grad": False, "loss": "dense", "graph": False,
            "uniform": False}
    case.update(options)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # One small request of a serving loop: latency of a single launch.
        _case("infer_3x128_fp16_256", "infer", "launcher", (128, 128, 128), 3, "fp16", 256),
        # The reference's headline network as one bulk evaluation.
        _case("infer_3x128_fp16_1m", "infer", "launcher", (128, 128, 128), 3, "fp16", 1048576),
        # The deeper variant at an ordinary batch, bf16 as models are now kept.
        _case("infer_5x128_bf16_64k", "infer", "module", (128, 128, 128), 5, "bf16", 65536),
        # A neural field evaluated over a volume: narrow rows, most of them.
        _case("infer_narrow_fp16_4m", "infer", "launcher", (32, 64, 16), 3, "fp16", 4194304, uniform=True),
        # torch's default element type, a batch that is no round number.
        _case("infer_3x128_fp32_200k", "infer", "module", (128, 128, 128), 3, "fp32", 200003),
        # Wider hidden layers, up to the streamed-weight kernel's limit ...
        _case("infer_3x256_fp16_128k", "infer", "module", (128, 256, 128), 3, "fp16", 131072),
        # ... and past it (networks that run layer by layer).
        _case("infer_3x512_fp16_16k", "infer", "module", (128, 512, 128), 3, "fp16", 16384),
        # The reference's training step with weight norm: a small batch,
        # replayed as a graph, and the largest one, run eagerly with its loss.
        _case("train_wn_3x128_fp16_4k", "train", "wn", (128, 128, 128), 3, "fp16", 4096, graph=True),
        _case("train_wn_3x128_fp16_128k", "train", "wn", (128, 128, 128), 3, "fp16", 131072, loss="sum"),
        # fp32 training with an input gradient (the MLP as a layer inside a model).
        _case("train_3x128_fp32_64k", "train", "module", (128, 128, 128), 3, "fp32", 65536, x_grad=True),
        # Mixed-precision training of a wider network, ragged batch.
        _case("train_3x256_amp_bf16_100k", "train", "module", (128, 256, 128), 3, "bf16", 100003, amp=True),
        # Fitting a coordinate network: three inputs, four outputs.
        _case("train_field_4x64_fp16_256k", "train", "module", (3, 64, 4), 4, "fp16", 262144, uniform=True),
    ]


def _log_rows(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    # One in three a whole number of row blocks, the others as they fall.
    return max(lo, n // 32 * 32) if rng.random() < 1 / 3 else n


def draw(rng):
    kind = rng.choice(["infer_128", "infer_128", "infer_field", "infer_wide", "infer_very_wide",
                       "train_128", "train_128", "train_field", "train_wide"])
    dtype16 = rng.choice(["fp16", "bf16"])
    if kind == "infer_128":
        layers = rng.choice([3, 3, 5])
        dtype = rng.choice(["fp16", "bf16", "fp32"])
        api = "launcher" if layers == 3 and rng.random() < 0.5 else "module"
        top = 262144 if dtype == "fp32" else 524288
        return _case(None, "infer", api, (128, 128, 128), layers, dtype, _log_rows(rng, 64, top))
    if kind == "infer_field":
        widths = (rng.choice([2, 3, 16, 32, 63]), 16 * rng.randint(2, 6), rng.randint(1, 16))
        return _case(None, "infer", "module", widths, rng.randint(2, 5), dtype16, _log_rows(rng, 1024, 1048576),
                     uniform=True)
    if kind == "infer_wide":
        widths = (16 * rng.randint(4, 16), 16 * rng.randint(9, 16), 8 * rng.randint(1, 16))
        return _case(None, "infer", "module", widths, rng.randint(2, 4), dtype16, _log_rows(rng, 256, 131072))
    if kind == "infer_very_wide":
        widths = (16 * rng.randint(2, 16), 16 * rng.randint(17, 32), 8 * rng.randint(1, 16))
        return _case(None, "infer", "module", widths, rng.randint(2, 4), dtype16, _log_rows(rng, 256, 16384))
    if kind == "train_128":
        layers = rng.choice([3, 3, 5])
        dtype = rng.choice(["fp16", "bf16", "fp32"])
        rows = _log_rows(rng, 1024, 65536 if dtype == "fp32" or layers == 5 else 131072)
        return _case(None, "train", rng.choice(["module", "wn"]), (128, 128, 128), layers, dtype, rows,
                     x_grad=rng.random() < 0.5, graph=rows <= 16384 and rng.random() < 0.5)
    if kind == "train_field":
        widths = (rng.choice([2, 3, 16, 32, 63]), 16 * rng.randint(2, 6), rng.randint(1, 16))
        return _case(None, "train", "module", widths, rng.randint(2, 5), dtype16, _log_rows(rng, 1024, 131072),
                     x_grad=rng.random() < 0.3, uniform=True)
    widths = (16 * rng.randint(4, 16), 16 * rng.randint(9, 16), 8 * rng.randint(1, 16))
    return _case(None, "train", rng.choice(["module", "wn"]), widths, rng.randint(2, 4), dtype16,
                 _log_rows(rng, 1024, 65536), amp=rng.random() < 0.5, x_grad=rng.random() < 0.3)


def _widths(case):
    return [case["d_in"]] + [case["hidden"]] * (case["layers"] - 1) + [case["d_out"]]


def _inputs(case, seed):
    """x, the weights ([in, out] each) and the upstream gradient, on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dims, rows = _widths(case), case["rows"]
    dtype = torch.float32 if case["amp"] else _DTYPE[case["dtype"]]
    if case["uniform"]:
        x = (torch.rand((rows, dims[0]), generator=gen, device="cuda") * 2 - 1).to(dtype)
    else:
        x = torch.randn((rows, dims[0]), generator=gen, device="cuda").to(dtype)
    ptype = torch.float32 if case["api"] == "wn" else dtype
    weights = [(torch.randn((dims[i], dims[i + 1]), generator=gen, device="cuda") / math.sqrt(dims[i])).to(ptype)
               for i in range(case["layers"])]
    dout = None
    if case["mode"] == "train" and case["loss"] == "dense":
        dout = torch.randn((rows, dims[-1]), generator=gen, device="cuda").to(_DTYPE[case["dtype"]])
    # Magnitudes of the weight-normalised columns, around their initial 1.
    g = 1 + 0.1 * torch.randn(sum(dims[1:]), generator=gen, device="cuda")
    return x, weights, dout, g


def _model(case, weights, g):
    five = case["layers"] == 5
    if case["api"] == "wn":
        cls = fused_mlp5.FusedMLP5SoftplusWN if five else fused_mlp.FusedMLPSoftplusWN
    else:
        cls = fused_mlp5.FusedMLP5Softplus if five else fused_mlp.FusedMLPSoftplus
    sizes = {} if five else {"n_layers": case["layers"]}
    model = cls(D=case["d_in"], H=case["hidden"], out_features=case["d_out"], **sizes).to("cuda", weights[0].dtype)
    with torch.no_grad():
        if case["api"] == "wn":
            model.v_all.copy_(torch.cat([w.reshape(-1) for w in weights]))
            model.g_all.copy_(g)
        else:
            for p, w in zip(model.weights, weights):
                p.copy_(w)
    return model


def _train_step(case, model, x, dout):
    if case["amp"]:
        with torch.autocast("cuda", dtype=_DTYPE[case["dtype"]]):
            out = model(x)
    else:
        out = model(x)
    wrt = list(model.parameters()) + ([x] if case["x_grad"] else [])
    if dout is None:
        grads = torch.autograd.grad(out.sum(), wrt)
    else:
        grads = torch.autograd.grad(out, wrt, dout)
    return [out.detach(), *grads]


def prepare(case, seed):
    x, weights, dout, g = _inputs(case, seed)
    state = {"case": case, "x": x, "weights": weights, "dout": dout}
    if case["api"] != "launcher":
        state["model"] = _model(case, weights, g)
    if case["mode"] == "train":
        x.requires_grad_(case["x_grad"])
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                _train_step(case, state["model"], x, dout)
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["outputs"] = _train_step(case, state["model"], x, dout)
    return state


def run(state):
    case = state["case"]
    if case["graph"]:
        state["graph"].replay()
        return state["outputs"]
    if case["mode"] == "train":
        return _train_step(case, state["model"], state["x"], state["dout"])
    if case["api"] == "launcher":
        return kernel._fused_mlp_fwd(state["x"], *state["weights"])
    with torch.no_grad():
        return state["model"](state["x"])


def work(case):
    """Each input read once, each output written once; two operations per
    multiply-add, and in training two more products of the same size per
    layer (one for the first layer when x needs no gradient)."""
    dims, rows = _widths(case), case["rows"]
    es = 4 if case["dtype"] == "fp32" else 2
    xs = 4 if case["amp"] else es
    ps = 4 if case["api"] == "wn" else xs
    params = sum(a * b for a, b in zip(dims, dims[1:])) + (sum(dims[1:]) if case["api"] == "wn" else 0)
    macs = rows * sum(a * b for a, b in zip(dims, dims[1:]))
    nbytes = rows * (dims[0] * xs + dims[-1] * es) + params * ps
    flops = 2 * macs
    if case["mode"] == "train":
        nbytes += params * ps + (rows * dims[-1] * es if case["loss"] == "dense" else 0)
        nbytes += rows * dims[0] * xs if case["x_grad"] else 0
        flops += 4 * macs - (0 if case["x_grad"] else 2 * rows * dims[0] * dims[1])
    return {"bytes": nbytes, "flops": flops}


# About four times the largest relative error seen against `exact` over the
# ranges of `draw`, forward alone and with gradients: roundings of the hidden
# activations and of the data gradients to the element type; for fp32 the
# split of every operand into two bf16 halves.
_REL = {("infer", "fp16"): 2e-3, ("infer", "bf16"): 2e-2, ("infer", "fp32"): 4e-5,
        ("train", "fp16"): 4e-3, ("train", "bf16"): 3e-2, ("train", "fp32"): 5e-5}


def tolerance(case):
    return {"rel": _REL[case["mode"], case["dtype"]]}


def exact(case, seed):
    x, weights, dout, g = _inputs(case, seed)
    # Autocast rounds the fp32 input and weights to its type; the exact value
    # is that of the rounded tensors (weight norm keeps its parameters).
    dt = _DTYPE[case["dtype"]]
    x = x.to(dt).double().requires_grad_(case["x_grad"])
    grad = case["mode"] == "train"
    if case["api"] == "wn":
        dims = _widths(case)
        v_all = torch.cat([w.reshape(-1) for w in weights]).double().requires_grad_(grad)
        g_all = g.double().requires_grad_(grad)
        params = [v_all, g_all]
        vs = v_all.split([a * b for a, b in zip(dims, dims[1:])])
        gs = g_all.split(dims[1:])
        ws = []
        for i in range(case["layers"]):
            v = vs[i].view(dims[i], dims[i + 1])
            ws.append(gs[i] * v / v.norm(dim=0))
    else:
        ws = params = [w.to(dt).double().requires_grad_(grad) for w in weights]
    with torch.set_grad_enabled(grad):
        a = x
        for i, w in enumerate(ws):
            a = a @ w
            if i + 1 < len(ws):
                a = F.softplus(a)
    if not grad:
        return a
    wrt = params + ([x] if case["x_grad"] else [])
    up = torch.ones_like(a) if dout is None else dout.double()
    return [a.detach(), *torch.autograd.grad(a, wrt, up)]
