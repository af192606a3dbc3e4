"""The work a user of this framework has it do, as cases that can be timed and checked.

Six kinds of call, each through the C-ABI as `fast_dl_amd.capi` binds it, with
device buffers the caller owns (the inputs and the outputs, the workspace a
GEMM asks for, the step's intermediates):

* ``gemm``   -- one product: square and rectangular, every layout, batches, few rows;
* ``layer``  -- a Linear + ReLU layer's training pass, as nn.Sequential and autograd run it;
* ``loss``   -- softmax probabilities, and the cross-entropy loss with its gradient;
* ``step``   -- the two-layer MLP training step;
* ``epoch``  -- an epoch's IDX rows gathered into fp32 and their labels.

``listed()`` spans the sizes from a 256 x 10 loss to the 4096^3 product;
``draw`` fills in the ranges between and around them.
"""
import math

import torch

from fast_dl_amd import capi

LR = 1e-3
EPILOGUES = {"none": capi.EPILOGUE_NONE, "bias": capi.EPILOGUE_BIAS,
             "bias_relu": capi.EPILOGUE_BIAS_RELU, "relu": capi.EPILOGUE_RELU,
             "relu_grad": capi.EPILOGUE_RELU_GRAD}


def listed():
    return [
        # the headline product
        gemm("gemm_4096", 4096, 4096, 4096),
        # no size a multiple of a tile or of 4: predicated edges, 4-byte rows
        gemm("gemm_1023_bias_relu", 1023, 1023, 1023, epilogue="bias_relu"),
        # attention scores: 64 small problems, the second operand transposed
        gemm("scores_64x128x128x64_nt", 128, 128, 64, layout="nt", batch=64),
        # one row through a 4096-wide layer: serving a single request
        gemm("serve_1x4096", 1, 4096, 4096, epilogue="bias_relu"),
        # the same layer for a small batch of requests
        gemm("serve_32x4096", 32, 4096, 4096, epilogue="bias_relu"),
        # the MNIST network's first layer, one mini-batch
        {"name": "layer_256x784x256", "kind": "layer", "rows": 256, "fan_in": 784, "fan_out": 256},
        # the same layer over the whole training set (full-batch gradient)
        {"name": "layer_60000x784x256", "kind": "layer", "rows": 60000, "fan_in": 784,
         "fan_out": 256},
        # the ten-class loss of one mini-batch: the smallest call
        {"name": "loss_256x10", "kind": "loss", "rows": 256, "classes": 10},
        # a thousand classes, a large batch
        {"name": "loss_4096x1000", "kind": "loss", "rows": 4096, "classes": 1000},
        # the MNIST training step
        {"name": "step_256x784x256x10", "kind": "step", "rows": 256, "fan_in": 784, "hidden": 256,
         "classes": 10},
        # a wider network on a larger batch, more classes than the fused heads take
        {"name": "step_2048x784x1024x100", "kind": "step", "rows": 2048, "fan_in": 784,
         "hidden": 1024, "classes": 100},
        # one epoch of the MNIST set in shuffled order
        {"name": "epoch_60000x784", "kind": "epoch", "rows": 60000, "row_bytes": 784},
    ]


def gemm(name, m, n, k, layout="nn", batch=1, epilogue="none"):
    case = {"kind": "gemm", "layout": layout, "batch": batch, "m": m, "n": n, "k": k,
            "epilogue": epilogue}
    return dict(case, name=name) if name else case


def draw(rng):
    def size(low, high):
        """Spread over the logarithm; half of them multiples of 16, the rest as they fall."""
        v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
        return max(low, v - v % 16) if rng.random() < 0.5 else v

    kind = rng.choice(["product", "product", "scores", "serve", "layer", "layer", "loss", "loss",
                       "step", "step", "epoch"])
    if kind == "product":
        return gemm(None, size(64, 4096), size(64, 4096), size(64, 4096),
                    layout=rng.choice(["nn", "nn", "nt", "tn"]),
                    epilogue=rng.choice(["none", "none", "bias", "bias_relu", "relu",
                                         "relu_grad"]))
    if kind == "scores":
        return gemm(None, size(32, 256), size(32, 256), size(16, 128), batch=size(8, 128),
                    layout=rng.choice(["nn", "nt"]))
    if kind == "serve":
        return gemm(None, size(1, 64), size(512, 8192), size(512, 8192),
                    epilogue=rng.choice(["bias", "bias_relu"]))
    if kind == "layer":
        return {"kind": "layer", "rows": size(32, 60000), "fan_in": size(32, 1024),
                "fan_out": size(10, 1024)}
    if kind == "loss":
        return {"kind": "loss", "rows": size(16, 8192), "classes": size(2, 1500)}
    if kind == "step":
        return {"kind": "step", "rows": size(16, 4096), "fan_in": size(64, 1024),
                "hidden": size(16, 1024), "classes": size(2, 128)}
    return {"kind": "epoch", "rows": size(64, 60000), "row_bytes": size(100, 3072)}


def work(case):
    """What a pass cannot do without: inputs read once, outputs written once, the products."""
    f = 4
    if case["kind"] == "gemm":
        m, n, k, b = case["m"], case["n"], case["k"], case["batch"]
        extra = {"none": 0, "relu": 0, "bias": n, "bias_relu": n,
                 "relu_grad": b * m * n}[case["epilogue"]]
        return {"bytes": f * (b * (m * k + k * n + m * n) + extra), "flops": 2.0 * b * m * n * k}
    if case["kind"] == "layer":
        r, i, o = case["rows"], case["fan_in"], case["fan_out"]
        # read x, dh, W, b; write y, h, dy, dx, dW, db, W, b
        return {"bytes": f * (2 * r * i + 4 * r * o + 3 * i * o + 3 * o),
                "flops": 6.0 * r * i * o}
    if case["kind"] == "loss":
        r, c = case["rows"], case["classes"]
        # read logits and labels; write probabilities, gradient and loss
        return {"bytes": f * 3 * r * c + 8 * r + f, "flops": 10.0 * r * c}
    if case["kind"] == "step":
        r, i, h, c = case["rows"], case["fan_in"], case["hidden"], case["classes"]
        # read x, labels and the parameters; write H, logits, G2, G1, dX, the gradients
        # and the parameters
        params = i * h + h + h * c + c
        return {"bytes": f * (2 * r * i + 2 * r * h + 2 * r * c + 3 * params) + 8 * r,
                "flops": 6.0 * r * h * (i + c)}
    r, b = case["rows"], case["row_bytes"]
    return {"bytes": r * (5.0 * b + 17.0), "flops": 1.0 * r * b}


# --------------------------------------------------------------------- inputs


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(scale)


def _pixels(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float32)


def _empty(*shape):
    return torch.empty(*shape, device="cuda", dtype=torch.float32)


def _labels(g, rows, classes):
    return torch.randint(0, classes, (rows,), generator=g, device="cuda", dtype=torch.int64)


def _operands(case, g):
    m, n, k, b = case["m"], case["n"], case["k"], case["batch"]
    layout, epi = case["layout"], case["epilogue"]
    # many small problems hold scores' operands (N(0, 1/8)), the others N(0, 1)
    scale = 1.0 if b == 1 else 0.125
    A = _normal(g, *((b, k, m) if layout[0] == "t" else (b, m, k)), scale=scale)
    B = _normal(g, *((b, n, k) if layout[1] == "t" else (b, k, n)), scale=scale)
    bias = _normal(g, n, scale=0.1) if epi.startswith("bias") else None
    aux = _normal(g, b, m, n) if epi == "relu_grad" else None
    return A, B, bias, aux


def _layer_inputs(case, g):
    r, i, o = case["rows"], case["fan_in"], case["fan_out"]
    x = _pixels(g, r, i)
    W = _normal(g, i, o, scale=math.sqrt(2.0 / i))
    b = _normal(g, o, scale=0.1)
    dh = _normal(g, r, o, scale=0.1 / r)  # what a mean loss sends back
    # On the ReLU's kink the rounding of y decides whether dh passes: none comes back there
    # (the window also covers what one update moves y by).
    y = x.double() @ W.double() + b.double()
    return x, W, b, dh.mul_(y.abs_() > 0.01)


def _loss_inputs(case, g):
    r, c = case["rows"], case["classes"]
    return _normal(g, r, c, scale=2.0), _labels(g, r, c)


def _step_inputs(case, g):
    r, i, h, c = case["rows"], case["fan_in"], case["hidden"], case["classes"]
    W1 = _normal(g, i, h, scale=math.sqrt(2.0 / i))
    b1 = _normal(g, h, scale=0.1)
    W2 = _normal(g, h, c, scale=math.sqrt(2.0 / h))
    b2 = _normal(g, c, scale=0.1)
    # Rows with a hidden unit on the ReLU's kink go last, and are left out: there the rounding
    # of one sum decides whether a whole gradient passes.
    x = _pixels(g, r + r // 8 + 64, i)
    clear = ((x.double() @ W1.double() + b1.double()).abs_() > 2e-5).all(1)
    x = x[torch.argsort((~clear).to(torch.int32), stable=True)[:r]].contiguous()
    return x, _labels(g, r, c), W1, b1, W2, b2


def _epoch_inputs(case, g):
    r, b = case["rows"], case["row_bytes"]
    images = torch.randint(0, 256, (r, b), generator=g, device="cuda", dtype=torch.uint8)
    labels = torch.randint(0, 10, (r,), generator=g, device="cuda", dtype=torch.uint8)
    index = torch.randperm(r, generator=g, device="cuda")
    return images, labels, index


# -------------------------------------------------------------------- program


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _ptr(t):
    return t.data_ptr() if t is not None else None


def _gemm_call(ta, tb, m, n, k, A, B, C, batch=1, bias=None, aux=None, epilogue=0):
    """One product as a program calls it: packed operands, with the workspace it asks for."""
    need = capi.workspace_size(ta, tb, m, n, k, batch)
    ws = torch.empty(need, device="cuda", dtype=torch.uint8) if need else None
    args = (ta, tb, m, n, k, A.data_ptr(), m if ta else k, m * k, B.data_ptr(), k if tb else n,
            k * n, C.data_ptr(), n, m * n, batch, _ptr(bias), _ptr(aux), epilogue, _ptr(ws), need,
            _stream())
    return args, ws


def prepare(case, seed):
    g = _generator(seed)
    if case["kind"] == "gemm":
        A, B, bias, aux = _operands(case, g)
        C = _empty(case["batch"], case["m"], case["n"])
        args, ws = _gemm_call(int(case["layout"][0] == "t"), int(case["layout"][1] == "t"),
                              case["m"], case["n"], case["k"], A, B, C, case["batch"], bias, aux,
                              EPILOGUES[case["epilogue"]])
        return {"run": _run_gemm, "args": args, "C": C, "keep": (A, B, bias, aux, ws)}
    if case["kind"] == "layer":
        return _prepare_layer(case, g)
    if case["kind"] == "loss":
        z, labels = _loss_inputs(case, g)
        probs, grad, loss = torch.empty_like(z), torch.empty_like(z), _empty(1)
        r, c, s = case["rows"], case["classes"], _stream()
        return {"run": _run_loss, "probs": probs, "grad": grad, "loss": loss, "keep": (z, labels),
                "softmax": (z.data_ptr(), probs.data_ptr(), r, c, s),
                "xent": (z.data_ptr(), labels.data_ptr(), loss.data_ptr(), grad.data_ptr(), r, c,
                         s)}
    if case["kind"] == "step":
        return _prepare_step(case, g)
    images, labels, index = _epoch_inputs(case, g)
    r, b = case["rows"], case["row_bytes"]
    x, y = _empty(r, b), torch.empty(r, device="cuda", dtype=torch.int64)
    return {"run": _run_epoch, "x": x, "y": y, "keep": (images, labels, index),
            "args": (images.data_ptr(), labels.data_ptr(), r, b, index.data_ptr(), r, 255.0,
                     x.data_ptr(), y.data_ptr(), _stream())}


def _prepare_layer(case, g):
    r, i, o = case["rows"], case["fan_in"], case["fan_out"]
    x, W, b, dh = _layer_inputs(case, g)
    y, h, dy = _empty(r, o), _empty(r, o), _empty(r, o)
    dx, dW, db = _empty(r, i), _empty(i, o), _empty(o)
    s = _stream()
    forward, ws_f = _gemm_call(0, 0, r, o, i, x, W, y, bias=b, epilogue=capi.EPILOGUE_BIAS)
    input_grad, ws_x = _gemm_call(0, 1, r, i, o, dy, W, dx)
    weight_grad, ws_w = _gemm_call(1, 0, i, o, r, x, dy, dW)
    return {"run": _run_layer, "outputs": (y, h, dy, dx, dW, db, W, b),
            "forward": forward, "relu": (y.data_ptr(), h.data_ptr(), r * o, s),
            "relu_grad": (dh.data_ptr(), h.data_ptr(), dy.data_ptr(), r * o, s),
            "input_grad": input_grad, "weight_grad": weight_grad,
            "bias_grad": (dy.data_ptr(), db.data_ptr(), r, o, s),
            "sgd_w": (W.data_ptr(), dW.data_ptr(), LR, i * o, s),
            "sgd_b": (b.data_ptr(), db.data_ptr(), LR, o, s),
            "keep": (x, dh, ws_f, ws_x, ws_w)}


def _prepare_step(case, g):
    r, i, h, c = case["rows"], case["fan_in"], case["hidden"], case["classes"]
    x, labels, W1, b1, W2, b2 = _step_inputs(case, g)
    H, logits, G2, G1 = _empty(r, h), _empty(r, c), _empty(r, c), _empty(r, h)
    dW1, db1, dW2, db2 = _empty(i, h), _empty(h), _empty(h, c), _empty(c)
    dX, loss = _empty(r, i), _empty(1)
    args = (x.data_ptr(), labels.data_ptr(), r, i, h, c, W1.data_ptr(), b1.data_ptr(),
            W2.data_ptr(), b2.data_ptr(), LR, H.data_ptr(), logits.data_ptr(), G2.data_ptr(),
            G1.data_ptr(), dW1.data_ptr(), db1.data_ptr(), dW2.data_ptr(), db2.data_ptr(),
            dX.data_ptr(), loss.data_ptr(), _stream())
    return {"run": _run_step, "args": args, "keep": (x, labels),
            "outputs": {"W1": W1, "b1": b1, "W2": W2, "b2": b2, "H": H, "logits": logits,
                        "G2": G2, "G1": G1, "dW1": dW1, "db1": db1, "dW2": dW2, "db2": db2,
                        "dX": dX, "loss": loss}}


def run(state):
    return state["run"](state)


def _run_gemm(state):
    capi.sgemm_ex_ws(*state["args"])
    return state["C"]


def _run_layer(state):
    capi.sgemm_ex_ws(*state["forward"])
    capi.relu(*state["relu"])
    capi.relu_backward(*state["relu_grad"])
    capi.sgemm_ex_ws(*state["input_grad"])
    capi.sgemm_ex_ws(*state["weight_grad"])
    capi.colsum(*state["bias_grad"])
    capi.sgd_update(*state["sgd_w"])
    capi.sgd_update(*state["sgd_b"])
    return state["outputs"]


def _run_loss(state):
    capi.softmax(*state["softmax"])
    capi.softmax_xent(*state["xent"])
    return state["probs"], state["grad"], state["loss"]


def _run_step(state):
    capi.mlp2_train_step(*state["args"])
    return state["outputs"]


def _run_epoch(state):
    capi.idx_gather(*state["args"])
    return state["x"], state["y"]


# ------------------------------------------------------------------- accuracy


def tolerance(case):
    """fp32 sums in another order.

    About four times the error against fp64: a product's grows with the length
    of its sums, the others' with their longest (the batch, or the layer's
    width), and the training step's carries through its layers.
    """
    if case["kind"] == "epoch":
        return "exact"  # one correctly rounded division per byte; whole labels
    if case["kind"] == "gemm":
        longest = case["k"]
    elif case["kind"] == "layer":
        longest = max(case["rows"], case["fan_in"], case["fan_out"])
    elif case["kind"] == "loss":
        return {"rel": 5e-7, "max": 1e-5}
    else:
        longest = max(case["rows"], case["fan_in"], case["hidden"])
    rel = 4e-7 + 7e-8 * math.sqrt(longest)
    return {"rel": rel, "max": 20 * rel}


def exact(case, seed):
    g = _generator(seed)
    if case["kind"] == "gemm":
        A, B, bias, aux = _operands(case, g)
        A, B = A.double(), B.double()
        A = A.transpose(1, 2).contiguous() if case["layout"][0] == "t" else A
        B = B.transpose(1, 2).contiguous() if case["layout"][1] == "t" else B
        C = torch.stack([a @ b for a, b in zip(A, B)])
        if bias is not None:
            C = C + bias.double()
        if case["epilogue"] in ("relu", "bias_relu"):
            C = C.clamp_min(0.0)
        return C * (aux > 0) if aux is not None else C
    if case["kind"] == "layer":
        x, W, b, dh = (t.double() for t in _layer_inputs(case, g))
        y = x @ W + b
        dy = dh * (y > 0)
        dW, db = x.t().contiguous() @ dy, dy.sum(0)
        dx = dy @ W.t().contiguous()
        return y, y.clamp_min(0.0), dy, dx, dW, db, W - LR * dW, b - LR * db
    if case["kind"] == "loss":
        z, labels = _loss_inputs(case, g)
        z = z.double()
        p = torch.softmax(z, 1)
        at = torch.arange(case["rows"], device="cuda")
        loss = -torch.log_softmax(z, 1)[at, labels].mean().reshape(1)
        grad = p.clone()
        grad[at, labels] -= 1.0
        return p, grad / case["rows"], loss
    if case["kind"] == "step":
        x, labels, *params = _step_inputs(case, g)
        x, (W1, b1, W2, b2) = x.double(), (t.double() for t in params)
        H = (x @ W1 + b1).clamp_min(0.0)
        logits = H @ W2 + b2
        at = torch.arange(case["rows"], device="cuda")
        G2 = torch.softmax(logits, 1)
        loss = -torch.log_softmax(logits, 1)[at, labels].mean().reshape(1)
        G2[at, labels] -= 1.0
        G2 /= case["rows"]
        G1 = (G2 @ W2.t().contiguous()) * (H > 0)
        dW1, db1 = x.t().contiguous() @ G1, G1.sum(0)
        dW2, db2 = H.t().contiguous() @ G2, G2.sum(0)
        dX = G1 @ W1.t().contiguous()
        return {"W1": W1 - LR * dW1, "b1": b1 - LR * db1, "W2": W2 - LR * dW2, "b2": b2 - LR * db2,
                "H": H, "logits": logits, "G2": G2, "G1": G1, "dW1": dW1, "db1": db1, "dW2": dW2,
                "db2": db2, "dX": dX, "loss": loss}
    images, labels, index = _epoch_inputs(case, g)
    return images[index].double() / 255.0, labels[index].to(torch.int64)
