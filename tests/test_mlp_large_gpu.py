"""The MLP step on layers large enough for one launch per product.

Shapes on both head forms (the fused one, and logits, cross-entropy and G1 as
their own launches) with odd sizes, with and without dX (whose buffer the
weight-gradient slices use), an unaligned dX, and labels that are no class.
Every output is within the derived bound of the fp64 step, and within the
2e-5 of it, normwise, that the structured shapes hold.
"""
import numpy as np
import pytest

import fast_dl_amd.capi as capi
from tests.conftest import rng
from tests.gpu_helpers import dev, host, say, stream
from tests.mlp_bounds import exact_step, step_bounds, worst_ratio

pytestmark = pytest.mark.gpu

LR = 0.1
PARAMS = ("W1", "b1", "W2", "b2")


def _step(X, labels, params, dx_offset):
    import torch

    B, I = X.shape
    Hd, C = params[0].shape[1], params[2].shape[1]
    t = {k: dev(v.copy()) for k, v in zip(PARAMS, params)}
    for name, shape in dict(H=(B, Hd), logits=(B, C), G2=(B, C), G1=(B, Hd), dW1=(I, Hd),
                            db1=(Hd,), dW2=(Hd, C), db2=(C,), loss=(1,)).items():
        t[name] = torch.full(shape, float("nan"), device="cuda")
    dx = torch.full((B * I + 8,), float("nan"), device="cuda")
    dX, dl = dev(X), dev(labels)
    capi.mlp2_train_step(dX.data_ptr(), dl.data_ptr(), B, I, Hd, C, *(t[k].data_ptr() for k in PARAMS),
                         LR, *(t[k].data_ptr() for k in ("H", "logits", "G2", "G1", "dW1", "db1",
                                                         "dW2", "db2")),
                         dx.data_ptr() + 4 * dx_offset if dx_offset is not None else None,
                         t["loss"].data_ptr(), stream())
    out = {k: host(v) for k, v in t.items()}
    flat = host(dx)
    if dx_offset is None:
        assert np.all(np.isnan(flat))
        out["dX"] = None
    else:
        assert np.all(np.isnan(flat[:dx_offset])) and np.all(np.isnan(flat[dx_offset + B * I:]))
        out["dX"] = flat[dx_offset: dx_offset + B * I].reshape(B, I)
    return out


@pytest.mark.parametrize("B,I,Hd,C", [(3000, 1000, 256, 10), (2101, 71, 901, 18),
                                      (4097, 257, 401, 12), (1031, 132, 1024, 33),
                                      (2500, 52, 1000, 2100), (600, 784, 900, 7)])
@pytest.mark.parametrize("dx_offset", [0, 1, None])
def test_large_step(device, B, I, Hd, C, dx_offset):
    g = rng(B + I + Hd + C)
    X = g.random((B, I)).astype(np.float32)
    labels = g.integers(0, C, B).astype(np.int64)
    labels[::9] = [-1, C][B % 2]
    params = [(g.standard_normal(s) * k).astype(np.float32)
              for s, k in (((I, Hd), np.sqrt(2.0 / I)), (Hd, 0.1), ((Hd, C), np.sqrt(2.0 / Hd)),
                           (C, 0.1))]
    say(f"large step B={B} I={I} H={Hd} C={C} dx={dx_offset}")
    gpu = _step(X, labels, params, dx_offset)
    ex = exact_step(X, labels, *params, LR)
    ratios = worst_ratio(gpu, ex, step_bounds(X, labels, *params, LR, ex))
    assert max(ratios.values()) <= 1.0, ratios
    for k, v in gpu.items():
        # G1's and dX's elements where a ReLU mask sits on its kink answer to the bound alone
        if v is None or k in ("G1", "loss"):
            continue
        err = np.max(np.abs(v - ex[k])) / np.max(np.abs(ex[k]))
        assert err <= 2e-5, f"{k}: {err:.2e}"


def test_large_step_repeats_bit_for_bit(device):
    g = rng(5)
    B, I, Hd, C = 2048, 200, 700, 20
    X = g.random((B, I)).astype(np.float32)
    labels = g.integers(0, C, B).astype(np.int64)
    params = [(g.standard_normal(s) * 0.05).astype(np.float32)
              for s in ((I, Hd), (Hd,), (Hd, C), (C,))]
    say("large step twice")
    a, b = (_step(X, labels, params, 0) for _ in range(2))
    assert all(np.array_equal(a[k], b[k]) for k in a)


def test_large_step_without_dx(device):
    # without dX the step takes one launch per product only where dW1's tiles fill the GPU
    g = rng(8)
    B, I, Hd, C = 2300, 820, 810, 10
    X = g.random((B, I)).astype(np.float32)
    labels = g.integers(0, C, B).astype(np.int64)
    params = [(g.standard_normal(s) * k).astype(np.float32)
              for s, k in (((I, Hd), np.sqrt(2.0 / I)), (Hd, 0.1), ((Hd, C), np.sqrt(2.0 / Hd)),
                           (C, 0.1))]
    say(f"large step without dX B={B} I={I} H={Hd} C={C}")
    gpu = _step(X, labels, params, None)
    ex = exact_step(X, labels, *params, LR)
    ratios = worst_ratio(gpu, ex, step_bounds(X, labels, *params, LR, ex))
    assert max(ratios.values()) <= 1.0, ratios


@pytest.mark.parametrize("B,I,Hd,C", [(2, 4, (1 << 24) + 8, 3), (130, 260, 4100, 40),
                                      (64, 800, 2500, 2052)])
def test_large_step_wide_layers(device, B, I, Hd, C):
    """Bias gradients wider than the strips of the reduction launch take their own."""
    import torch

    g = torch.Generator(device="cuda").manual_seed(B + Hd)

    def rand(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * scale

    X, labels = rand(B, I), torch.arange(B, device="cuda") % C
    W1, b1, W2, b2 = rand(I, Hd, scale=I ** -0.5), rand(Hd), rand(Hd, C, scale=Hd ** -0.5), rand(C)
    new = {"W1": W1.clone(), "b1": b1.clone(), "W2": W2.clone(), "b2": b2.clone()}
    out = {n: torch.full(s, float("nan"), device="cuda")
           for n, s in dict(H=(B, Hd), logits=(B, C), G2=(B, C), G1=(B, Hd), dW1=(I, Hd),
                            db1=(Hd,), dW2=(Hd, C), db2=(C,), dX=(B, I), loss=(1,)).items()}
    say(f"large step, wide layers B={B} I={I} H={Hd} C={C}")
    capi.mlp2_train_step(X.data_ptr(), labels.data_ptr(), B, I, Hd, C,
                         *(t.data_ptr() for t in new.values()), LR,
                         *(t.data_ptr() for t in out.values()), stream())
    # fp64, from the step's own H and G1 masks on
    H = out["H"].double()
    assert torch.allclose(H, (X.double() @ W1.double() + b1).clamp_min(0), rtol=1e-5, atol=1e-5)
    logits = H @ W2.double() + b2
    p = torch.softmax(logits, 1)
    p[torch.arange(B), labels] -= 1.0
    G2 = p / B
    G1 = (G2 @ W2.double().t().contiguous()) * (H > 0)
    want = {"G2": G2, "G1": G1, "db2": G2.sum(0), "db1": G1.sum(0),
            "dW2": H.t().contiguous() @ G2, "dW1": X.double().t().contiguous() @ G1,
            "dX": G1 @ W1.double().t().contiguous()}
    # rounding errors of a sum of n terms add like a random walk's steps, eps * sqrt(n) / 3
    # of its norm at most; the gradients of logits pass theirs on
    tol = 5e-6 + 4e-8 * np.sqrt(max(B, I, Hd, C))
    for name, w in want.items():
        err = (out[name].double() - w).norm() / w.norm()
        assert err <= tol, f"{name}: {err:.2e}"
    for name, w, dw in (("W1", W1, "dW1"), ("b1", b1, "db1"), ("W2", W2, "dW2"), ("b2", b2, "db2")):
        step = LR * out[dw]
        assert torch.equal(new[name], w - step)
