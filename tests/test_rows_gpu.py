"""Row softmax and softmax cross-entropy at the edges of their row forms.

A row of up to 2048 columns sits in the registers of 4, 16 or 64 lanes (with
16-byte accesses where rows are 16-byte aligned and longer than 64 columns),
longer rows take a block each; the cross-entropy runs on one block or, with a
gradient buffer, on many with their loss sums kept in its first floats.
References are numpy in fp64.  Bounds: an exponential is within 2 ulp, its
argument's rounding adds eps * |z - max|, a sum of n terms n * eps at most.
"""
import numpy as np
import pytest

import fast_dl_amd.capi as capi
from tests.conftest import rng
from tests.gpu_helpers import dev, host, say, stream

pytestmark = pytest.mark.gpu

EPS = float(np.finfo(np.float32).eps)

# (rows, columns): both sides of every row form, with one block and with many
SHAPES = [(1, 1), (700, 1), (257, 4), (769, 4), (3, 5), (600, 16), (129, 17), (300, 64),
          (33, 65), (20, 68), (40, 128), (41, 129), (5, 256), (35, 257), (64, 260), (37, 512),
          (36, 513), (4, 1000), (2100, 1000), (50, 1023), (51, 1024), (34, 1025), (33, 1028),
          (7, 2047), (70, 2048), (2, 2049), (40, 2049), (3, 7000), (4500, 10),
          (17000, 66), (70000, 3), (3073, 1), (4100, 2051)]


def _softmax64(z):
    z = z.astype(np.float64)
    m = z.max(1, keepdims=True)
    e = np.exp(z - m)
    s = e.sum(1, keepdims=True)
    spread = np.minimum(m - z, 200.0)  # beyond it the probability is below fp32's smallest
    bound = (8.0 + spread + np.sum(e * spread, 1, keepdims=True) / s
             + np.minimum(z.shape[1], 64)) * EPS
    return e / s, np.log(s[:, 0]) + m[:, 0], bound


def loss_bound(z, lab):
    """Each row's share of the loss times the batch, and a bound on the mean's error."""
    batch, classes = z.shape
    z64 = z.astype(np.float64)
    m = z64.max(1)
    e = np.exp(z64 - m[:, None])
    s = e.sum(1)
    lse = np.log(s) + m
    at = np.flatnonzero((lab >= 0) & (lab < classes))
    shares = np.zeros(batch)
    shares[at] = lse[at] - z64[at, lab[at]]
    # a share: log(sum) off by the sum's relative error (exponentials within 2 ulp, their
    # arguments' rounding, its additions) and its own few roundings
    spread = np.minimum(m[:, None] - z64, 200.0)
    rel = 4.0 + np.sum(e * spread, 1) / s + min(classes, 64)
    size = np.abs(lse) + np.abs(z64).max(1) + 1.0
    # the mean: shares of one sign through at most `adds` additions (a lane's rows, the
    # exchanges and the waves of a block, the partial sums of up to 4096 blocks)
    adds = 60 + batch / 1024
    tol = np.sum((rel + 4.0 * size)[at]) + adds * np.abs(shares).sum()
    return shares, float(tol) * EPS / batch + 1e-30


def _offset(a, shift):
    """A device copy of `a` that starts `shift` floats past an allocation."""
    import torch

    buf = torch.empty(a.size + shift, device="cuda")
    view = buf[shift:].view(a.shape)
    view.copy_(dev(a))
    return view


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("shift", [0, 1])
def test_softmax_rows(device, rows, cols, shift):
    import torch

    z = (rng(rows * 3 + cols).standard_normal((rows, cols)) * 4).astype(np.float32)
    if cols > 2:
        z[::3, cols // 2] = -np.inf  # a masked column
    d, out = _offset(z, shift), _offset(np.full_like(z, np.nan), shift)
    say(f"softmax rows {rows}x{cols} shift={shift}")
    capi.softmax(d.data_ptr(), out.data_ptr(), rows, cols, stream())
    ref, _, bound = _softmax64(z)
    assert np.all(np.abs(host(out) - ref) <= bound * ref + 1e-37)
    capi.softmax(d.data_ptr(), d.data_ptr(), rows, cols, stream())  # in place
    assert torch.equal(d, out)


@pytest.mark.parametrize("batch,classes", SHAPES)
@pytest.mark.parametrize("shift", [0, 1])
def test_softmax_xent_rows(device, batch, classes, shift):
    import torch

    g = rng(batch * 7 + classes)
    z = (g.standard_normal((batch, classes)) * 3).astype(np.float32)
    lab = g.integers(0, classes, batch).astype(np.int64)
    lab[::5] = [-1, classes, 1 << 40][batch % 3]  # no class: left out of the loss
    d, dl = _offset(z, shift), dev(lab)
    grad = _offset(np.full_like(z, np.nan), shift)
    loss = torch.full((1,), float("nan"), device="cuda")
    say(f"softmax_xent rows {batch}x{classes} shift={shift}")
    capi.softmax_xent(d.data_ptr(), dl.data_ptr(), loss.data_ptr(), grad.data_ptr(), batch,
                      classes, stream())
    p, lse, bound = _softmax64(z)
    shares, loss_tol = loss_bound(z, lab)
    at = np.flatnonzero((lab >= 0) & (lab < classes))
    ref = p.copy()
    ref[at, lab[at]] -= 1.0
    grad_tol = (bound * p + 3 * EPS * np.abs(ref)) / batch + 1e-37
    assert abs(float(host(loss)[0]) - shares.sum() / batch) <= loss_tol
    assert np.all(np.abs(host(grad) - ref / batch) <= grad_tol)
    # loss alone, gradient alone, and the gradient over the logits: the same rows
    only = torch.full((1,), float("nan"), device="cuda")
    capi.softmax_xent(d.data_ptr(), dl.data_ptr(), only.data_ptr(), None, batch, classes, stream())
    assert abs(float(host(only)[0]) - shares.sum() / batch) <= loss_tol
    alone = torch.full_like(grad, float("nan"))
    capi.softmax_xent(d.data_ptr(), dl.data_ptr(), None, alone.data_ptr(), batch, classes,
                      stream())
    assert np.all(np.abs(host(alone) - ref / batch) <= grad_tol)
    capi.softmax_xent(d.data_ptr(), dl.data_ptr(), only.data_ptr(), d.data_ptr(), batch, classes,
                      stream())
    assert abs(float(host(only)[0]) - shares.sum() / batch) <= loss_tol
    assert np.all(np.abs(host(d) - ref / batch) <= grad_tol)


@pytest.mark.parametrize("batch,classes", [(256, 10), (1000, 100), (8192, 1500), (300, 4000),
                                           (5000, 2100)])
def test_loss_error_is_that_of_short_sums(device, batch, classes):
    """Over seeds, the loss is off by about its last place, with a gradient and without.

    Shares and sums rounded independently leave about half a unit in the last place
    (6e-8) of a sum of few levels; one long chain of additions shows as several.
    """
    import torch

    err = {"both": [], "loss": []}
    say(f"loss error {batch}x{classes}")
    for seed in range(16):
        g = torch.Generator(device="cuda").manual_seed(seed)
        z = torch.randn(batch, classes, generator=g, device="cuda") * 2
        y = torch.randint(0, classes, (batch,), generator=g, device="cuda")
        at = torch.arange(batch, device="cuda")
        want = float(-torch.log_softmax(z.double(), 1)[at, y].mean())
        loss, grad = torch.empty(1, device="cuda"), torch.empty_like(z)
        for form in err:
            capi.softmax_xent(z.data_ptr(), y.data_ptr(), loss.data_ptr(),
                              grad.data_ptr() if form == "both" else None, batch, classes,
                              stream())
            err[form].append((float(host(loss)[0]) - want) / want)
    for form, e in err.items():
        assert np.sqrt(np.mean(np.square(e))) <= 1.2e-7, form


def test_loss_keeps_infinities(device):
    # a row whose label is masked out loses without bound; the others' losses do not hide it
    import torch

    for batch, classes in ((40, 10), (300, 2050), (5000, 100)):
        z = rng(classes).standard_normal((batch, classes)).astype(np.float32)
        lab = np.zeros(batch, np.int64)
        z[batch // 2, 0] = -np.inf
        d, dl, loss = dev(z), dev(lab), torch.zeros(1, device="cuda")
        say(f"loss infinity {batch}x{classes}")
        for grad in (None, torch.empty_like(d)):
            capi.softmax_xent(d.data_ptr(), dl.data_ptr(), loss.data_ptr(),
                              grad.data_ptr() if grad is not None else None, batch, classes,
                              stream())
            assert float(host(loss)[0]) == np.inf


# both sides of the lines between strips of 4 columns and blocks of 32
@pytest.mark.parametrize("rows,cols", [(2048, 64), (2049, 64), (2499, 1024), (2500, 1024),
                                       (2600, 769), (3000, 1001), (2999, 333), (2100, 2044),
                                       (2100, 2048), (2100, 2049), (16384, 1056), (4000, 512)])
@pytest.mark.parametrize("shift", [0, 1, 4])
def test_colsum_forms(device, rows, cols, shift):
    import torch

    x = rng(rows + cols + 1).standard_normal((rows, cols)).astype(np.float32)
    d = _offset(x, shift)
    out = torch.full((cols + 1,), float("nan"), device="cuda")
    say(f"colsum forms {rows}x{cols} shift={shift}")
    capi.colsum(d.data_ptr(), out.data_ptr(), rows, cols, stream())
    # the longer of the two forms' chains: one of eight row groups of a block
    bound = (rows / 8 + 16) * EPS * np.abs(x).astype(np.float64).sum(0)
    assert np.all(np.abs(host(out)[:cols] - x.astype(np.float64).sum(0)) <= bound)
    assert np.isnan(host(out)[cols])


@pytest.mark.parametrize("rows,cols", [(2049, 1), (2049, 3), (3000, 4), (2100, 34), (4096, 36),
                                       (5119, 100), (9000, 257), (30001, 8)])
@pytest.mark.parametrize("shift", [0, 1])
def test_colsum_tall(device, rows, cols, shift):
    import torch

    x = rng(rows + cols).standard_normal((rows, cols)).astype(np.float32)
    d = _offset(x, shift)
    out = torch.full((cols + 1,), float("nan"), device="cuda")
    say(f"colsum tall {rows}x{cols} shift={shift}")
    capi.colsum(d.data_ptr(), out.data_ptr(), rows, cols, stream())
    # a thread adds every 1024th row, then 6 exchanges and 16 waves
    depth = rows / 1024 + 24
    bound = depth * EPS * np.abs(x).astype(np.float64).sum(0)
    assert np.all(np.abs(host(out)[:cols] - x.astype(np.float64).sum(0)) <= bound)
    assert np.isnan(host(out)[cols])


@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1027, 65541, (8 << 20) + 5])
@pytest.mark.parametrize("shift", [0, 1])
def test_elementwise(device, n, shift):
    import torch

    g = rng(n)
    a, b = (g.standard_normal(n).astype(np.float32) for _ in range(2))
    b[:: 7], b[:: 11] = 0.0, -0.0
    a[:: 13] = np.nan
    da, db = _offset(a, shift), _offset(b, shift)
    out = _offset(np.zeros(n + 4, np.float32), shift)
    say(f"elementwise n={n} shift={shift}")
    capi.relu(da.data_ptr(), out.data_ptr(), n, stream())
    assert np.array_equal(host(out)[:n], np.fmax(np.float32(0), a))
    capi.relu_backward(da.data_ptr(), db.data_ptr(), out.data_ptr(), n, stream())
    assert np.array_equal(host(out)[:n], np.where(b > 0, a, np.float32(0)), equal_nan=True)
    capi.sgd_update(db.data_ptr(), da.data_ptr(), 0.3, n, stream())
    assert np.array_equal(host(db), b - np.float32(0.3) * a, equal_nan=True)
    assert torch.all(out[n:] == 0)
