"""GPU parity of the MLP training step (forward, MSE, backward) against
oracle/train.py.

Bar: loss within 1e-4 relative; per layer, ||dW - ref||_F <= 1e-2 ||ref||_F and
likewise for db (the GPU rounds g = 2 (y - t) and every propagated gradient to
fp16, the oracle keeps float64).  At the full C5 size: the same bars against
the torch-CPU restatement of the oracle, the loss equals the mean squared error
of the forward path, and the gradient of the whole set equals the
point-weighted mean of the gradients of its two halves.

The forward sums in a different fp32 order than the oracle, so a few
activations round to a neighbouring fp16 value; where that flips a ReLU mask
(an activation at zero on one side only) the gradient of that one point
differs entirely.  The 1e-2 bars hold for about a thousand points or more,
where one such point weighs little."""
import numpy as np
import pytest
import torch

import rdv_project_amd as rdv
from oracle import train as T
from rdv_project_amd import workloads as WL

pytestmark = pytest.mark.gpu


def _chain(layers):
    m = None
    for i, (w, b) in enumerate(layers):
        lin = rdv.linear(w.cuda(), b.cuda(), f16=True)
        m = lin if m is None else m >> lin
        if i + 1 < len(layers):
            m = m >> rdv.relu
    return m


def _fro(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def _check(loss, grads, ref_loss, ref_grads, what):
    assert abs(float(loss) - ref_loss) <= 1e-4 * abs(ref_loss), f"{what}: loss {float(loss)} vs {ref_loss}"
    for l, ((dw, db), (rw, rb)) in enumerate(zip(grads, ref_grads)):
        ew, eb = _fro(dw.cpu().numpy(), rw), _fro(db.cpu().numpy(), rb)
        assert np.isfinite(dw.cpu().numpy()).all() and np.isfinite(db.cpu().numpy()).all()
        assert ew <= 1e-2 and eb <= 1e-2, f"{what}: layer {l} relative error dW {ew:.3g}, db {eb:.3g}"


@pytest.mark.parametrize("n", [4096, 1000, 4167])  # 4167: 131 tiles, the last 64-point pair tile half past n
def test_c5_shape_matches_oracle(n):
    x, t, layers = WL.c5(n)
    layers = [(w, torch.randn(w.shape[0], generator=torch.Generator().manual_seed(i)) * 0.1)
              for i, (w, _) in enumerate(layers)]  # non-zero biases exercise db and the bias path
    m = _chain(layers)
    loss, grads = rdv.mse_backward(m, x.cuda(), t.cuda())
    torch.cuda.synchronize()
    ref_loss, ref_grads = T.mse_grads(x.float().numpy(), [(w.numpy(), b.numpy()) for w, b in layers], t.numpy())
    _check(loss.item(), grads, ref_loss, ref_grads, f"C5 n={n}")


def test_other_widths_and_tail():
    g = torch.Generator().manual_seed(21)
    dims = [16, 64, 32, 8]
    layers = []
    for i in range(3):
        lim = (6.0 / dims[i]) ** 0.5
        layers.append(((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) * lim,
                       torch.randn(dims[i + 1], generator=g) * 0.1))
    layers = [(w.half().float(), b) for w, b in layers]
    x = torch.randn(777, 16, generator=g).half()
    t = torch.randn(777, 8, generator=g)
    loss, grads = rdv.mse_backward(_chain(layers), x.cuda(), t.cuda())
    ref_loss, ref_grads = T.mse_grads(x.float().numpy(), [(w.numpy(), b.numpy()) for w, b in layers], t.numpy())
    _check(loss.item(), grads, ref_loss, ref_grads, "16-64-32-8")


@pytest.mark.parametrize("dims,n", [
    ([48, 128, 128, 128, 128, 128, 128, 8], 1500),  # two forward groups (the second on a stored input), odd L, 8-wide head
    ([32, 96, 64, 128, 24], 333),                   # even L, a 24-wide head (padded to 32 in the gradient buffer)
])
def test_generic_chains(dims, n):
    g = torch.Generator().manual_seed(len(dims) * 1000 + n)
    layers = []
    for i in range(len(dims) - 1):
        lim = (6.0 / dims[i]) ** 0.5
        layers.append((((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) * lim).half().float(),
                       torch.randn(dims[i + 1], generator=g) * 0.1))
    x = torch.randn(n, dims[0], generator=g).half()
    t = torch.randn(n, dims[-1], generator=g)
    loss, grads = rdv.mse_backward(_chain(layers), x.cuda(), t.cuda())
    ref_loss, ref_grads = T.mse_grads(x.float().numpy(), [(w.numpy(), b.numpy()) for w, b in layers], t.numpy())
    _check(loss.item(), grads, ref_loss, ref_grads, "-".join(map(str, dims)))


def test_each_call_returns_its_own_loss():
    """Two calls on different data return two loss tensors holding two losses
    (a list of un-read losses keeps every step's value); a caller-supplied
    loss buffer is the one written."""
    x, t, layers = WL.c5(2048)
    m = _chain(layers)
    xd, td = x.cuda(), t.cuda()
    la, _ = rdv.mse_backward(m, xd, td)
    lb, _ = rdv.mse_backward(m, xd, td * 2.0 + 1.0)
    assert la is not lb and la.data_ptr() != lb.data_ptr()
    ref_a, _ = T.mse_grads(x.float().numpy(), [(w.numpy(), b.numpy()) for w, b in layers], t.numpy())
    ref_b, _ = T.mse_grads(x.float().numpy(), [(w.numpy(), b.numpy()) for w, b in layers], t.numpy() * 2.0 + 1.0)
    assert abs(la.item() - ref_a) <= 1e-4 * abs(ref_a) and abs(lb.item() - ref_b) <= 1e-4 * abs(ref_b)
    own = torch.full((), -1.0, device="cuda")
    lc, _ = rdv.mse_backward(m, xd, td, loss=own)
    assert lc is own and abs(own.item() - ref_a) <= 1e-4 * abs(ref_a)


def test_unsupported_chain_raises():
    layers = [(torch.zeros(64, 3), torch.zeros(64)), (torch.zeros(4, 64), torch.zeros(4))]
    with pytest.raises(NotImplementedError):
        rdv.mse_backward(_chain(layers), torch.zeros(64, 3).cuda(), torch.zeros(64, 4).cuda())


def test_c5_full_config_properties():
    x, t, layers = WL.c5()
    n = x.shape[0]
    m = _chain(layers)
    xd, td = x.cuda(), t.cuda()
    loss, grads = rdv.mse_backward(m, xd, td)
    full = [(dw.clone(), db.clone()) for dw, db in grads]
    loss = loss.item()
    # the loss is the forward's mean squared error
    y = m(rdv.wrap(xd.float())).as_tensor("torch")
    mse = torch.mean((y.double() - td.double()) ** 2).item()
    assert abs(loss - mse) <= 1e-4 * mse, f"loss {loss} vs forward MSE {mse}"
    # the gradient of the set is the point-weighted mean of the gradients of its halves
    h = n // 2
    _, ga = rdv.mse_backward(m, xd[:h], td[:h])
    ga = [(dw.clone(), db.clone()) for dw, db in ga]
    _, gb = rdv.mse_backward(m, xd[h:], td[h:])
    for l, ((fw, fb), (aw, ab), (bw, bb)) in enumerate(zip(full, ga, gb)):
        cw = (aw.double() * h + bw.double() * (n - h)) / n
        cb = (ab.double() * h + bb.double() * (n - h)) / n
        assert torch.isfinite(fw).all() and torch.isfinite(fb).all()
        ew = (torch.linalg.norm(fw.double() - cw) / torch.linalg.norm(cw)).item()
        eb = (torch.linalg.norm(fb.double() - cb) / torch.linalg.norm(cb)).item()
        assert ew <= 1e-4 and eb <= 1e-4, f"layer {l}: halves disagree ({ew:.3g}, {eb:.3g})"


@pytest.mark.timeout(300)  # ~3 TFLOP of CPU work: ~15 s on 16 cores, longer on fewer
def test_c5_full_config_against_cpu_restatement():
    """The whole C5 step (4,194,304 points) against oracle/torch_cpu.train_step
    (the oracle's computation as torch-CPU fp32 with autograd, checked against
    it by test_oracle_torch_cpu), summed over 262,144-point chunks weighted by
    their share of the points; the bars of the oracle comparisons above."""
    import os
    from oracle import torch_cpu as TC
    x, t, layers = WL.c5()
    n = x.shape[0]
    m = _chain(layers)
    loss, grads = rdv.mse_backward(m, x.cuda(), t.cuda())
    loss = loss.item()
    grads = [(dw.cpu().double().numpy(), db.cpu().double().numpy()) for dw, db in grads]
    threads = torch.get_num_threads()
    torch.set_num_threads(max(1, min(16, len(os.sched_getaffinity(0)))))
    try:
        params = [(w.float().clone().requires_grad_(True), b.float().clone().requires_grad_(True))
                  for w, b in layers]
        ref_loss = 0.0
        ref = [(np.zeros(w.shape), np.zeros(b.shape)) for w, b in params]
        xf = x.float()
        for i in range(0, n, 262144):
            c = min(262144, n - i)
            lc = TC.train_step(xf[i:i + c], t[i:i + c], params)
            ref_loss += lc.item() * c / n
            for (rw, rb), (w, b) in zip(ref, params):
                rw += w.grad.double().numpy() * (c / n)
                rb += b.grad.double().numpy() * (c / n)
    finally:
        torch.set_num_threads(threads)
    _check(loss, [(torch.from_numpy(dw), torch.from_numpy(db)) for dw, db in grads], ref_loss, ref,
           "C5 full size vs the CPU restatement")


@pytest.mark.parametrize("n", [1, 33, 1000, 20011])  # one point; a tile and a point; ragged; a tile for most waves
@pytest.mark.parametrize("dims", [
    [16, 32, 8], [48] + [32] * 5 + [16], [64] + [32] * 4 + [8],               # 32 wide, 1 to 5 hidden layers
    [16, 64, 16], [32] + [64] * 4 + [16], [48, 64, 64, 8], [64] + [64] * 4 + [8],  # 64 wide, 1 to 4; 1 to 4 input chunks
])
def test_narrow_chains(dims, n):
    """The chains one kernel trains (equal hidden widths of 32 or 64), at the edges of its tiles and input chunks,
    against the oracle at the step's bars: loss 1e-4, per layer 1e-2 of the gradient's norm."""
    g = torch.Generator().manual_seed(len(dims) * 100 + n)
    layers = []
    for i in range(len(dims) - 1):
        lim = (6.0 / dims[i]) ** 0.5
        layers.append((((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) * lim).half().float(),
                       torch.randn(dims[i + 1], generator=g) * 0.1))
    x = torch.randn(n, dims[0], generator=g).half()
    t = torch.randn(n, dims[-1], generator=g)
    loss, grads = rdv.mse_backward(_chain(layers), x.cuda(), t.cuda())
    ref_loss, ref_grads = T.mse_grads(x.float().numpy(), [(w.numpy(), b.numpy()) for w, b in layers], t.numpy())
    _check(loss.item(), grads, ref_loss, ref_grads, f"{dims} n={n}")


@pytest.mark.parametrize("inputs", [32, 48, 64])
def test_narrow_head_rows(inputs):
    """Every row of the head's gradient, 16 outputs behind four 64-wide layers (at 48 and 64 inputs the head's blocks
    do not fit the accumulation registers), at several tiles per wave: a row that lost a sixteenth of its points would
    be 25% off.  1e-2 of each row's norm, the step's bar."""
    dims, n = [inputs] + [64] * 4 + [16], 70011
    g = torch.Generator().manual_seed(inputs)
    layers = []
    for i in range(len(dims) - 1):
        lim = (6.0 / dims[i]) ** 0.5
        layers.append((((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) * lim).half().float(),
                       torch.randn(dims[i + 1], generator=g) * 0.1))
    x = torch.randn(n, inputs, generator=g).half()
    t = torch.randn(n, 16, generator=g)
    loss, grads = rdv.mse_backward(_chain(layers), x.cuda(), t.cuda())
    ref_loss, ref_grads = T.mse_grads(x.float().numpy(), [(w.numpy(), b.numpy()) for w, b in layers], t.numpy())
    _check(loss.item(), grads, ref_loss, ref_grads, f"{dims} n={n}")
    dw, ref = grads[-1][0].cpu().double().numpy(), ref_grads[-1][0]
    rows = np.linalg.norm(dw - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert (rows <= 1e-2).all(), f"head rows off by {np.round(rows, 4)}"


def _non_finite_reference(x, t, layers):
    """The step with the kernels' treatment of infinities and NaN: ReLU maps a NaN to 0, activations and gradients are
    rounded to fp16 (past 65504: infinite), a gradient is masked by selection; the products are IEEE's."""
    with np.errstate(all="ignore"):
        h = [x.astype(np.float64)]
        for i, (w, b) in enumerate(layers):
            z = (h[-1] @ w.astype(np.float64).T + b).astype(np.float32)
            if i + 1 < len(layers):
                h.append(np.fmax(z.astype(np.float16), np.float16(0)).astype(np.float64))
        g = (2 * (z - t)).astype(np.float16).astype(np.float64)
        grads = []
        for l in range(len(layers) - 1, -1, -1):
            grads.insert(0, (g.T @ h[l], g.sum(0)))
            if l:
                g = np.where(h[l] > 0, (g @ layers[l][0].astype(np.float64)).astype(np.float16).astype(np.float64), 0.0)
        return [(dw / t.size, db / t.size) for dw, db in grads]


@pytest.mark.parametrize("n", [70, 100])  # the last tile: 6 points; 4
@pytest.mark.parametrize("dims", [[16, 64, 8], [64, 32, 32, 8], [32, 64, 64, 16], [64] + [64] * 4 + [16]])
@pytest.mark.parametrize("where,value", [
    ("target", float("nan")), ("target", float("inf")), ("target", 1e5),  # 1e5: the gradient overflows fp16
    ("x", float("nan")), ("x", float("inf")), ("x", 60000.0),             # 60000: activations overflow
    ("last x", float("inf")), ("last x", 60000.0),                        # in the row that ends a partial tile
])
def test_narrow_chains_keep_non_finite_values_apart(dims, n, where, value):
    """One non-finite value reaches the gradient entries it has a part in and no others: the same entries are finite as
    in the reference, within 1e-2 of their norm."""
    g = torch.Generator().manual_seed(len(dims))
    layers = [(((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) * (6.0 / dims[i]) ** 0.5).half().float(),
               torch.randn(dims[i + 1], generator=g) * 0.1) for i in range(len(dims) - 1)]
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, dims[0], generator=g).half()
    t = torch.randn(n, dims[-1], generator=g)
    if where == "target":
        t[5, 3] = value
    else:
        x[7 if where == "x" else n - 1, 5] = value
    _, grads = rdv.mse_backward(_chain(layers), x.cuda(), t.cuda())
    ref = _non_finite_reference(x.numpy(), t.numpy(), [(w.numpy(), b.numpy()) for w, b in layers])
    for l, (got, want) in enumerate(zip(grads, ref)):
        for a, b, what in zip(got, want, ("dW", "db")):
            a = a.cpu().double().numpy()
            finite = np.isfinite(b)
            assert (np.isfinite(a) == finite).all(), f"layer {l} {what}: {(np.isfinite(a) != finite).sum()} entries"
            err = np.linalg.norm(a[finite] - b[finite])
            assert err <= 1e-2 * np.linalg.norm(b[finite]), f"layer {l} {what}: {err}"


@pytest.mark.parametrize("dims,n", [
    ([16, 32, 8], 140011), ([48] + [32] * 5 + [16], 140011), ([64] + [32] * 4 + [8], 200001),  # 2,048 waves: 2 to 4 tiles each
    ([16, 64, 16], 70001), ([48, 64, 64, 8], 70001), ([32] + [64] * 3 + [16], 140011), ([64] + [64] * 4 + [8], 70001),  # 1,024
])
def test_narrow_chains_over_several_tiles(dims, n):
    """The kernel's tile loop past its first turn: the prefetched inputs, the gradients, db and loss carried over tiles,
    ragged ends, against the oracle at the step's bars."""
    g = torch.Generator().manual_seed(n)
    layers = []
    for i in range(len(dims) - 1):
        lim = (6.0 / dims[i]) ** 0.5
        layers.append((((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) * lim).half().float(),
                       torch.randn(dims[i + 1], generator=g) * 0.1))
    x = torch.randn(n, dims[0], generator=g).half()
    t = torch.randn(n, dims[-1], generator=g)
    loss, grads = rdv.mse_backward(_chain(layers), x.cuda(), t.cuda())
    ref_loss, ref_grads = T.mse_grads(x.float().numpy(), [(w.numpy(), b.numpy()) for w, b in layers], t.numpy())
    _check(loss.item(), grads, ref_loss, ref_grads, f"{dims} n={n}")
