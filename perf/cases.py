"""The framework's work as a user's program has it done, for timing and comparing builds.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)`
one more of the same ranges; `prepare` makes what the program holds before the
call (inputs, networks, operators), `run` is one pass through the public entry
points, `work` the bytes and operations it cannot do without, `tolerance` what
another correct implementation may differ by and `exact` the result in 64 bits.

Kinds of case:
  map           m(x): a coordinate / feature network over rows of points
  conv_nchw     Winograd3x3Conv2d on NCHW fp16 images
  conv_winograd Conv2DTensorOpWinograd3x3 on a channels-last fp32 image
  conv_direct   Conv2DTensorOpFast / Conv2DTensorOp on a channels-last fp32 image
  linear        LinearTensorOp* on rows of features
  render        Cameras >> EmissionAbsorption
  profile       Cameras >> VolumeProfile
  train         mse_backward: loss and gradients of a network
"""
import math

import torch

import rdv_project_amd as rdv

# ------------------------------------------------------------------ cases


def _map(rows, features, octaves, hidden, depth, out, f16):
    """depth hidden layers of `hidden` units; octaves > 0: frequency-encoded input, padded to a multiple of 16."""
    return dict(kind="map", rows=rows, features=features, octaves=octaves, hidden=hidden, depth=depth, out=out, f16=f16)


def _nchw(batch, h, w, cin, cout):
    return dict(kind="conv_nchw", batch=batch, h=h, w=w, cin=cin, cout=cout)


def _wino(h, w, cin, cout):
    return dict(kind="conv_winograd", h=h, w=w, cin=cin, cout=cout)


def _direct(h, w, cin, cout, k, f16):
    return dict(kind="conv_direct", h=h, w=w, cin=cin, cout=cout, k=k, f16=f16)


def _linear(rows, features, out, f16):
    return dict(kind="linear", rows=rows, features=features, out=out, f16=f16)


def _render(width, height, samples, depth):
    return dict(kind="render", width=width, height=height, samples=samples, depth=depth)


def _profile(width, height, step, environment_samples):
    return dict(kind="profile", width=width, height=height, step=step, environment_samples=environment_samples)


def _train(rows, features, hidden, depth, out):
    return dict(kind="train", rows=rows, features=features, hidden=hidden, depth=depth, out=out)


def listed():
    def named(name, case):
        return dict(case, name=name)

    return [
        # a query of a small coordinate network at a handful of points (picking, a probe line), not a whole number of
        # 32-row groups: latency
        named("map_1k", _map(1000, 3, 0, 64, 4, 4, True)),
        # the headline network: a frequency-encoded field evaluated on a million points
        named("map_freq_1m", _map(1 << 20, 3, 6, 64, 3, 4, True)),
        # a wider network over precomputed features, whose shape has no kernel of its own
        named("map_wide_1m", _map(1 << 20, 64, 0, 128, 3, 16, True)),
        # the exact-fp32 form of a coordinate network (Linear layers), one 256 x 256 image of points
        named("map_f32_64k", _map(1 << 16, 3, 0, 64, 4, 4, False)),
        # one layer of an fp16 image network in PyTorch's layout
        named("conv_nchw_256", _nchw(1, 256, 256, 64, 64)),
        # the reference's own Winograd operator: channels-last fp32 image, 48 channels (its largest)
        named("conv_winograd_256", _wino(256, 256, 48, 48)),
        # a direct convolution layer of an image network, fp16 operands
        named("conv_direct_256", _direct(256, 256, 64, 64, 3, True)),
        # a wide per-layer network: one linear tensor operation
        named("linear_1024", _linear(65536, 1024, 1024, True)),
        # one frame of the volume renderer
        named("render_512", _render(512, 512, 128, 3)),
        # the features of a learned renderer, one frame: marches, a light ray and ratio-tracked environment rays
        named("profile_512", _profile(512, 512, 0.004, 4)),
        # a training step of a small field network on a batch of 2^18 points
        named("train_64w", _train(1 << 18, 32, 64, 4, 16)),
        # a training step of a deep network on four million points
        named("train_128w", _train(1 << 22, 32, 128, 8, 16)),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["map", "map", "map", "conv_nchw", "conv_winograd", "conv_direct", "linear", "linear", "render",
                       "profile", "train", "train"])
    if kind == "map":
        f16 = rng.random() < 0.75
        rows = _log(rng, 64, (1 << 20) if f16 else (1 << 18))
        if rng.random() < 0.6:  # coordinates
            octaves = rng.choice([0, 0, 6, 4]) if f16 else 0
            return _map(rows, 3, octaves, rng.choice([32, 64, 64, 64]), rng.randint(2, 4), rng.choice([1, 3, 4]), f16)
        return _map(rows, rng.choice([16, 32, 48, 64]), 0, rng.choice([32, 64, 96, 128] if f16 else [32, 48, 64]),
                    rng.randint(2, 4), rng.choice([1, 3, 4, 16]), f16)
    if kind == "conv_nchw":
        return _nchw(rng.choice([1, 1, 2, 4]), 2 * _log(rng, 32, 256), 2 * _log(rng, 32, 256),
                     rng.choice([16, 32, 48, 64]), rng.choice([16, 32, 64, 128]))
    if kind == "conv_winograd":
        return _wino(2 * _log(rng, 32, 256), 2 * _log(rng, 32, 256), rng.choice([16, 32, 48]),
                     rng.choice([16, 32, 48]))
    if kind == "conv_direct":
        f16 = rng.random() < 0.75
        return _direct(32 * rng.randint(2, 12), rng.randint(64, 400), rng.choice([16, 32, 48, 64]),
                       rng.choice([16, 32, 64, 128]), rng.choice([1, 3, 3, 5]), f16)
    if kind == "linear":
        f16 = rng.random() < 0.75
        features, out = 16 * _log(rng, 2, 64), 32 * _log(rng, 1, 32)
        if not f16:
            features, out = min(features, 512), min(out, 512)
        return _linear(64 * _log(rng, 8, 1024), features, out, f16)
    if kind == "render":
        return _render(_log(rng, 64, 512), _log(rng, 64, 512), rng.choice([32, 64, 96, 128]), rng.choice([3, 3, 2]))
    if kind == "profile":
        return _profile(_log(rng, 64, 400), _log(rng, 64, 400), rng.choice([0.004, 0.006, 0.01]), rng.randint(1, 4))
    return _train(_log(rng, 1 << 12, 1 << 19), rng.choice([16, 32, 48, 64]), rng.choice([32, 64, 64, 96, 128]),
                  rng.randint(2, 5), rng.choice([8, 16]))


# ------------------------------------------------------------------ inputs


class _Rng:
    """Device tensors drawn from one seed, in call order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def uniform(self, shape, lo, hi):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def normal(self, shape, std):
        return torch.randn(shape, generator=self.g, device="cuda") * std


def _enc_width(case):
    """(encoded width, width padded to a multiple of 16) of a map case."""
    w = case["features"] * (1 + 2 * case["octaves"])
    return w, (w if case["octaves"] == 0 else (w + 15) // 16 * 16)


def _layers(rng, dims, used=None):
    """(W [out, in], b [out]) fp32 per layer: He-uniform weights, PyTorch's default bias range.  used: how many of
    the first layer's inputs are not padding."""
    layers = []
    for i in range(len(dims) - 1):
        fan = used if i == 0 and used else dims[i]
        w = rng.uniform((dims[i + 1], dims[i]), -math.sqrt(6.0 / fan), math.sqrt(6.0 / fan))
        if i == 0:
            w[:, fan:] = 0.0
        layers.append((w, rng.uniform((dims[i + 1],), -1.0, 1.0) / math.sqrt(fan)))
    return layers


def _chain(layers, f16, head=None, encoding=None):
    m = encoding
    for i, (w, b) in enumerate(layers):
        lin = rdv.linear(w, b, f16=f16)
        m = lin if m is None else m >> lin
        if i + 1 < len(layers):
            m = m >> rdv.relu
    return m if head is None else m >> head


def _dims(case):
    first = _enc_width(case)[1] if case["kind"] == "map" else case["features"]
    return [first] + [case["hidden"]] * case["depth"] + [case["out"]]


def _pose(seed):
    """A camera 3.5 away from the box's centre, looking at it."""
    g = torch.Generator().manual_seed(seed)
    az, el = (torch.rand(2, generator=g) * torch.tensor([2 * math.pi, 2.0]) - torch.tensor([0.0, 1.0])).tolist()
    o = [3.5 * math.cos(el) * math.sin(az), 3.5 * math.sin(el), 3.5 * math.cos(el) * math.cos(az)]
    return torch.tensor([o + [0.0, 0.0, 0.0] + [0.0, 1.0, 0.0]])


def _data(case, seed):
    """The case's tensors, without anything of the framework."""
    rng, kind = _Rng(seed), case["kind"]
    if kind == "map":
        layers = _layers(rng, _dims(case), _enc_width(case)[0])
        return dict(x=rng.uniform((case["rows"], case["features"]), -1.0, 1.0), layers=layers)
    if kind == "conv_nchw":
        x = rng.uniform((case["batch"], case["cin"], case["h"], case["w"]), 0.0, 1.0).half()
        w = rng.normal((case["cout"], case["cin"], 3, 3), math.sqrt(2.0 / (9 * case["cin"]))).half()
        return dict(x=x, w=w, b=rng.uniform((case["cout"],), -0.1, 0.1))
    if kind in ("conv_winograd", "conv_direct"):
        k = case.get("k", 3)
        x = rng.uniform((case["h"] * case["w"], case["cin"]), -1.0, 1.0)
        w = rng.normal((k, k, case["cin"], case["cout"]), math.sqrt(2.0 / (k * k * case["cin"])))
        return dict(x=x, w=w, b=rng.uniform((case["cout"],), -0.1, 0.1))
    if kind == "linear":
        (w, b), = _layers(rng, [case["features"], case["out"]])
        return dict(x=rng.normal((case["rows"], case["features"]), 1.0), w=w, b=b)
    if kind == "render":
        return dict(layers=_layers(rng, [3] + [64] * case["depth"] + [4]), pose=_pose(seed))
    if kind == "profile":
        return dict(layers=_layers(rng, [3, 64, 64, 64, 1]), pose=_pose(seed))
    layers = _layers(rng, _dims(case))
    x = rng.normal((case["rows"], case["features"]), 1.0).half()
    return dict(x=x, target=rng.normal((case["rows"], case["out"]), 1.0), layers=layers)


def _lattice(n):
    """Voxel centres of an n^3 grid over [-1, 1]^3, x fastest."""
    c = (torch.arange(n, dtype=torch.float32, device="cuda") + 0.5) / n * 2 - 1
    zz, yy, xx = torch.meshgrid(c, c, c, indexing="ij")
    return torch.stack([xx, yy, zz], -1).reshape(-1, 3).contiguous()


def prepare(case, seed):
    rdv.set_synchronous(False)  # launches ordered on torch's stream
    d, kind = _data(case, seed), case["kind"]
    if kind == "map":
        enc = None
        if case["octaves"]:
            enc = rdv.FrequencyEncoding(case["features"], case["octaves"], pad_to=_enc_width(case)[1])
        return dict(kind=kind, m=_chain(d["layers"], case["f16"], encoding=enc), x=d["x"])
    if kind == "conv_nchw":
        return dict(kind=kind, conv=rdv.Winograd3x3Conv2d(d["w"], d["b"]), x=d["x"],
                    out=torch.empty((case["batch"], case["cout"], case["h"], case["w"]), dtype=torch.float16,
                                    device="cuda"))
    if kind == "conv_winograd":
        return dict(kind="op", op=rdv.Conv2DTensorOpWinograd3x3(d["x"], d["w"], d["b"], case["h"], case["w"]))
    if kind == "conv_direct":
        cls = rdv.Conv2DTensorOpFast if case["f16"] else rdv.Conv2DTensorOp
        return dict(kind="op", op=cls(d["x"], d["w"], d["b"], case["h"], case["w"]))
    if kind == "linear":
        cls = rdv.LinearTensorOpFast if case["f16"] else rdv.LinearTensorOp
        return dict(kind="op", op=cls(d["x"], d["w"], d["b"]))
    if kind == "render":
        cams = rdv.Cameras(case["width"], case["height"], d["pose"].cuda())
        return dict(kind=kind, sensor=cams >> rdv.EmissionAbsorption(_chain(d["layers"], True),
                                                                    samples=case["samples"]))
    if kind == "profile":
        ext = _chain(d["layers"], True, head=rdv.softplus)
        dens = ext(rdv.wrap(_lattice(64))).as_tensor("torch").reshape(64, 64, 64, 1) * 1.3 + 1e-3
        majorant = rdv.MajorantGrid(rdv.TensorGrid(dens), [8, 8, 8])
        vp = rdv.VolumeProfile(ext, majorant, rdv.Constant([1.0, 0.9, 0.8]), rdv.Constant([0.6, 0.7, 0.8]),
                               [0.9, 0.5, 0.1], density_scale=4.0, g=0.3, step_size=case["step"],
                               environment_samples=case["environment_samples"])
        cams = rdv.Cameras(case["width"], case["height"], d["pose"].cuda())
        return dict(kind=kind, sensor=cams >> vp, seed=seed)
    grads = [(torch.empty_like(w), torch.empty_like(b)) for w, b in d["layers"]]
    return dict(kind=kind, m=_chain(d["layers"], True), x=d["x"], target=d["target"], grads=grads,
                loss=torch.empty((), device="cuda"))


def run(state):
    kind = state["kind"]
    if kind == "map":
        return state["m"](state["x"]).as_tensor("torch")
    if kind == "conv_nchw":
        return state["conv"](state["x"], relu=True, out=state["out"])
    if kind == "op":
        state["op"].evaluate()
        return state["op"].as_type("torch")
    if kind == "render":
        return state["sensor"]().as_tensor("torch")
    if kind == "profile":
        rdv.RandomLibrary.seed(state["seed"])  # a reproducible frame
        return state["sensor"]().as_tensor("torch")
    loss, grads = rdv.mse_backward(state["m"], state["x"], state["target"], grads=state["grads"], loss=state["loss"])
    return {"loss": loss, "grads": [list(g) for g in grads]}


# ------------------------------------------------------------------ work


def _macs(dims):
    return sum(a * b for a, b in zip(dims, dims[1:]))


def work(case):
    kind = case["kind"]
    if kind == "map":
        dims = _dims(case)
        return {"bytes": 4 * (case["rows"] * (case["features"] + case["out"]) + _macs(dims)),
                "flops": 2 * case["rows"] * _macs(dims)}
    if kind == "conv_nchw":
        px = case["batch"] * case["h"] * case["w"]
        return {"bytes": 2 * px * (case["cin"] + case["cout"]) + 2 * 16 * case["cin"] * case["cout"],
                "flops": 2 * 4 * px * case["cin"] * case["cout"]}  # F(2x2, 3x3): 16 products per 2 x 2 outputs
    if kind == "conv_winograd":
        px = case["h"] * case["w"]
        return {"bytes": 4 * px * (case["cin"] + case["cout"]) + 2 * 16 * case["cin"] * case["cout"],
                "flops": 2 * 4 * px * case["cin"] * case["cout"]}
    if kind == "conv_direct":
        px, taps = case["h"] * case["w"], case["k"] ** 2
        return {"bytes": 4 * px * (case["cin"] + case["cout"]) + 4 * taps * case["cin"] * case["cout"],
                "flops": 2 * taps * px * case["cin"] * case["cout"]}
    if kind == "linear":
        return {"bytes": 4 * case["rows"] * (case["features"] + case["out"]) + 2 * case["features"] * case["out"],
                "flops": 2 * case["rows"] * case["features"] * case["out"]}
    if kind == "render":
        rays = case["width"] * case["height"]
        dims = [3] + [64] * case["depth"] + [4]
        # about nine rays of ten meet the box
        return {"bytes": 12 * rays, "flops": int(0.9 * rays) * case["samples"] * 2 * _macs(dims)}
    if kind == "profile":
        rays = case["width"] * case["height"]
        # nine rays of ten meet the box, on a chord of about 2.2: the tau march once, and half of it for the light ray
        steps = 1.5 * 2.2 / case["step"]
        return {"bytes": 4 * rays * 16, "flops": int(0.9 * rays * steps * 2 * _macs([3, 64, 64, 64, 1]))}
    dims, n = _dims(case), case["rows"]
    forward, first = _macs(dims), dims[0] * dims[1]
    return {"bytes": n * (2 * case["features"] + 4 * case["out"]) + 4 * 2 * forward,
            "flops": 2 * n * (3 * forward - first)}


def tolerance(case):
    """About four times what a reordering of the sums changes (the same network with its hidden units permuted), or,
    for the convolutions, the flips of an fp16 rounding that a reordering can cause."""
    kind = case["kind"]
    if kind == "map":  # a flipped fp16 rounding of a hidden value travels to the output; fp32 sums only reorder
        return {"rel": 2e-4, "max": 0.01} if case["f16"] else {"rel": 2e-6, "max": 1e-5}
    if kind == "conv_nchw":  # fp16 outputs
        return {"rel": 5e-4, "max": 4e-3}
    if kind == "conv_winograd":  # fp16 transformed inputs
        return {"rel": 2e-4, "max": 2e-3}
    if kind in ("conv_direct", "linear"):  # fp32 sums of fixed products
        return {"rel": 4e-6, "max": 5e-5}
    if kind == "render":
        return {"rel": 1e-5, "max": 2e-4}
    if kind == "profile":  # a depth moves by a step, a tracked ray draws other numbers: few rays, by their whole value
        return {"rel": 0.03, "max": 0.99}
    return {"rel": 5e-4, "max": 4e-3}


# ------------------------------------------------------------------ 64 bits


def _forward64(x, layers):
    for i, (w, b) in enumerate(layers):
        x = torch.addmm(b.double(), x, w.double().t())
        if i + 1 < len(layers):
            x = x.clamp_min(0.0)
    return x


def _encode64(x, octaves, width):
    parts = [x]
    for k in range(octaves):
        parts += [torch.sin(2.0 ** k * math.pi * x), torch.cos(2.0 ** k * math.pi * x)]
    y = torch.cat(parts, 1)
    return torch.nn.functional.pad(y, (0, width - y.shape[1]))


def _conv64(x, w, b, h, wd):
    """'same' convolution of x [h * wd, cin] with w [k, k, cin, cout], tap by tap."""
    k, cin = w.shape[0], w.shape[2]
    p = torch.nn.functional.pad(x.double().reshape(h, wd, cin), (0, 0, k // 2, k - 1 - k // 2, k // 2, k - 1 - k // 2))
    y = b.double().expand(h * wd, -1).clone()
    for i in range(k):
        for j in range(k):
            y += p[i:i + h, j:j + wd].reshape(h * wd, cin) @ w[i, j].double()
    return y


def _camera_rays64(pose, width, height):
    """Pinhole rays through the pixel centres: vertical field of view pi / 4, the image's own aspect ratio."""
    p = pose.double().cuda()[0]
    o, t, up = p[0:3], p[3:6], p[6:9]

    def unit(v):
        return v / v.norm(dim=-1, keepdim=True)

    z = unit(t - o)
    xa = unit(torch.linalg.cross(up, z))
    ya = torch.linalg.cross(z, xa)
    sx = ((torch.arange(width, device="cuda", dtype=torch.float64) + 0.5) / width * 2 - 1) * (width / height)
    sy = (torch.arange(height, device="cuda", dtype=torch.float64) + 0.5) / height * 2 - 1
    w = xa * sx[None, :, None] + ya * sy[:, None, None] + z * (1.0 / math.tan(math.pi / 8))
    return o, unit(w).reshape(-1, 3)


def _render64(d, case):
    o, w = _camera_rays64(d["pose"], case["width"], case["height"])
    out, s = torch.zeros((w.shape[0], 3), dtype=torch.float64, device="cuda"), case["samples"]
    for i in range(0, w.shape[0], 8192):
        v = w[i:i + 8192]
        inv = 1.0 / v
        t0 = (-o * inv - inv.abs()).amax(1).clamp_min(0.0)
        t1 = (-o * inv + inv.abs()).amin(1)
        dt = ((t1 - t0).clamp_min(0.0) / s)[:, None]
        t = t0[:, None] + (torch.arange(s, device="cuda", dtype=torch.float64) + 0.5) * dt
        f = _forward64((o + t[..., None] * v[:, None, :]).reshape(-1, 3), d["layers"]).reshape(-1, s, 4)
        tau = torch.nn.functional.softplus(f[..., 0], threshold=200.0) * dt
        weight = torch.exp(-(tau.cumsum(1) - tau)) * -torch.expm1(-tau)
        out[i:i + 8192] = (weight[..., None] * torch.sigmoid(f[..., 1:])).sum(1)
    return out.reshape(1, case["height"], case["width"], 3)


def _train64(d):
    layers, n = d["layers"], d["x"].shape[0]
    count = n * d["target"].shape[1]
    loss, grads = 0.0, [[torch.zeros(t.shape, dtype=torch.float64, device="cuda") for t in wb] for wb in layers]
    for i in range(0, n, 1 << 17):
        h = [d["x"][i:i + (1 << 17)].double()]
        for k, (w, b) in enumerate(layers):
            y = torch.addmm(b.double(), h[-1], w.double().t())
            h.append(y.clamp_min(0.0) if k + 1 < len(layers) else y)
        e = h[-1] - d["target"][i:i + (1 << 17)].double()
        loss = loss + e.square().sum() / count
        g = e * (2.0 / count)
        for k in reversed(range(len(layers))):
            grads[k][0] += g.t() @ h[k]
            grads[k][1] += g.sum(0)
            if k:
                g = (g @ layers[k][0].double()) * (h[k] > 0)
    return {"loss": loss, "grads": grads}


def exact(case, seed):
    kind = case["kind"]
    if kind == "profile":
        return None  # random draws and a state machine per ray: no closed form
    d = _data(case, seed)
    if kind == "map":
        out = []
        for x in d["x"].double().split(1 << 17):
            if case["octaves"]:
                x = _encode64(x, case["octaves"], _enc_width(case)[1])
            out.append(_forward64(x, d["layers"]))
        return torch.cat(out)
    if kind == "conv_nchw":
        w, h, wd = d["w"].permute(2, 3, 1, 0).contiguous(), case["h"], case["w"]
        out = [_conv64(x.permute(1, 2, 0).reshape(h * wd, -1), w, d["b"], h, wd).t().reshape(-1, h, wd) for x in d["x"]]
        return torch.stack(out).clamp_min(0.0)
    if kind in ("conv_winograd", "conv_direct"):
        return _conv64(d["x"], d["w"], d["b"], case["h"], case["w"])
    if kind == "linear":
        return torch.addmm(d["b"].double(), d["x"].double(), d["w"].double().t())
    if kind == "render":
        return _render64(d, case)
    return _train64(d)
