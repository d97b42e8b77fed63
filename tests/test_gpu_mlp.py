"""GPU parity of the fused MLP path against oracle/mlp.py (through the rdv API,
which calls the C ABI).  Bar: |y - ref| <= 2e-3 + 1e-2 |ref| for fp16 layers;
fp32 chains and the fp32 tail group: rtol 1e-5, atol 1e-6."""
import glob
import os

import numpy as np
import pytest
import torch

import rdv_project_amd as rdv
from oracle import mlp as O
from rdv_project_amd import workloads as WL

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def _chain(layers, acts, f16=True, enc=None):
    m = enc
    for (w, b), a in zip(layers, acts):
        lin = rdv.linear(w.cuda(), b.cuda(), f16=f16) if not isinstance(f16, list) else \
            rdv.linear(w.cuda(), b.cuda(), f16=f16.pop(0))
        m = lin if m is None else m >> lin
        if a == "relu":
            m = m >> rdv.relu
        elif a == "density_rgb":
            m = m >> rdv.density_rgb
        elif a == "softplus":
            m = m >> rdv.softplus
        elif a == "sigmoid":
            m = m >> rdv.sigmoid
        else:
            assert a == "none", a
    return m


def _np_layers(layers):
    return [(w.numpy(), b.numpy()) for w, b in layers]


def _assert_fp16_parity(y, ref, what):
    ok = O.within_tolerance(y, ref)
    if not ok.all():
        idx = np.argwhere(~ok)[:5]
        err = np.abs(y.astype(np.float64) - ref)
        raise AssertionError(f"{what}: {int((~ok).sum())} of {ok.size} outside |d| <= 2e-3 + 1e-2|ref|; "
                             f"first {idx.tolist()}, max abs err {err.max():.3g}")


def test_c1_full_config_matches_oracle():
    x, layers = WL.c1()
    acts = ["relu"] * 4 + ["none"]
    m = _chain(layers, acts)
    y = m(rdv.wrap(x.cuda())).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16"] * 5)
    assert y.shape == (65536, 4)
    _assert_fp16_parity(y, ref, "C1")


def test_c1_after_a_kernel_that_leaves_infinities_in_lds():
    """Regression: the one-launch kernel that builds its fragments from the
    layers' fp32 buffers once read layer 0's unused K slots (features 3..15 of
    a 3-wide input) from LDS it had not written.  Where an earlier kernel left
    values beyond fp16 range there, 0 * Inf = NaN and ReLU turned every point's
    output into 0.  A 3x3 conv whose operands are all 1e5 (fp16 infinity)
    first runs on every CU; the chain must still match the oracle."""
    H = W = 256
    C = K = 64
    op = rdv.Conv2DTensorOpSimple3x3(torch.full((H * W, C), 1e5).cuda(), torch.full((3, 3, C, K), 1e5).cuda(),
                                     torch.zeros(K).cuda(), H, W)
    op.evaluate()
    torch.cuda.synchronize()
    x, layers = WL.c1()
    acts = ["relu"] * 4 + ["none"]
    y = _chain(layers, acts)(rdv.wrap(x.cuda())).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16"] * 5)
    _assert_fp16_parity(y, ref, "C1 after the conv")


def test_c2_full_config_matches_oracle():
    x, layers = WL.c2()
    acts = ["relu"] * 3 + ["none"]
    enc = rdv.FrequencyEncoding(3, WL.C2_OCTAVES, pad_to=WL.C2_PAD)
    m = _chain(layers, acts, enc=enc)
    y = m(rdv.wrap(x.cuda())).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16"] * 4, encoding=(WL.C2_OCTAVES, WL.C2_PAD))
    assert y.shape == (1 << 20, 4)
    _assert_fp16_parity(y, ref, "C2")


def test_c4_mlp_density_rgb_head():
    layers = WL.c4_mlp()
    g = WL.gen(21)
    x = torch.rand(50000, 3, generator=g) * 2 - 1
    acts = ["relu"] * 3 + ["density_rgb"]
    y = _chain(layers, acts)(x.cuda()).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16"] * 4)
    _assert_fp16_parity(y, ref, "C4 mlp")


@pytest.mark.parametrize("cfg", ["c1", "c2", "c4"])
def test_fused_kernels_with_nonzero_bias(cfg):
    """The benchmark configurations have zero biases (the packer then selects the
    bias-free path); this runs the same fused kernels with biases seeded."""
    g = WL.gen(31)
    if cfg == "c2":
        x, layers = WL.c2(20000)
        enc = rdv.FrequencyEncoding(3, WL.C2_OCTAVES, pad_to=WL.C2_PAD)
        acts, encoding = ["relu"] * 3 + ["none"], (WL.C2_OCTAVES, WL.C2_PAD)
    elif cfg == "c1":
        x, layers = WL.c1(20000)
        enc, acts, encoding = None, ["relu"] * 4 + ["none"], None
    else:
        x = torch.rand(20000, 3, generator=g) * 2 - 1
        layers = WL.c4_mlp()
        enc, acts, encoding = None, ["relu"] * 3 + ["density_rgb"], None
    layers = [(w, torch.rand(w.shape[0], generator=g) * 0.5 - 0.25) for w, _ in layers]
    y = _chain(layers, acts, enc=enc)(x.cuda()).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16"] * len(layers), encoding=encoding)
    _assert_fp16_parity(y, ref, f"{cfg} with bias")


@pytest.mark.parametrize("n", [1, 17, 31, 32, 33, 65, 4096 + 19])
def test_row_counts_and_fp32_tail(n):
    x, layers = WL.c1(n)
    acts = ["relu"] * 4 + ["none"]
    y = _chain(layers, acts)(x.cuda()).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16"] * 5)
    _assert_fp16_parity(y, ref, f"n={n}")
    n_full = (n // 32) * 32
    if n > n_full:  # the partial group follows the fp32 rule, so it matches far tighter
        np.testing.assert_allclose(y[n_full:], ref[n_full:], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(GOLDEN, "chain_*.npz"))))
def test_golden_vectors(path):
    z = np.load(path, allow_pickle=False)
    dims = list(z["dims"])
    layers = [(torch.from_numpy(z[f"W{i}"]), torch.from_numpy(z[f"b{i}"])) for i in range(len(dims) - 1)]
    acts = [str(a) for a in z["acts"]]
    precs = [str(p) for p in z["precs"]]
    m = _chain(layers, acts, f16=[p == "f16" for p in precs])
    y = m(torch.from_numpy(z["x"]).cuda()).as_tensor("torch").cpu().numpy()
    if all(p == "f32" for p in precs):
        np.testing.assert_allclose(y, z["y"], rtol=1e-5, atol=1e-6)
    else:
        _assert_fp16_parity(y, z["y"], os.path.basename(path))


@pytest.mark.parametrize("dims,f16,n,kernel", [
    ([5, 37, 19, 7], True, 1000, "mlp_generic_f16<2,lds>"),          # odd widths, partial tiles and chunks
    ([3, 64, 64, 4], False, 1000, "mlp_chain_f32_reg_kernel"),        # exact fp32 Linear chain
    ([64, 128, 128, 16], True, 1000, "mlp_generic_f16<4,lds>"),
    ([64, 128, 128, 16], True, 40_000, "mlp_generic_f16<4,lds>"),     # several tiles per wave
    ([17, 96, 200, 33], True, 777, "mlp_generic_f16<8,lds>"),         # 3, 7 and 2 M tiles
    ([3, 256, 256, 4], True, 3000, "mlp_generic_f16<8,global>"),      # fragments beyond the LDS cap
    ([256, 32, 1], True, 500, "mlp_generic_f16<1,lds>"),              # 16 K chunks in layer 0
    ([8] + [32] * 15 + [2], True, 2048, "mlp_generic_f16<1,lds>"),    # 16 layers
    # raw 16-byte rows of at most 64 features: layer 0's input is loaded a tile ahead
    ([36, 96, 48, 8], True, 1000, "mlp_generic_f16<4,lds>"),          # 3 K chunks, pieces past D are zeros
    ([12, 40, 3], True, 4115, "mlp_generic_f16<2,lds>"),              # 1 K chunk, partial last tile
    ([20, 64, 64, 4], True, 33, "mlp_generic_f16<2,lds>"),            # fewer tiles than waves
])
def test_generic_chains(dims, f16, n, kernel):
    g = WL.gen(5)
    layers = [((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) / dims[i] ** 0.5 * 1.7,
               torch.rand(dims[i + 1], generator=g) * 0.2 - 0.1) for i in range(len(dims) - 1)]
    acts = ["relu"] * (len(dims) - 2) + ["none"]
    x = torch.rand(n, dims[0], generator=g) * 2 - 1
    m = _chain(layers, acts, f16=f16)
    y = m(x.cuda()).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16" if f16 else "f32"] * len(layers))
    if f16:
        _assert_fp16_parity(y, ref, str(dims))
        assert np.abs(ref).max() > 0.05  # the chain did not collapse to ~0
    else:
        np.testing.assert_allclose(y, ref, rtol=1e-5, atol=1e-6)
    from rdv_project_amd import _chain as CH, _lib
    p = CH.plan_chain(m, dims[0])
    assert _lib.load().rdv_mlp_kernel_name(p.desc).decode() == kernel


@pytest.mark.parametrize("dims,precs,enc", [
    ([3, 64, 64, 64, 64, 4], ["f32"] * 5, None),                   # C1's network, exact fp32 Linear layers
    ([5, 37, 19, 7], ["f32"] * 3, None),                            # odd widths: a tail quartet in every layer
    ([3, 48, 64, 4], ["f32", "f16", "f32"], None),                  # a LinearFast layer between Linear ones
    ([39, 64, 64, 4], ["f32"] * 3, 6),                              # FREQ(6) encoding of 3 inputs
])
def test_f32_chain_register_kernel_equals_row_kernel(dims, precs, enc):
    """Chains that are not all LinearFast run on the vector ALUs in the
    reference's per-output order: 256 rows or more on the register kernel,
    fewer on the one-thread-per-row kernel.  Rows 0..95 of a 5,000-row call
    must equal, bit for bit, the same rows evaluated alone (three whole groups
    of 32, so the same LinearFast rule), and the oracle."""
    g = WL.gen(41)
    d_in = 3 if enc else dims[0]
    layers = [((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) / dims[i] ** 0.5 * 1.7,
               torch.rand(dims[i + 1], generator=g) * 0.2 - 0.1) for i in range(len(dims) - 1)]
    acts = ["relu"] * (len(dims) - 2) + ["none"]
    x = torch.rand(5000, d_in, generator=g) * 2 - 1
    encoder = rdv.FrequencyEncoding(3, enc) if enc else None
    m = _chain(layers, acts, f16=[p == "f16" for p in precs], enc=encoder)
    y = m(x.cuda()).as_tensor("torch").cpu().numpy().copy()
    y_small = m(x[:96].contiguous().cuda()).as_tensor("torch").cpu().numpy()
    assert np.array_equal(y[:96], y_small)
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, precs, encoding=(enc, None) if enc else None)
    if all(p == "f32" for p in precs):
        # the encoding's fp32 sinpi / cospi against the oracle's float64 sin / cos rounded to fp32
        tol = dict(rtol=1e-4, atol=1e-5) if enc else dict(rtol=1e-5, atol=1e-6)
        np.testing.assert_allclose(y, ref, **tol)
    else:
        _assert_fp16_parity(y, ref, str(dims))
    from rdv_project_amd import _chain as CH, _lib
    assert _lib.load().rdv_mlp_kernel_name(CH.plan_chain(m, d_in).desc).decode() == "mlp_chain_f32_reg_kernel"


@pytest.mark.parametrize("n", [1, 15, 17, 31, 144, 9000])  # 16-row tiles: one, part of one, more than a wave takes
@pytest.mark.parametrize("dims,precs", [
    ([1, 1], ["f32"]), ([4, 16, 16], ["f32"] * 2), ([15, 17, 5], ["f32"] * 2),   # tile edges
    ([64, 64, 64, 1], ["f32"] * 3), ([33, 63, 49, 16], ["f32", "f16", "f32"]),    # straight-line and branching layers
    ([3] + [64] * 11 + [2], ["f32"] * 12),                                        # parameters past the LDS: read from rows
    ([65, 128, 250, 256, 3], ["f32"] * 4),                                        # the wide kernel, some layers from rows
])
def test_f32_chain_edges(dims, precs, n):
    """Exact-fp32 chains at the edges of their 16-wide tiles, against float64:
    layer by layer each output is an fp32 FMA chain over k inputs, off by at
    most gamma(k + 2) of the sum of its magnitudes; the bound is carried through
    the layers (ReLU does not grow it).  LinearFast layers round their inputs
    and weights to fp16 (2^-11 relative each) first."""
    g = WL.gen(57)
    layers = [((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) / dims[i] ** 0.5 * 1.7,
               torch.rand(dims[i + 1], generator=g) * 0.2 - 0.1) for i in range(len(dims) - 1)]
    acts = ["relu"] * (len(dims) - 2) + ["none"]
    x = torch.rand(n, dims[0], generator=g) * 2 - 1
    y = _chain(layers, acts, f16=[p == "f16" for p in precs])(x.cuda()).as_tensor("torch").cpu().double()
    u, v, e = 2.0 ** -24, x.double(), torch.zeros(n, dims[0], dtype=torch.float64)
    for i, (w, b) in enumerate(layers):
        w, k = w.double(), dims[i] + 2
        r = k * u / (1 - k * u) + (2.01 * 2.0 ** -11 if precs[i] == "f16" else 0.0)
        e = e @ w.abs().t() * (1 + r) + r * (v.abs() @ w.abs().t() + b.double().abs())
        v = v @ w.t() + b.double()
        if acts[i] == "relu":
            v = v.clamp_min(0.0)
    assert bool(((y - v).abs() <= e).all()), float(((y - v).abs() / e).max())


@pytest.mark.parametrize("acts", [
    ["softplus", "relu", "none"],       # a transcendental hidden activation
    ["relu", "none", "sigmoid"],        # a linear hidden layer, sigmoid head
    ["relu", "relu", "density_rgb"],
])
def test_generic_hidden_and_head_activations(acts):
    g = WL.gen(9)
    dims = [6, 48, 40, 4]
    layers = [((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) / dims[i] ** 0.5 * 1.7,
               torch.rand(dims[i + 1], generator=g) * 0.2 - 0.1) for i in range(3)]
    x = torch.rand(2048, dims[0], generator=g) * 2 - 1
    y = _chain(layers, acts)(x.cuda()).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16"] * 3)
    _assert_fp16_parity(y, ref, "-".join(acts))


def test_generic_unaligned_rows_take_scalar_loads():
    """x viewed 4 bytes past a 16-byte boundary: layer 0 reads its row with
    scalar loads instead of 16-byte ones; the result is the same."""
    g = WL.gen(10)
    dims = [16, 64, 8]
    layers = [((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) / dims[i] ** 0.5,
               torch.zeros(dims[i + 1])) for i in range(2)]
    acts = ["relu", "none"]
    base = torch.empty(512 * 16 + 1, device="cuda")
    x = base[1:].view(512, 16)
    x.copy_((torch.rand(512, 16, generator=g) * 2 - 1).cuda())
    assert x.data_ptr() % 16 == 4
    m = _chain(layers, acts)
    y = m(rdv.wrap(x)).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.cpu().numpy(), _np_layers(layers), acts, ["f16"] * 2)
    _assert_fp16_parity(y, ref, "unaligned x")


def test_freq_encoding_odd_octaves_generic_path():
    g = WL.gen(8)
    x = torch.rand(777, 2, generator=g) * 2 - 1
    enc = rdv.FrequencyEncoding(2, 5)  # 22 features, no padding, not instantiated
    layers = [((torch.rand(32, 22, generator=g) * 2 - 1) * 0.4, torch.zeros(32)),
              ((torch.rand(3, 32, generator=g) * 2 - 1) * 0.3, torch.zeros(3))]
    acts = ["relu", "none"]
    y = _chain(layers, acts, enc=enc)(x.cuda()).as_tensor("torch").cpu().numpy()
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), acts, ["f16", "f16"], encoding=(5, 22))
    _assert_fp16_parity(y, ref, "freq(2,5)")


def test_f16_all_entry_matches_on_full_groups():
    """rdv_mlp_forward_f16_all runs the tail on the matrix cores too; full groups are identical."""
    import ctypes as C
    from rdv_project_amd import _chain as CH, _lib
    x, layers = WL.c1(1000)
    m = _chain(layers, ["relu"] * 4 + ["none"])
    xd = x.cuda()
    y_ref = m(xd).as_tensor("torch").clone()
    p = CH.plan_chain(m, 3)
    packed = CH.packed_params(m, p)
    y2 = torch.empty_like(y_ref)
    _lib.check(_lib.load().rdv_mlp_forward_f16_all(C.byref(p.desc), C.c_void_p(packed.data_ptr()),
                                                   C.c_void_p(xd.data_ptr()), C.c_void_p(y2.data_ptr()),
                                                   C.c_int64(1000), None))
    torch.cuda.synchronize()
    assert torch.equal(y2[:992], y_ref[:992])
    ref = O.mlp_forward(x.numpy(), _np_layers(layers), ["relu"] * 4 + ["none"], ["f16"] * 5)
    full = O.chain(x.numpy()[992:], _np_layers(layers), ["relu"] * 4 + ["none"], ["f16"] * 5, True)
    _assert_fp16_parity(y2[992:].cpu().numpy(), full, "f16 tail")
    assert ref.shape == (1000, 4)


def test_generic_prefetched_and_scalar_inputs_agree_bitwise():
    """A runtime-shaped chain over 16-byte aligned rows (layer 0's input loaded a
    tile ahead in registers) and over the same rows 4 bytes off (loaded chunk by
    chunk, element by element): the same values, bit for bit."""
    import ctypes as C
    from rdv_project_amd import _chain as CH, _lib
    g = WL.gen(17)
    dims = [36, 96, 48, 8]
    layers = [((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) / dims[i] ** 0.5 * 1.7,
               torch.rand(dims[i + 1], generator=g) * 0.2 - 0.1) for i in range(3)]
    m = _chain(layers, ["relu", "relu", "none"])
    n = 2050
    x = (torch.rand(n, dims[0], generator=g) * 2 - 1).cuda()
    shifted = torch.empty(n * dims[0] + 4, device="cuda")
    shifted[1:1 + n * dims[0]].copy_(x.reshape(-1))
    assert shifted.data_ptr() % 16 == 0 and x.data_ptr() % 16 == 0
    p = CH.plan_chain(m, dims[0])
    assert _lib.load().rdv_mlp_kernel_name(p.desc).decode() == "mlp_generic_f16<4,lds>"
    packed = CH.packed_params(m, p)
    ya = torch.empty(n, dims[-1], device="cuda")
    yb = torch.empty_like(ya)
    lib = _lib.load()
    _lib.check(lib.rdv_mlp_forward_f16_all(C.byref(p.desc), C.c_void_p(packed.data_ptr()), C.c_void_p(x.data_ptr()),
                                           C.c_void_p(ya.data_ptr()), C.c_int64(n), None))
    _lib.check(lib.rdv_mlp_forward_f16_all(C.byref(p.desc), C.c_void_p(packed.data_ptr()),
                                           C.c_void_p(shifted.data_ptr() + 4), C.c_void_p(yb.data_ptr()),
                                           C.c_int64(n), None))
    torch.cuda.synchronize()
    assert torch.equal(ya, yb)
    ref = O.mlp_forward(x.cpu().numpy(), _np_layers(layers), ["relu", "relu", "none"], ["f16"] * 3)
    _assert_fp16_parity(ya[:2048].cpu().numpy(), ref[:2048], "prefetched input")


@pytest.mark.parametrize("case", ["c1", "c2", "c1_bias", "generic"])
@pytest.mark.parametrize("n", [4096, 1000, 31])
def test_unpacked_entry_matches_packed_path(case, n):
    """rdv_mlp_forward_unpacked (the layers' own fp32 buffers, converted inside
    the compile-time kernel, or packed into a workspace for other chains) gives
    the bits of rdv_mlp_pack + rdv_mlp_forward, tail rows included."""
    import ctypes as C
    from rdv_project_amd import _chain as CH, _lib
    enc = None
    if case.startswith("c1"):
        x, layers = WL.c1(n)
        acts = ["relu"] * 4 + ["none"]
        if case == "c1_bias":
            layers = [(w, torch.rand(w.shape[0], generator=WL.gen(i)) * 0.2 - 0.1) for i, (w, _) in enumerate(layers)]
    elif case == "c2":
        x, layers = WL.c2(n)
        acts = ["relu"] * 3 + ["none"]
        enc = rdv.FrequencyEncoding(3, WL.C2_OCTAVES, pad_to=WL.C2_PAD)
    else:
        g = WL.gen(23)
        dims = [20, 96, 40, 6]
        x = torch.rand(n, 20, generator=g) * 2 - 1
        layers = [((torch.rand(dims[i + 1], dims[i], generator=g) * 2 - 1) / dims[i] ** 0.5,
                   torch.rand(dims[i + 1], generator=g) * 0.2 - 0.1) for i in range(3)]
        acts = ["relu", "relu", "none"]
    m = _chain(layers, acts, enc=enc)
    xd = x.cuda()
    lib = _lib.load()
    p = CH.plan_chain(m, int(x.shape[1]))
    packed = CH.packed_params(m, p)
    ya = torch.empty(n, p.out_features, device="cuda")
    _lib.check(lib.rdv_mlp_forward(C.byref(p.desc), C.c_void_p(packed.data_ptr()), C.c_void_p(xd.data_ptr()),
                                   C.c_void_p(ya.data_ptr()), C.c_int64(n), None))
    nb = int(lib.rdv_mlp_unpacked_workspace_bytes(C.byref(p.desc)))
    assert (nb == 0) == (case != "generic")
    _, ws, bs = CH._param_arrays(p)
    yb = torch.full_like(ya, float("nan"))
    if nb:
        raw = torch.empty(nb + 256, dtype=torch.uint8, device="cuda")
        wsp = raw.data_ptr() + (-raw.data_ptr()) % 256
        assert lib.rdv_mlp_forward_unpacked(C.byref(p.desc), ws, bs, C.c_void_p(xd.data_ptr()),
                                            C.c_void_p(yb.data_ptr()), C.c_int64(n), C.c_void_p(wsp),
                                            C.c_int64(nb - 256), None) == _lib.RDV_ERR_WORKSPACE
    else:
        wsp = None
    _lib.check(lib.rdv_mlp_forward_unpacked(C.byref(p.desc), ws, bs, C.c_void_p(xd.data_ptr()),
                                            C.c_void_p(yb.data_ptr()), C.c_int64(n), C.c_void_p(wsp),
                                            C.c_int64(nb), None))
    torch.cuda.synchronize()
    assert torch.equal(ya, yb)
    y = m(rdv.wrap(xd)).as_tensor("torch")  # the API path takes the unpacked entry
    assert torch.equal(y, ya)


def test_output_buffer_cached_per_structure_and_shape():
    x, layers = WL.c1(256)
    m1 = _chain(layers, ["relu"] * 4 + ["none"])
    m2 = _chain(layers, ["relu"] * 4 + ["none"])
    a = m1(x.cuda())
    b = m2(x.cuda())
    assert a is b  # same structure, same row shape -> same evaluator output (maths:1466-1476)
    c = m1(x[:128].cuda())
    assert c is not a and c.shape == (128, 4)


def test_inplace_weight_update_is_seen():
    x, layers = WL.c1(64)
    w0 = layers[0][0].cuda()
    lin0 = rdv.linear(w0, layers[0][1].cuda(), f16=True)
    m = lin0
    for w, b in layers[1:]:
        m = m >> rdv.relu >> rdv.linear(w.cuda(), b.cuda(), f16=True)
    y1 = m(x.cuda()).as_tensor("torch").clone()
    w0.mul_(0.5)  # in place, same pointer
    y2 = m(x.cuda()).as_tensor("torch").clone()
    assert not torch.equal(y1, y2)
    ref = O.mlp_forward(x.numpy(), [(w0.cpu().numpy(), layers[0][1].numpy())] + _np_layers(layers[1:]),
                        ["relu"] * 4 + ["none"], ["f16"] * 5)
    _assert_fp16_parity(y2.cpu().numpy(), ref, "updated weights")


def test_weight_update_without_version_bump_is_seen():
    """A write through `.data` (or any alias that torch's version counter does
    not track) is seen by the next call: the packed block is rebuilt from the
    weight buffers at every call, as the reference reads its weights through
    pointers at every dispatch."""
    x, layers = WL.c1(64)
    w0 = layers[0][0].cuda()
    m = rdv.linear(w0, layers[0][1].cuda(), f16=True)
    for w, b in layers[1:]:
        m = m >> rdv.relu >> rdv.linear(w.cuda(), b.cuda(), f16=True)
    y1 = m(x.cuda()).as_tensor("torch").clone()
    v = w0._version
    w0.data.mul_(0.25)
    assert w0._version == v  # the counter did not move
    y2 = m(x.cuda()).as_tensor("torch").clone()
    assert not torch.equal(y1, y2)
    ref = O.mlp_forward(x.numpy(), [(w0.cpu().numpy(), layers[0][1].numpy())] + _np_layers(layers[1:]),
                        ["relu"] * 4 + ["none"], ["f16"] * 5)
    _assert_fp16_parity(y2.cpu().numpy(), ref, "weights updated through .data")


def test_shape_errors_raise_before_launch():
    x, layers = WL.c1(64)
    m = _chain(layers, ["relu"] * 4 + ["none"])
    with pytest.raises(TypeError):
        m(torch.zeros(64, 5, device="cuda"))
    with pytest.raises(TypeError):
        rdv.linear(torch.zeros(8, 3), torch.zeros(8)) >> rdv.linear(torch.zeros(4, 9), torch.zeros(4))
    with pytest.raises(AssertionError):
        rdv.linear(torch.zeros(8, 3), torch.zeros(7))


def test_profiling_counter():
    x, layers = WL.c1(4096)
    m = _chain(layers, ["relu"] * 4 + ["none"])
    rdv.profiling(True)
    rdv.reset_submit_times()
    m(x.cuda())
    t = rdv.profiling_submit_times()
    rdv.profiling(False)
    assert t > 0.0


def test_dispatch_map_evaluator_and_deferred_kwargs():
    """rdv.dispatch(MapEvaluator(map, input, output), rows) runs the same
    kernels as map(x); keyword arguments to a call bind deferred names for
    that call only."""
    x, layers = WL.c1(1000)
    m = _chain(layers, ["relu"] * 4 + ["none"])
    xd = x.cuda()
    want = m(rdv.wrap(xd), scale=torch.ones(1, device="cuda")).as_tensor("torch").clone()
    y = torch.full((1000, 4), float("nan"), device="cuda")
    rdv.dispatch(rdv.MapEvaluator(m, rdv.wrap(xd), y), 1000)
    assert torch.equal(y, want)
    with pytest.raises(RuntimeError):
        rdv.Deferred("scale").resolve()  # unbound again after the call


@pytest.mark.parametrize("n", [5, 9000])
@pytest.mark.parametrize("dims", [[1, 3], [3, 5], [7, 3], [33, 6], [101, 5], [255, 130]])
def test_f32_chain_keeps_negative_zero(dims, n):
    """Every product rounds to -0 on top of a sum of -0: the outputs are -0 to the sign bit, as of a loop of fused
    multiply-adds, at widths that the 4-wide matrix products pad."""
    g = WL.gen(3)
    w = torch.rand(dims[1], dims[0], generator=g) * 1e-30 + 1e-31
    x = -torch.rand(n, dims[0], generator=g) * 1e-30 - 1e-31
    y = _chain([(w, torch.full((dims[1],), -0.0))], ["none"], f16=[False])(x.cuda()).as_tensor("torch").cpu()
    assert bool((y == 0).all()) and bool(torch.signbit(y).all()), f"{int((~torch.signbit(y)).sum())} of {y.numel()} are +0"
