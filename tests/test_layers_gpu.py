"""``mlpmk_fwd_layers``: the one-launch forward of 16-bit networks wider than
256 or deeper than 5 layers (csrc/fwd_layers.hip), through ``fallback.fwd``,
against the CPU oracle (/root/reference/kernel.py:60-123 takes any width).

Sizes where the kernel changes its split: tiles of 32 and 64 rows and their
remainders, feature groups of 64 (widths just above a multiple, layers of at
most half or a quarter of the workgroup's features), ragged output widths and
inputs that are padded to a multiple of 8.  Tolerances are those of the other
16-bit forwards: fp16 outputs and activations within 1e-2 + 1e-2 |ref| of the
oracle that rounds h to fp16 between layers, bf16 within 3e-2.
"""
import ctypes

import numpy as np
import pytest
import torch

from mlpmk import _lib, fallback, ops
from oracle import mlp_oracle as orc

A = 1 << 20  # a 16-byte aligned address that is never read


def _workspace(dims, code):
    n = ctypes.c_int64(-1)
    p, _k = _lib.int_array(list(dims))
    return _lib.get().mlpmk_fwd_layers_workspace_size(len(dims) - 1, p, code, ctypes.byref(n)), n.value


@pytest.mark.parametrize("dims,code,want", [
    ((128, 512, 512, 128), 1, 2 * (128 * 512 + 512 * 512 + 512 * 128)),
    ((8, 8, 1), 2, 2 * 2 * 64 * 64),
    ((72, 100, 5), 1, None),            # a hidden width that is no multiple of 8
    ((128, 520, 128), 1, None),
    ((128, 512, 513), 2, None),
    ((128, 512, 128), 0, None),         # fp32 tensors
    ((16,) * 10, 1, None),              # nine layers
])
def test_workspace_and_supported_shapes(dims, code, want):
    rc, n = _workspace(dims, code)
    assert (rc, n) == ((0, want) if want is not None else (2, -1))


def test_validation_before_any_launch():
    lib = _lib.get()
    dims = (128, 512, 128)
    pd, _k = _lib.int_array(list(dims))
    w = (_lib.c_void_p * 2)(A, A)
    need = _workspace(dims, 1)[1]

    def call(x=A, out=A, ws=A, nb=need, m=4, wp=w):
        return lib.mlpmk_fwd_layers(2, pd, 1, x, wp, out, None, ws, nb, m, None)

    assert call(m=0) == 0
    assert call(m=-1) == 1 and call(x=None) == 1 and call(out=A + 2) == 3 and call(wp=None) == 1
    assert call(ws=None) == 1 and call(nb=need - 1) == 1 and call(ws=A + 8) == 3


SHAPES = [
    ((128, 512, 512, 128), [1, 31, 64, 65, 8192, 8193, 20000]),
    ((128, 272, 272, 128), [33, 1000]),
    ((64, 320, 24, 8), [129]),              # a quarter of the features, then one feature group
    ((200, 512, 448), [97]),                # output width above a whole number of groups
    ((16, 264, 264, 264, 3), [257]),        # ragged output, widths just above 256
    ((128, 512, 511), [70]),
    ((3, 512, 512, 4), [100, 9000]),        # padded input
    ((32,) * 9, [300]),                     # eight layers
    ((8, 8, 1), [5]),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dims,m", [(d, m) for d, ms in SHAPES for m in ms])
@pytest.mark.parametrize("elem", ["f16", "bf16"])
def test_layers_forward_and_stash_match_oracle(dims, m, elem):
    tol, dt = (1e-2, torch.float16) if elem == "f16" else (3e-2, torch.bfloat16)
    kw = {} if elem == "f16" else {"elem": "bf16"}
    x, ws = orc.make_inputs(dims, m, seed=m + len(dims), **kw)
    xd = torch.from_numpy(x).cuda().to(dt)
    wd = [torch.from_numpy(w).cuda().to(dt) for w in ws]
    res = fallback._fwd_layers(xd, wd, True)
    assert res is not None, "the kernel takes this network"
    out, hs = res
    ref, ref_h = orc.forward(x, ws, round_hidden=True, return_hidden=True, **kw)
    ok, err, _ = orc.allclose_report(out.float().cpu().numpy(), ref, tol, tol)
    assert ok, f"out: max|err| {err}"
    for i, (h, r) in enumerate(zip(hs, ref_h)):
        ok, err, _ = orc.allclose_report(h.cpu().numpy(), r, tol, tol)
        assert ok, f"h{i + 1}: max|err| {err}"
    assert torch.equal(fallback.fwd(xd, wd), out)  # inference: the same bits
    # the tile size changes no bit
    head = min(m, 40)
    assert torch.equal(fallback.fwd(xd[:head], wd), out[:head])


@pytest.mark.gpu
def test_layers_large_and_nonfinite_rows():
    dims, m = (128, 320, 320, 128), 500
    x, ws = orc.make_inputs(dims, m, seed=3)
    big = np.arange(m) % 7 == 0
    x[big] = (x[big].astype(np.float32) * 300.0).astype(np.float16)
    x[5, 3], x[300, 0] = np.inf, np.nan
    out = fallback.fwd(torch.from_numpy(x).cuda(), [torch.from_numpy(w).cuda() for w in ws]).float().cpu().numpy()
    ref = orc.forward(x, ws, round_hidden=True)
    bad = np.zeros(m, bool)
    bad[[5, 300]] = True
    assert not np.isfinite(out[bad]).any() and np.isfinite(out[~bad]).all()
    ok, err, _ = orc.allclose_report(out[~bad & ~big], ref[~bad & ~big], 1e-2, 1e-2)
    assert ok, err
    assert np.abs(out[big] - ref[big]).max() <= 2e-3 * np.abs(ref[big]).max()


@pytest.mark.gpu
def test_layers_small_activations_keep_their_digits():
    # softplus(z) = e^z (1 - e^z / 2 ...) for z << 0: the fp32 stash within a
    # few ulp of the float64 value of the same fp32 z (z = x w exactly: one
    # input feature), as the elementwise kernel of the layer-by-layer path is.
    # (The bound allows e^z from one rounded product, 1.2e-6 at z = -20; the test
    # over the whole range below holds it to 4 ulp.)
    z = torch.linspace(-20, 24, 352, device="cuda").bfloat16()
    x = torch.zeros((4, 8), device="cuda", dtype=torch.bfloat16)
    x[:, 0] = 1
    w0 = torch.zeros((8, 352), device="cuda", dtype=torch.bfloat16)
    w0[0] = z
    _, (h,) = fallback.fwd(x, [w0, torch.zeros((352, 8), device="cuda", dtype=torch.bfloat16)], stash=True)
    ref = torch.log1p(torch.exp(z.double()))
    assert ((h[0].double() - ref).abs() / ref).max().item() < 2e-6


@pytest.mark.gpu
def test_calls_the_kernel_does_not_take_still_run():
    # off a 16-byte boundary, fp32, a hidden width that is no multiple of 8, a
    # batch of more than two dimensions: the library-GEMM route, as before
    g = torch.Generator(device="cuda").manual_seed(0)
    flat = torch.randn(1 + 50 * 128, generator=g, device="cuda").half()
    x = flat[1:].view(50, 128)
    ws = [(torch.randn(s, generator=g, device="cuda") / 16).half() for s in ((128, 512), (512, 64))]
    assert fallback._fwd_layers(x, ws, False) is None
    assert fallback._fwd_layers(x.float(), [w.float() for w in ws], False) is None
    assert fallback._fwd_layers(x, [ws[0][:, :300].contiguous(), ws[1][:300]], False) is None
    x3 = x.reshape(2, 25, 128)
    assert fallback._fwd_layers(x3, ws, False) is None
    ref = torch.nn.functional.softplus(x.double() @ ws[0].double()) @ ws[1].double()
    for got in (fallback.fwd(x, ws), fallback.fwd(x.clone(), ws), fallback.fwd(x3, ws).reshape(50, 64)):
        torch.testing.assert_close(got.double(), ref, atol=1e-2, rtol=1e-2)
    assert ops.fwd_supported([128, 512, 64]) is False


def _classes(a):
    """0 finite, 1 +inf, 2 -inf, 3 NaN"""
    a = np.asarray(a, np.float32)
    return np.where(np.isnan(a), 3, np.where(np.isposinf(a), 1, np.where(np.isneginf(a), 2, 0)))


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(128, 272, 272, 128), (16, 264, 24, 8), (40, 288, 264, 8, 264, 5), (24, 320, 320, 16)])
@pytest.mark.parametrize("elem", ["f16", "bf16"])
def test_infinities_stay_where_the_oracle_has_them(dims, elem):
    # Weights of one sign per output column, none of them zero: an infinite
    # input (or a hidden value past the element type) gives +inf or softplus(-inf)
    # = 0, and no inf - inf or inf * 0 on the way.  A feature that pads a hidden
    # width must add nothing to that.
    dt = torch.float16 if elem == "f16" else torch.bfloat16
    m = 200
    x, ws = orc.make_inputs(dims, m, seed=7, elem=elem)
    rng = np.random.default_rng(8)
    sign = [np.where(rng.random(d) < (0.25 if i else 0.0), -1.0, 1.0).astype(np.float32) for i, d in enumerate(dims[1:])]
    ws = [orc.round_elem((np.abs(np.asarray(w, np.float32)) + 2.0 ** -6) * (0.125 if i else 1.0), elem) * s
          for i, (w, s) in enumerate(zip(ws, sign))]
    x = np.asarray(x, np.float32)
    x[3, 5], x[70, 0], x[130, 2] = np.inf, -np.inf, np.nan
    x[150] = orc.round_elem(np.abs(x[150]) * (3e4 if elem == "f16" else 1e38), elem)  # h past the largest element
    with np.errstate(invalid="ignore", over="ignore"):
        ref, ref_h = orc.forward(x, ws, round_hidden=True, return_hidden=True, elem=elem)
        ref = orc.round_elem(ref, elem)
    assert (_classes(ref)[3] != 3).all() and (_classes(ref)[[3, 150]] == 1).any() and np.isfinite(ref[70]).all()
    out, hs = fallback._fwd_layers(torch.from_numpy(x).cuda().to(dt), [torch.from_numpy(w).cuda().to(dt) for w in ws], True)
    for got, want in zip([out, *hs], [ref, *ref_h]):
        got = got.float().cpu().numpy()
        assert np.array_equal(_classes(got), _classes(want))
        fin = np.isfinite(want)
        fin[150] = False
        ok, err, _ = orc.allclose_report(got[fin], want[fin], 1e-2 if elem == "f16" else 3e-2, 1e-2 if elem == "f16" else 3e-2)
        assert ok, err


def test_empty_widths_are_left_to_the_library_route():
    # a layer of no features is no network of this kernel, and no error either
    for dims in ((16, 0, 8), (0, 320, 8), (16, 320, 0)):
        assert fallback._layers_workspace(dims, torch.float16) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(16, 0, 8), (0, 320, 8), (16, 320, 0), (5, 0, 0, 4)])
def test_networks_with_an_empty_layer_run(dims):
    from mlpmk.autograd import fused_mlp

    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn((9, dims[0]), generator=g, device="cuda").half().requires_grad_()
    ws = [torch.randn(s, generator=g, device="cuda").half().requires_grad_() for s in zip(dims, dims[1:])]
    out = fused_mlp(x, *ws)
    ref = x.double()
    for i, w in enumerate(ws):
        ref = ref @ w.double()
        ref = torch.nn.functional.softplus(ref) if i + 1 < len(ws) else ref
    torch.testing.assert_close(out.double(), ref, atol=1e-1, rtol=1e-2)
    grads = torch.autograd.grad(out.sum(), [x, *ws])
    want = torch.autograd.grad(ref.sum(), [x, *ws])
    for got, r in zip(grads, want):
        assert got.dtype == torch.float16 and got.shape == r.shape
        torch.testing.assert_close(got.double(), r.double(), atol=1e-1, rtol=2e-2)


@pytest.mark.gpu
def test_layers_softplus_keeps_its_digits_over_the_whole_range():
    # z = x w exactly, as above, down to where e^z leaves the normal fp32 range
    # (-87.3) and up past the threshold of 20, at fp16 steps.  The two-part
    # product leaves e^z with the roundings of the exponential (1 ulp), of the
    # correction and of the sum: 4 ulp of 2^-23 in all, as in the elementwise
    # kernel of the layer-by-layer path, which is held to the same bound.
    z = torch.cat([torch.linspace(-87, 24, 4096), torch.linspace(-1.5, 1.5, 4096)]).half().reshape(16, 512)
    for part in z.cuda():
        x = torch.zeros((4, 8), device="cuda", dtype=torch.float16)
        x[:, 0] = 1
        w0 = torch.zeros((8, 512), device="cuda", dtype=torch.float16)
        w0[0] = part
        _, (h,) = fallback._fwd_layers(x, [w0, torch.zeros((512, 8), device="cuda", dtype=torch.float16)], True)
        d = part.double()
        ref = torch.clamp(d, min=0) + torch.log1p(torch.exp(-d.abs()))
        for name, got in (("fwd_layers", h[0]), ("softplus_f32", fallback.softplus_f32(part.float()))):
            err = ((got.double() - ref).abs() / ref).max().item()
            assert err <= 4 * 2.0 ** -23, (name, part[0].item(), part[-1].item(), err)


@pytest.mark.parametrize("dims,m,gemms", [
    ((8, 8, 1), 399999, False), ((8, 8, 1), 400000, True), ((8, 8, 8, 8), 400000, True), ((16, 8, 16), 400000, True),
    ((24, 8, 8, 24), 1048575, False), ((24, 8, 8, 24), 1048576, True), ((63, 8, 8, 1), 1048576, True),
    ((16,) * 7, 4194304, False), ((16, 24, 16), 4194304, False), ((128, 512, 512, 128), 1048576, False),
])
def test_narrow_networks_of_many_rows_go_to_the_gemms(dims, m, gemms):
    assert fallback._gemms_faster(dims, m) is gemms


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(8, 8, 1), (3, 8, 8, 16)])
def test_both_routes_of_a_narrow_network_agree(dims):
    m = 400000
    x, ws = orc.make_inputs(dims, m, seed=1)
    xd, wd = torch.from_numpy(x).cuda(), [torch.from_numpy(w).cuda() for w in ws]
    assert fallback._fwd_layers(xd, wd, True) is None
    out, hs = fallback.fwd(xd, wd, stash=True)
    part, phs = fallback._fwd_layers(xd[: m - 1], wd, True)
    # fp32 accumulation and softplus on both routes: the stash within a few fp32
    # ulp of the largest terms, an output element within a rounding of h and out
    torch.testing.assert_close(out[: m - 1], part, atol=2.0 ** -9, rtol=2.0 ** -9)
    torch.testing.assert_close(hs[0][: m - 1], phs[0], atol=2e-6, rtol=2e-6)
    assert all(h.shape == (m, d) and h.dtype == torch.float32 for h, d in zip(hs, dims[1:]))
