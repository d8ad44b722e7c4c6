"""The two-pass backward (csrc/bwd_tp.hip) at the sizes where its kernels
change form: data-gradient tiles of 32 and 64 rows, weight-gradient blocks of
64 x 64 (4 waves), 128 x 128 (two groups of 4 waves that add up through LDS)
and 128 x 256 (8 waves), chunks of one, a few and many passes, ragged last
rows and the three forms of dL/dout, against float64 products of the same
tensors and stash (/root/reference/mlp_fused.md:88-95).  Tolerances: 16-bit as in
test_wide_gpu.py (2e-2 |ref| + 2e-3 max|ref|, Frobenius 1e-2; bf16 three
times that), fp32 as in test_fp32_gpu.py (1e-3, 1e-4, 5e-4)."""
import numpy as np
import pytest
import torch

from mlpmk import ops

pytestmark = pytest.mark.gpu

CASES = [
    # fp32: QUAD below 32,768 rows, PAIR from there (not below 64 features)
    ((128, 128, 128, 128), 32767, "f32"), ((128, 128, 128, 128), 32768, "f32"), ((128, 128, 128, 128), 65600, "f32"),
    ((32, 80, 112, 96, 24), 40001, "f32"), ((64, 64, 48, 8), 40001, "f32"), ((128, 128, 16), 70001, "f32"),
    # widths above 128: QUAD below 24,576, WIDE from there
    ((128, 256, 256, 128), 24575, "f16"), ((128, 256, 256, 128), 24576, "f16"), ((128, 256, 256, 128), 24701, "bf16"),
    ((144, 208, 16, 256, 136), 30001, "f16"), ((256, 256, 8), 25000, "bf16"), ((16, 144, 144, 144, 144, 72), 26000, "f16"),
    # data-gradient tiles: 32 rows up to 16,384, 64 from there
    ((128, 256, 256, 128), 16384, "f16"), ((128, 256, 256, 128), 16385, "f16"), ((96, 160, 104), 3, "f16"),
    ((128, 128, 128, 128), 33, "f16"), ((64, 128, 64, 32, 128, 120), 16449, "f32"),
    # weight-gradient forms by rows times blocks of 64 x 64 (48, 80, 32, 8, 20)
    ((256, 256, 256, 256), 11249, "f16"), ((256, 256, 256, 256), 11250, "bf16"), ((256,) * 6, 6750, "f16"),
    ((128, 256, 256, 128), 44999, "f16"), ((128, 256, 256, 128), 45000, "f16"), ((128, 128, 128), 109999, "f32"),
    ((128, 128, 128), 110000, "f32"), ((256, 256, 8), 27003, "f16"),
    # tiles of 32 and 64 rows by the rows that the CU with most gets, by the
    # hidden widths, and with resident weights
    ((128, 128, 128, 128), 131071, "f32"), ((128, 128, 128, 128), 131073, "f32"), ((32, 96, 96, 16), 20000, "f32"),
    ((32, 96, 96, 16), 24577, "f32"), ((16, 128, 128, 24), 16385, "f32"), ((16, 144, 144, 72), 24576, "bf16"),
    ((16, 144, 144, 72), 24577, "bf16"), ((64, 192, 208, 40), 16385, "f16"),
    # weights read in place below 32,768 rows, packed first from there
    ((128, 256, 256, 128), 32767, "bf16"), ((128, 256, 256, 128), 32768, "bf16"), ((144, 208, 72), 32768, "f16"),
    ((96, 160, 104), 33011, "bf16"), ((144, 176, 208, 136), 33011, "bf16"), ((256, 256, 256, 8), 32769, "f16"),
    ((16, 144, 144, 144, 144, 72), 32768, "bf16"), ((176, 256, 16, 256, 144, 136), 33011, "f16"),
]


@pytest.mark.parametrize("dims,m,elem", CASES)
@pytest.mark.parametrize("how", ["dense", "row", "scalar"])
def test_two_pass_backward_forms(dims, m, elem, how):
    dt = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[elem]
    rng = np.random.default_rng(m)
    x = torch.from_numpy(rng.standard_normal((m, dims[0]), dtype=np.float32)).to(dt)
    ws = [torch.from_numpy(rng.standard_normal((dims[i], dims[i + 1]), dtype=np.float32) / np.sqrt(dims[i])).to(dt)
          for i in range(len(dims) - 1)]
    xd, wd = x.cuda(), [w.cuda() for w in ws]
    _, hs = ops.fwd(xd, wd, stash=True)
    shape = {"dense": (m, dims[-1]), "row": (1, dims[-1]), "scalar": (1, 1)}[how]
    dout = torch.from_numpy(rng.standard_normal(shape, dtype=np.float32)).to(dt).cuda().expand(m, dims[-1])
    dws = [torch.full(tuple(w.shape), float("nan"), device="cuda") for w in ws]
    dx = torch.empty_like(xd)
    ops.bwd(xd, wd, hs, dout, dws, dx, accumulate=False)
    # float64 gradients of the same stash, on the GPU (plain products)
    dz = dout.double()
    tol, scale_tol, fro = {"f16": (2e-2, 2e-3, 1e-2), "bf16": (6e-2, 6e-3, 3e-2), "f32": (1e-3, 1e-4, 5e-4)}[elem]
    for l in range(len(ws) - 1, -1, -1):
        a = hs[l - 1].double() if l > 0 else xd.double()
        ref = a.t().contiguous() @ dz.contiguous()
        err = (dws[l].double() - ref).abs()
        assert bool((err <= tol * ref.abs() + scale_tol * ref.abs().max()).all()), f"dW{l + 1}: {err.max().item()}"
        assert (err.norm() / ref.norm()).item() <= fro, f"dW{l + 1}"
        dh = dz @ wd[l].double().t().contiguous()
        dz = dh * -torch.expm1(-hs[l - 1].double()) if l > 0 else dh
    rows = dz.abs().amax(dim=1, keepdim=True)
    assert bool(((dx.double() - dz).abs() <= max(tol / 2, 2e-4) * (dz.abs() + rows)).all()), "dx"


def _classes(t):
    """0 finite, 1 +inf, 2 -inf, 3 NaN"""
    return torch.isnan(t) * 3 + torch.isposinf(t) * 1 + torch.isneginf(t) * 2


@pytest.mark.parametrize("dims,m,elem", [
    ((80, 112, 48, 96, 24), 300, "f16"), ((16, 96, 80, 8), 5000, "bf16"), ((64, 80, 40), 33, "f16"),
    ((144, 208, 16, 256, 136), 1000, "f16"), ((96, 160, 104), 20000, "bf16"),       # weights as they are
    ((144, 208, 176, 136), 40001, "f16"), ((96, 160, 104), 32768, "bf16"),          # packed
])
def test_an_infinite_output_gradient_stays_infinite(dims, m, elem):
    # Weights and activations of one sign: dL/dout = inf in one place gives inf
    # everywhere it reaches and NaN nowhere.  The K-steps that pad a layer's
    # features to whole turns must add nothing to that.
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[elem]
    g = torch.Generator(device="cuda").manual_seed(m)
    x = (torch.rand((m, dims[0]), generator=g, device="cuda") + 0.1).to(dt)
    ws = [((torch.rand(s, generator=g, device="cuda") + 0.5) / s[0]).to(dt) for s in zip(dims, dims[1:])]
    _, hs = ops.fwd(x, ws, stash=True)
    dout = (torch.rand((m, dims[-1]), generator=g, device="cuda") + 0.1).to(dt)
    dout[m // 2, 3], dout[m - 1, 6] = float("inf"), float("-inf")
    dws = [torch.full(tuple(w.shape), float("nan"), device="cuda") for w in ws]
    dx = torch.empty_like(x)
    ops.bwd(x, ws, hs, dout, dws, dx, accumulate=False)
    want = torch.zeros((m, 1), dtype=torch.long, device="cuda")
    want[m // 2], want[m - 1] = 1, 2
    assert torch.equal(_classes(dx), want.expand(m, dims[0]))
    top = torch.zeros(dims[-1], dtype=torch.long, device="cuda")
    top[3], top[6] = 1, 2
    assert torch.equal(_classes(dws[-1]), top.expand(dims[-2], dims[-1]))
    for d in dws[:-1]:  # +inf of one row and -inf of the other meet
        assert torch.isnan(d).all()


@pytest.mark.parametrize("elem", ["f16", "f32"])
def test_output_gradient_rows_more_than_2_gib_apart(elem):
    # A column slice of a very wide gradient: the rows of a tile span more than
    # 2^31 bytes, and what lies between them (NaN here) is never an operand.
    dt, dims, m = (torch.float16, (144, 208, 72), 32) if elem == "f16" else (torch.float32, (80, 112, 72), 32)
    es = 2 if elem == "f16" else 4
    stride = (1 << 31) // (31 * es) // 8 * 8 + 4096
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn((m, dims[0]), generator=g, device="cuda").to(dt)
    ws = [(torch.randn(s, generator=g, device="cuda") / s[0] ** 0.5).to(dt) for s in zip(dims, dims[1:])]
    _, hs = ops.fwd(x, ws, stash=True)
    dout = torch.randn((m, dims[-1]), generator=g, device="cuda").to(dt)
    far = torch.full((m * stride,), float("nan"), dtype=dt, device="cuda").as_strided((m, dims[-1]), (stride, 1))
    far.copy_(dout)
    res = []
    for d in (dout, far):
        dws = [torch.zeros(tuple(w.shape), device="cuda") for w in ws]
        dx = torch.empty_like(x)
        ops.bwd(x, ws, hs, d, dws, dx)
        res.append([dx, *dws])
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dims,m,elem", [((144, 176, 208, 136), 33011, "bf16"), ((128, 256, 256, 128), 32768, "f16"),
                                         ((96, 160, 104), 40001, "f16"), ((16, 144, 144, 144, 144, 72), 32768, "bf16")])
def test_a_workspace_without_room_for_the_packed_weights_serves(dims, m, elem):
    # Both forms at one batch: the same fragments in the same order give the
    # bits of dx; dW differs by the order of its atomics only.
    from mlpmk import _lib

    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[elem]
    L = len(dims) - 1
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn((m, dims[0]), generator=g, device="cuda").to(dt)
    ws = [(torch.randn(s, generator=g, device="cuda") / s[0] ** 0.5).to(dt) for s in zip(dims, dims[1:])]
    _, hs = ops.fwd(x, ws, stash=True)
    dout = torch.randn((m, dims[-1]), generator=g, device="cuda").to(dt)
    need = ops.bwd_workspace_bytes(dims, m, True, dtype=dt)
    packed = sum(-(-k // 32) * (-(-n // 64) * 4) * 1024 for k, n in zip(dims, dims[1:]))
    lib, dev = _lib.get(), x.device
    buf = torch.empty(need, dtype=torch.uint8, device="cuda")
    res = []
    for nbytes, want in ((need, 0), (need - packed, 0), (need - packed - 256, 1)):
        dws = [torch.zeros(tuple(w.shape), device="cuda") for w in ws]
        dx = torch.full_like(x, float("nan"))
        buf[nbytes:] = 0xA5
        arr = lambda ts: (_lib.c_void_p * len(ts))(*[t.data_ptr() for t in ts])  # noqa: E731
        rc = ops._launch(dev, lib.mlpmk_bwd_ws, L, _lib.dims_array(dims), ops._fwd_code(dt), x.data_ptr(), arr(ws),
                         arr(hs), dout.data_ptr(), dims[-1], dx.data_ptr(), arr(dws), buf.data_ptr(), nbytes, m)
        torch.cuda.synchronize()
        assert rc == want and bool((buf[nbytes:] == 0xA5).all())
        if rc == 0:
            res.append((dx, dws))
    assert torch.equal(res[0][0], res[1][0]) and bool(torch.isfinite(res[0][0]).all())
    for a, b in zip(res[0][1], res[1][1]):
        assert ((a - b).norm() / a.norm()).item() < 1e-5  # fp32 sums in another order
