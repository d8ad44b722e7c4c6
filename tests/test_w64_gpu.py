"""Runtime-width kernels compiled at width 64 (csrc/fwd_w64.hip, the GB64
networks of csrc/bwd.hip): every depth, widths on both sides of the 64-feature
limit, batches around the row blocks and the two backward forms, against the
CPU oracle (/root/reference/kernel.py:60-123, mlp_fused.md:88-95).  Tolerances
as for the 128-wide runtime-width kernels: outputs 1e-2, weight gradients per
entry 2e-2 |ref| + 2e-3 max|ref| and relative Frobenius 1e-2."""
import numpy as np
import pytest
import torch

from mlpmk import ops
from oracle import mlp_oracle as orc

SHAPES = [(64, 64, 64), (16, 16, 1), (16, 64, 48, 5), (64, 80, 64, 64), (32, 64, 64, 64, 4), (64, 16, 32, 48, 64),
          (16, 64, 64, 64, 64, 8), (48, 32, 64, 16, 64, 64)]


@pytest.mark.parametrize("L", [4, 5])
def test_deep_backward_without_a_workspace_is_refused(L):
    # as at width 128, although these kernels need no hand-over of dz
    from mlpmk import _lib

    if torch.cuda.is_available():
        pytest.skip("argument checks only")
    lib = _lib.get()
    dims = (64,) * (L + 1)
    pd, _k = _lib.int_array(list(dims))
    a = [1 << 20] * L
    arr = (_lib.c_void_p * L)(*a)
    rc = lib.mlpmk_bwd(L, pd, 1, 1 << 20, arr, arr, 1 << 20, 64, None, arr, 65536, None)
    assert rc == 1 and b"workspace" in lib.mlpmk_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("dims", SHAPES)
@pytest.mark.parametrize("m", [1, 129, 16384, 16385, 40001])
def test_w64_forward_and_backward_match_oracle(dims, m):
    x, ws = orc.make_inputs(dims, m, seed=m % 1000 + len(dims))
    xd = torch.from_numpy(x).cuda()
    wd = [torch.from_numpy(w).cuda() for w in ws]
    out, hs = ops.fwd(xd, wd, stash=True)
    ref, ref_h = orc.forward(x, ws, return_hidden=True)
    ok, err, _ = orc.allclose_report(out.float().cpu().numpy(), ref, 1e-2, 1e-2)
    assert ok, f"out {err}"
    assert torch.equal(ops.fwd(xd, wd), out)
    for h, r in zip(hs, ref_h):
        ok, err, _ = orc.allclose_report(h.cpu().numpy(), r, 1e-2, 1e-2)
        assert ok, f"stash {err}"
    rng = np.random.default_rng(m)
    dout = rng.standard_normal((m, dims[-1])).astype(np.float16)
    dws = [torch.full((dims[i], dims[i + 1]), float("nan"), device="cuda") for i in range(len(ws))]
    dx = torch.empty_like(xd)
    ops.bwd(xd, wd, hs, torch.from_numpy(dout).cuda(), dws, dx, accumulate=False)
    rdws, rdx = orc.backward(x, ws, [h.cpu().numpy() for h in hs], dout.astype(np.float32))
    ok, err, _ = orc.allclose_report(dx.float().cpu().numpy(), rdx, 1e-2, 1e-2)
    assert ok, f"dx {err}"
    for i, (d, r) in enumerate(zip(dws, rdws)):
        g, scale = d.cpu().numpy().astype(np.float64), np.abs(r).max()
        assert np.all(np.abs(g - r) <= 2e-2 * np.abs(r) + 2e-3 * scale), f"dW{i + 1}"
        assert np.linalg.norm(g - r) <= 1e-2 * np.linalg.norm(r), f"dW{i + 1}"
