"""``mlpmk_convert`` (csrc/convert.hip): casts, zero padding and cropping of
several matrices in one launch, bit for bit what torch's conversions give
(the casts around the reference's kernels are the framework's,
/root/reference/mlp_fused.md:159-172)."""
import itertools

import pytest
import torch

from mlpmk import _lib, ops

A = 1 << 20


def test_validation_before_any_launch():
    lib = _lib.get()

    def call(src=A, sd=0, dst=A, dd=1, shape=(4, 4, 4, 4), n=1):
        return lib.mlpmk_convert(n, (_lib.c_void_p * 1)(src), (_lib.c_int * 1)(sd), (_lib.c_void_p * 1)(dst),
                                 (_lib.c_int * 1)(dd), (_lib.c_int64 * 4)(*shape), None)

    assert call(n=0) == 0 and call(shape=(4, 4, 0, 4)) == 0
    assert call(n=17) == 1 and call(n=-1) == 1 and call(sd=7) == 1 and call(shape=(-1, 4, 4, 4)) == 1
    assert call(src=None) == 1 and call(dst=A + 4) == 3 and call(src=A + 2) == 3 and call(src=A + 1, sd=1) == 3
    assert call(shape=(1 << 16, 1 << 16, 4, 4)) == 2


def test_cpu_tensors_and_other_types_take_torch_operations():
    s = torch.arange(6.0, dtype=torch.float64).reshape(2, 3)
    d = torch.empty((3, 2), dtype=torch.float16)
    ops.convert([(s, d)], torch.device("cpu"))
    assert d.tolist() == [[0, 1], [3, 4], [0, 0]]


TYPES = [torch.float32, torch.float16, torch.bfloat16]


def _special(dt):
    bits = torch.tensor([0, 1, -2**31, 0x7f800000, -0x800000, 0x7fc00000, 0x00000001, 0x007fffff, 0x33000000, 0x33000001,
                         0x477fefff, 0x477ff000, 0x3f808000, 0x3f818000, 0x7f7fffff, 0x38800000, 0x387fc000],
                        dtype=torch.int64).to(torch.int32).view(torch.float32)
    return bits.to(dt)


@pytest.mark.gpu
@pytest.mark.parametrize("sd,dd", list(itertools.product(TYPES, TYPES)))
def test_convert_matches_torch_bit_for_bit(sd, dd):
    g = torch.Generator(device="cuda").manual_seed(1)
    shapes = [((1, 1), (1, 1)), ((5, 3), (5, 16)), ((5, 16), (3, 16)), ((7, 4), (7, 8)), ((3, 64), (16, 64)),
              ((1000, 63), (1000, 64)), ((100, 17), (90, 5)), ((33, 128), (33, 128)), ((0, 4), (2, 4)), ((9, 9), (9, 9))]
    pairs = []
    for s, d in shapes:
        src = (torch.randn(s, generator=g, device="cuda") * 1e3).to(sd)
        sp = _special(sd).cuda()
        src.view(-1)[: min(src.numel(), sp.numel())] = sp[: src.numel()]
        pairs.append((src, torch.full(d, 7.0, dtype=dd, device="cuda")))
    flat = torch.randn(1 + 40 * 8, generator=g, device="cuda").to(sd)
    pairs.append((flat[1:].view(40, 8), torch.empty((40, 8), dtype=dd, device="cuda")))  # off a 16-byte boundary
    assert all(ops._convertible(s, s.device) for s, _ in pairs)
    ops.convert(pairs, pairs[0][0].device)
    view = torch.int32 if dd == torch.float32 else torch.int16
    for s, d in pairs:
        ref = torch.zeros_like(d)
        r, c = min(s.shape[0], d.shape[0]), min(s.shape[1], d.shape[1])
        ref[:r, :c] = s[:r, :c].to(dd)
        nan = torch.isnan(ref)
        assert torch.equal(torch.isnan(d), nan)
        assert torch.equal(d.view(view)[~nan], ref.view(view)[~nan]), (s.shape, d.shape)


@pytest.mark.gpu
def test_padded_module_gradients_have_the_parameters_types():
    import fused_mlp

    for dt in (torch.float16, torch.float32):
        model = fused_mlp.FusedMLPSoftplus(D=3, H=64, out_features=5, n_layers=3).cuda().to(dt)
        x = torch.rand(777, 3, device="cuda").to(dt).requires_grad_()
        out = model(x)
        dout = torch.randn_like(out)
        got = torch.autograd.grad(out, [x, *model.weights], dout)
        xs = x.detach().double().requires_grad_()
        ws = [w.detach().double().requires_grad_() for w in model.weights]
        a = xs
        for i, w in enumerate(ws):
            a = a @ w
            if i < 2:
                a = torch.nn.functional.softplus(a)
        want = torch.autograd.grad(a, [xs, *ws], dout.double())
        for g, r in zip(got, want):
            assert g.dtype == dt and g.shape == r.shape
            assert ((g.double() - r).norm() / r.norm()).item() < 1e-2


def test_more_matrices_than_one_call_takes_go_in_several(monkeypatch):
    calls = []

    def launch(dev, fn, *args):
        calls.append(len(args[0]) // 8 if isinstance(args[0], list) else args[0])
        return 0

    monkeypatch.setattr(ops, "_launch", launch)
    items = [v for i in range(35) for v in (A, 0, A, 1, 4, 4, 4, 4)]
    ops._convert_raw(torch.device("cuda", 0), items)
    assert calls == [16, 16, 3]
    ops._convert_raw(torch.device("cuda", 0), [])
    assert len(calls) == 3


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layers", [16, 17, 33])
def test_deep_16_bit_modules_train(layers, dt):
    # one gradient per layer to convert: more of them than one call takes
    import fused_mlp

    torch.manual_seed(layers)
    model = fused_mlp.FusedMLPSoftplus(D=24, H=32, out_features=8, n_layers=layers).cuda()
    with torch.no_grad():
        for w in model.weights:
            w *= 1.5  # gradients of every layer between 1e-2 and 1e4: normal in both types
    model.to(dt)
    x = torch.randn(129, 24, device="cuda").to(dt).requires_grad_()
    out = model(x)
    got = torch.autograd.grad(out, [x, *model.weights], torch.ones_like(out))
    ws = [w.detach().double().requires_grad_() for w in model.weights]
    xs = x.detach().double().requires_grad_()
    a = xs
    for i, w in enumerate(ws):
        a = a @ w
        if i + 1 < layers:
            h = torch.nn.functional.softplus(a)
            a = h + (h.to(dt).double() - h).detach()  # rounded between layers, as the network rounds it
    want = torch.autograd.grad(a, [xs, *ws], torch.ones_like(a))
    # each layer's data gradient is rounded to dt once: 2^-11 (2^-8) a layer
    tol = 4 * layers ** 0.5 * (2.0 ** -11 if dt == torch.float16 else 2.0 ** -8)
    for g, r in zip(got, want):
        assert g.dtype == dt and g.shape == r.shape
        assert ((g.double() - r).norm() / r.norm()).item() <= tol


@pytest.mark.parametrize("pad", [0, 13])
@pytest.mark.parametrize("layout", ["rows", "transposed", "slice", "expanded"])
def test_strided_inputs_are_cast_while_they_are_gathered(monkeypatch, layout, pad):
    g = torch.Generator().manual_seed(0)
    x = {"rows": lambda: torch.randn((40, 3), generator=g), "transposed": lambda: torch.randn((3, 40), generator=g).t(),
         "slice": lambda: torch.randn((40, 9), generator=g)[:, 2:5],
         "expanded": lambda: torch.randn((1, 3), generator=g).expand(40, 3)}[layout]()
    w = torch.randn((3, 16), generator=g)
    seen, convert = [], ops.convert
    monkeypatch.setattr(ops, "convert", lambda pairs, dev: (seen.extend(s for s, _ in pairs), convert(pairs, dev)))
    xc, (wc,) = ops.as_inputs(x, [w], torch.float16, pad)
    assert xc.is_contiguous() and wc.is_contiguous()
    assert torch.equal(xc, torch.nn.functional.pad(x, (0, pad)).half())
    assert torch.equal(wc, torch.nn.functional.pad(w, (0, 0, 0, pad)).half())
    # only what lies in rows reaches the conversion launch
    assert [s.data_ptr() for s in seen] == ([x.data_ptr()] if layout == "rows" else []) + [w.data_ptr()]


@pytest.mark.gpu
@pytest.mark.parametrize("sd,dd", list(itertools.product(TYPES, TYPES)))
@pytest.mark.parametrize("off", [0, 1, 3])
def test_padding_to_whole_pieces_from_any_element_boundary(sd, dd, off):
    # pieces of eight that lie in the row, straddle its end, or lie past it or
    # past the last row, from sources that start off a 16-byte boundary
    g = torch.Generator(device="cuda").manual_seed(off)
    view = torch.int32 if dd == torch.float32 else torch.int16
    pairs = []
    for (r, c), (dr, dc) in [((301, 63), (301, 64)), ((70, 13), (70, 16)), ((3, 8), (5, 16)), ((9, 7), (9, 8)),
                             ((40, 24), (41, 24)), ((17, 100), (20, 112)), ((33, 21), (30, 16)), ((6, 17), (6, 20))]:
        src = torch.randn(off + r * c, generator=g, device="cuda").to(sd)[off:].view(r, c)
        pairs.append((src, torch.full((dr, dc), 7.0, dtype=dd, device="cuda")))
    ops.convert(pairs, pairs[0][0].device)
    for s, d in pairs:
        ref = torch.zeros_like(d)
        r, c = min(s.shape[0], d.shape[0]), min(s.shape[1], d.shape[1])
        ref[:r, :c] = s[:r, :c].to(dd)
        assert torch.equal(d.view(view), ref.view(view)), (s.shape, d.shape)
