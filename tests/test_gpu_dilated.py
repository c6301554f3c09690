"""Dilated neighborhoods: all sub-grids of one size in one launch, against the dense-mask oracle."""
import pytest
import torch

from _util import O, assert_close, ensure_built, make_inputs

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("shape,ks,dil,dtype,layout", [
    ((2, 3, 28, 28, 32), 7, 4, BF16, "proj"),    # sub-grids of one window: a single 7x7 tile each
    ((1, 2, 37, 31, 32), 5, 3, BF16, "plain"),   # two sizes on both axes: four launches
    ((2, 2, 38, 54, 48), 7, 2, F16, "proj"),     # head_dim below a built one, inner tiles
    ((1, 1, 67, 70, 64), 13, 5, BF16, "plain"),  # largest window: two waves per block of keys
    ((1, 2, 44, 45, 128), 11, 4, F16, "proj"),   # one halo in LDS at a time, border tiles only
    ((1, 2, 24, 26, 64), 3, 8, BF16, "odd"),     # upstream gradient the 16-byte loads cannot take:
                                                 # the backward runs sub-grid by sub-grid
])
def test_dilated_sub_grids_in_one_launch(shape, ks, dil, dtype, layout):
    ensure_built()
    from e_natten_amd import natten2d
    q, k, v, g = make_inputs(shape, dtype, seed=23)
    print("case dilated", shape, dtype, "k=%d dilation=%d" % (ks, dil), layout, flush=True)
    scale = shape[-1] ** -0.5
    qr, kr, vr = (t.double().requires_grad_(True) for t in (q, k, v))
    o_ref = O.natten2d_dilated_dense_mask(qr, kr, vr, ks, dil, scale)
    ref = torch.autograd.grad(o_ref, (qr, kr, vr), g.double())
    if layout == "proj":
        qkv = torch.stack([t.permute(0, 2, 3, 1, 4) for t in (q, k, v)], dim=3).cuda()
        qg, kg, vg = (t.permute(0, 3, 1, 2, 4).requires_grad_(True) for t in qkv.unbind(3))
    else:
        qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    gg = g.cuda()
    if layout == "odd":
        buf = torch.empty(gg.numel() + 1, dtype=dtype, device="cuda")
        gg = buf[1:].view(shape).copy_(gg)
    o = natten2d(qg, kg, vg, ks, scale, dil)
    got = torch.autograd.grad(o, (qg, kg, vg), gg)
    assert o.is_contiguous() and all(t.is_contiguous() for t in got)
    assert_close(tuple(t.detach().cpu() for t in (o, *got)), (o_ref.detach(), *ref), dtype, "dilated")


def test_every_kind_of_window_traced_by_torch_compile():
    # as one graph: the operators carry meta kernels; the compiled function runs the same kernels
    ensure_built()
    from e_natten_amd import natten1d, natten2d, ops
    if not ops.NATIVE_BINDING:
        pytest.skip("native torch binding not built")

    def f(q, k, v, rpb, s):
        a = natten2d(q * 1.0, k, v, 5, 0.2, 2) + natten2d(q, k, v, 5, 0.2, rpb=rpb)
        a = a + natten2d(q, k, v, (3, 5), 0.2)
        return (a.float() ** 2).sum() + natten1d(s, s, s, 6, 0.2, is_causal=True).float().sum()

    q, k, v, _ = make_inputs((2, 2, 24, 20, 32), BF16, seed=5)
    x = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    x.append(torch.randn(2, 9, 9, device="cuda", dtype=BF16, requires_grad=True))
    x.append(torch.randn(2, 2, 200, 32, device="cuda", dtype=F16, requires_grad=True))
    want = f(*x)
    got = torch.compile(f, backend="aot_eager", fullgraph=True)(*x)
    assert torch.equal(got.detach(), want.detach())
    for a, b in zip(torch.autograd.grad(got, x), torch.autograd.grad(want, x)):
        assert torch.equal(a, b)
