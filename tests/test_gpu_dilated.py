"""Dilated neighborhoods: all sub-grids of one size in one launch, against the dense-mask oracle."""
import ctypes

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
    ((2, 2, 26, 32, 64), 13, 2, F16, "proj"),    # whole sub-grids of 208 pixels, the window as large
    ((1, 3, 21, 40, 56), 5, 3, F16, "plain"),    # whole ones of two sizes, head_dim below a built one
    ((2, 1, 40, 48, 16), 3, 7, BF16, "plain"),   # ... of four sizes, 30 to 42 pixels
    ((1, 2, 28, 30, 32), 7, 2, BF16, "plain"),   # 210 pixels: two beyond the middle size
    ((3, 22, 32, 32, 64), 5, 2, F16, "proj"),    # 256 pixels: the largest, whole in the backward only
    ((9, 8, 16, 24, 32), 7, 2, BF16, "proj"),    # 96 pixels: all of the smallest size
    ((2, 64, 14, 15, 32), 7, 1, BF16, "proj"),   # undilated images taken whole in the backward
    ((3, 90, 9, 10, 40), 9, 1, F16, "plain"),    # ... and in the forward
    ((1, 2, 34, 32, 32), 9, 2, BF16, "plain"),   # 272 pixels: one row more than a workgroup takes
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
    assert (dil == 1 or o.is_contiguous()) and all(t.is_contiguous() for t in got)
    assert_close(tuple(t.detach().cpu() for t in (o, *got)), (o_ref.detach(), *ref), dtype, "dilated")


def test_column_walk_keeps_rows_of_its_own_sub_grid_only():
    # 4032 tiles over 512 workgroups in segments of a third of a column: the tile after a segment lies
    # one row of tiles lower in the next sub-grid of the same batch entry and head
    ensure_built()
    from e_natten_amd import natten2d
    shape, ks, dil = (8, 7, 96, 48, 128), 5, 2
    q, k, v, g = make_inputs(shape, BF16, seed=47)
    print("case column walk", shape, "k=%d dilation=%d" % (ks, dil), flush=True)
    scale = shape[-1] ** -0.5
    x = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    o = natten2d(*x, ks, scale, dil)
    got = [t.detach().cpu() for t in (o, *torch.autograd.grad(o, x, g.cuda()))]
    for i in range(dil):
        for j in range(dil):
            sub = (slice(0, 1), slice(None), slice(i, None, dil), slice(j, None, dil))
            ref_x = [t[sub].double().requires_grad_(True) for t in (q, k, v)]
            o_ref = O.natten2d_dense_mask(*ref_x, ks, scale)
            ref = (o_ref.detach(), *torch.autograd.grad(o_ref, ref_x, g[sub].double()))
            assert_close([t[sub] for t in got], ref, BF16, "sub-grid %d %d" % (i, j))


@pytest.mark.parametrize("shape,ks,dtype", [
    ((9, 38, 41, 35, 32), 7, BF16),   # four sizes of sub-grids, 3078 tiles in each
    ((9, 40, 40, 36, 64), 3, F16),    # 3240 tiles
    ((8, 64, 32, 34, 128), 5, BF16),  # 3072 tiles: the backward only
    ((8, 32, 32, 30, 128), 11, F16),  # 1024 tiles
    ((19, 37, 40, 36, 48), 5, BF16),  # a head_dim between the built ones: 6327 tiles, the backward only
])
def test_large_sub_grids_run_one_after_the_other(shape, ks, dtype):
    ensure_built()
    from e_natten_amd import natten2d
    print("case large sub-grids", shape, dtype, "k=%d dilation=2" % ks, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(83)
    B, N, H, W, d = shape
    x = torch.randn((B, H, W, 4, N, d), generator=gen, device="cuda", dtype=dtype)
    q, k, v, g = (t.permute(0, 3, 1, 2, 4) for t in x.unbind(3))
    q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
    o = natten2d(q, k, v, ks, d ** -0.5, 2)
    got = (o, *torch.autograd.grad(o, (q, k, v), g))
    one = (slice(B - 1, B), slice(N - 2, N))  # (every image is the same computation on other data)
    xr = [t[one].detach().cpu().double().requires_grad_(True) for t in (q, k, v)]
    o_ref = O.natten2d_dilated_dense_mask(*xr, ks, 2, d ** -0.5)
    ref = (o_ref.detach(), *torch.autograd.grad(o_ref, xr, g[one].cpu().double()))
    assert_close([t.detach()[one].cpu() for t in got], ref, dtype, "large sub-grids")


@pytest.mark.parametrize("shape,ks,dil,dtype", [
    ((8, 16, 14, 14, 64), 9, 1, BF16),
    ((2, 64, 14, 14, 32), 7, 1, F16),
    ((2, 64, 9, 10, 40), 9, 1, F16),
    ((2, 4, 28, 28, 32), 7, 2, BF16),
    ((1, 6, 32, 32, 64), 5, 2, F16),
])
def test_keys_and_values_with_a_common_component(shape, ks, dil, dtype):
    # dP is then large against its spread over a window, and an error of delta, which the whole
    # window shares, is multiplied by the common component of the keys
    ensure_built()
    from e_natten_amd import natten2d
    q, k, v, g = make_inputs(shape, torch.float32, seed=53)
    q, k, v, g = (t.to(dtype) for t in (q, k + 2, v + 2, g))
    print("case common component", shape, dtype, "k=%d dilation=%d" % (ks, dil), flush=True)
    scale = shape[-1] ** -0.5
    x = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    o = natten2d(*x, ks, scale, dil)
    got = [t.detach().cpu()[:1] for t in (o, *torch.autograd.grad(o, x, g.cuda()))]
    x = [t[:1].double().requires_grad_(True) for t in (q, k, v)]
    o_ref = O.natten2d_dilated_dense_mask(*x, ks, dil, scale)
    ref = (o_ref.detach(), *torch.autograd.grad(o_ref, x, g[:1].double()))
    for name, a, b in zip(("O", "dQ", "dK", "dV"), got, ref):
        norm = ((a.double() - b).norm() / b.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        # a bfloat16 rounding is 1.7e-3 of a tensor in 2-norm (float16: an eighth); P and dS carry one
        # each, and in dQ keys of rms sqrt(5) multiply it, of which only the spread of 1 shows in the
        # result: sqrt(2 * 5) * 1.7e-3 = 5.4e-3, and half as much again for the results' own
        assert norm <= (8e-3 if dtype == BF16 else 1e-3), (name, norm)


def test_logits_far_from_zero():
    # images taken whole, logits of -1e32 that are equal over a window: the probabilities are uniform
    ensure_built()
    from e_natten_amd import natten2d
    H, W, ks = 9, 10, 9
    q, k, v, _ = make_inputs((3, 90, H, W, 32), BF16, seed=61)
    q, k = torch.zeros_like(q), torch.zeros_like(k)
    q[..., 0], k[..., 0] = 1e16, -1e16
    o = natten2d(q.cuda(), k.cuda(), v.cuda(), ks).cpu().double()
    ref = (O.neighbour_mask(H, W, ks).double() / ks ** 2 @ v.double().flatten(2, 3)).view(v.shape)
    norm = ((o - ref).norm() / ref.norm()).item()
    print("    O 2-norm %.2e" % norm, flush=True)
    assert norm <= 4e-3, norm  # (the rounding of the result, 1.7e-3, and of P)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_gradient_strides_that_16_byte_stores_do_not_take(axis):
    # images that would be taken whole; a batch, head or row stride of the gradients that is no
    # multiple of 8 elements
    from e_natten_amd import _lib
    lib = ensure_built()
    B, N, H, W, D = shape = (2, 65, 14, 14, 32)
    ks = 7
    print("case gradient strides", shape, "axis", axis, flush=True)
    q, k, v, g = (t.cuda() for t in make_inputs(shape, BF16, seed=67))
    o = torch.empty_like(q)
    lse = torch.empty(shape[:-1], dtype=torch.float32, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert lib.enatten2d_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), B, N, H, W, D,
                             ks, _lib.BF16, None, None, None, None, 0.2, st) == 0
    strides = [N * H * W * D, H * W * D, W * D, D]
    for i in range(axis, -1, -1):  # 4 more elements along `axis`, the outer axes made to fit
        strides[i] = strides[i + 1] * shape[i + 1] + (4 if i == axis else 0)
    res = []
    for gs in (None, strides):
        views = [torch.zeros(B * (strides[0] if gs else N * H * W * D), dtype=BF16, device="cuda").as_strided(
            shape, (*(gs or (N * H * W * D, H * W * D, W * D, D)), 1)) for _ in range(3)]
        ws = torch.empty(lib.enatten2d_bwd_workspace_bytes(B, N, H, W, D, ks, _lib.BF16), dtype=torch.uint8,
                         device="cuda")
        assert lib.enatten2d_bwd_into(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), g.data_ptr(), lse.data_ptr(),
            *(t.data_ptr() for t in views), ws.data_ptr(), B, N, H, W, D, ks, _lib.BF16, None, None, None, None,
            None, (ctypes.c_int64 * 4)(*gs) if gs else None, 0.2, st) == 0
        res.append(views)
    torch.cuda.synchronize()
    assert_close([t.cpu() for t in (o, *res[1])], [t.cpu() for t in (o, *res[0])], BF16, "axis %d" % axis)


def test_more_images_than_a_launch_of_one_workgroup_each_holds():
    # 8.4e6 images of 98 pixels: 512 threads for each would be more than the 2^32 of a launch.  q, k, v and
    # dO are one image, expanded: every image's results are those of the first
    ensure_built()
    shape, ks = ((1 << 23) + 8, 1, 7, 14, 8), 7
    print("case many images", shape, flush=True)
    one = make_inputs((1, *shape[1:]), BF16, seed=71)
    q, k, v, g = (t.cuda().expand(shape) for t in one)
    o, lse = torch.ops.enatten.na2d_fwd(q, k, v, ks, 0.3)
    x = [t.double().requires_grad_(True) for t in one[:3]]
    o_ref = O.natten2d_dense_mask(*x, ks, 0.3)
    ref = (o_ref.detach(), *torch.autograd.grad(o_ref, x, one[3].double()))
    got = (o, *torch.ops.enatten.na2d_bwd(q, k, v, o, lse, g, ks, 0.3))
    assert_close([t[:1].cpu() for t in got], ref, BF16, "first image")
    for t in got:
        for part in t.split(1 << 20):
            assert (part == t[:1]).all()
    del o, lse, got, t, part
    torch.cuda.empty_cache()


def test_values_that_are_not_finite_stay_in_their_windows():
    # sub-grids that a workgroup takes whole: a NaN in v reaches the queries that see it, and the
    # keys that those see, alone
    ensure_built()
    from e_natten_amd import natten2d
    ks, dil, side, at = 5, 2, 28, (9, 14)
    q, k, v, g = make_inputs((1, 66, side, side, 32), BF16, seed=29)  # (more images than CUs)
    clean = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    v[:, :, at[0], at[1]] = float("nan")
    dirty = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    res = []
    for x in (clean, dirty):
        o = natten2d(*x, ks, 0.2, dil)
        res.append([t.detach().float().cpu() for t in (o, *torch.autograd.grad(o, x, g.cuda()))])
    # along an axis: the window of each position of the residue class, as positions of the axis
    def windows(c):
        n = side // dil
        start = lambda i: min(max(i - ks // 2, 0), n - ks)
        return {i * dil + c % dil: [j * dil + c % dil for j in range(start(i), start(i) + ks)] for i in range(n)}
    rows, cols = windows(at[0]), windows(at[1])
    sees, reached = torch.zeros(side, side, dtype=torch.bool), torch.zeros(side, side, dtype=torch.bool)
    for y in (y for y in rows if at[0] in rows[y]):
        for x in (x for x in cols if at[1] in cols[x]):
            sees[y, x] = True
            for ky in rows[y]:
                reached[ky, cols[x]] = True
    for name, c, d, touched in zip(("O", "dQ", "dK", "dV"), *res,
                                   (sees, sees, reached, torch.zeros_like(sees))):
        assert d[:, :, touched].isnan().all(), name
        # (bfloat16 results of the same sums in another order, P and dS rounded to it on one side)
        c, d = c[:, :, ~touched], d[:, :, ~touched]
        norm = ((c - d).norm() / c.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        assert norm <= 6e-3, (name, norm)


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
