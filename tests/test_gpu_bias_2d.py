"""Relative position bias on the matrix-core kernels, against the dense-mask oracle."""
import pytest
import torch

from _util import BF16_REL, O, ensure_built, make_inputs

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("shape,ks,dtype,layout", [
    ((2, 3, 14, 14, 32), 7, BF16, "proj"),      # border tiles only
    ((1, 2, 41, 35, 32), 5, F16, "plain"),      # inner tiles, ragged sides
    ((1, 2, 33, 30, 32), 3, BF16, "plain"),     # 6 tokens to a row: lane groups take turns
    ((2, 2, 40, 48, 64), 9, BF16, "proj"),      # tokens in two blocks, four to a row in the second
    ((8, 16, 32, 40, 64), 7, F16, "plain"),     # 16x8 tiles
    ((1, 2, 30, 41, 48), 7, BF16, "proj"),      # head_dim below a built one
    ((1, 2, 40, 31, 64), 13, BF16, "plain"),    # 16 tokens to a row, two waves per block of keys
    ((4, 20, 32, 40, 64), 11, F16, "plain"),    # one halo in LDS at a time, 16x8 tiles
    ((1, 2, 24, 32, 128), 5, BF16, "plain"),
    ((1, 1, 26, 29, 128), 9, F16, "proj"),      # one halo in LDS at a time
    ((1, 1, 22, 13, 128), 13, BF16, "plain"),   # frame body only; window = image on one axis
    ((1, 2, 5, 5, 16), 5, F16, "plain"),        # window = image
])
def test_bias(shape, ks, dtype, layout):
    ensure_built()
    from e_natten_amd import natten2d
    print("case bias", shape, dtype, "k=%d" % ks, layout, flush=True)
    q, k, v, g = make_inputs(shape, dtype, seed=37)
    scale = shape[-1] ** -0.5
    gen = torch.Generator().manual_seed(5)
    rpb = torch.randn(shape[1], 2 * ks - 1, 2 * ks - 1, generator=gen).to(dtype)
    if layout == "proj":
        qkv = torch.stack([t.permute(0, 2, 3, 1, 4) for t in (q, k, v)], dim=3).cuda()
        qg, kg, vg = (t.permute(0, 3, 1, 2, 4).requires_grad_(True) for t in qkv.unbind(3))
    else:
        qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    bg = rpb.cuda().requires_grad_(True)
    o = natten2d(qg, kg, vg, ks, scale, rpb=bg)
    got = (o, *torch.autograd.grad(o, (qg, kg, vg, bg), g.cuda()))
    # (the last heads only where there are many: a head is the same computation on other data; its
    # bias gradient sums over the whole batch)
    heads = slice(max(0, shape[1] - 3), None)
    qr, kr, vr, br = (t[:, heads].double().requires_grad_(True) for t in (q, k, v, rpb.unsqueeze(0)))
    o_ref = O.natten2d_window_dense_mask(qr, kr, vr, (ks, ks), scale=scale, rpb=br[0])
    ref = (o_ref.detach(), *torch.autograd.grad(o_ref, (qr, kr, vr, br), g[:, heads].double()))
    for name, x, r in zip(("O", "dQ", "dK", "dV", "dRPB"), got, ref):
        x = x.detach()
        x = (x[:, heads] if name != "dRPB" else x[heads].unsqueeze(0)).cpu()
        err, norm = O.rel_err(x, r), ((x.double() - r).norm() / r.norm()).item()
        print("   ", name, "max-abs / max %.2e" % err, "2-norm %.2e" % norm, flush=True)
        assert err <= BF16_REL, (name, err)
        # P and dS are carried to 16 bits or more: what is left is the rounding of the results (2^-9
        # of an element for bfloat16, 2^-12 for float16)
        assert norm <= (4e-3 if dtype == BF16 else 5e-4), (name, norm)
    again = torch.autograd.grad(natten2d(qg, kg, vg, ks, scale, rpb=bg), (qg, kg, vg, bg), g.cuda())
    assert all(torch.equal(a, b) for a, b in zip(again, got[1:])), "not bit-reproducible"


def _dense(q, k, v, rpb, ks, scale):
    """O in float64 through an explicit softmax (a fused one may not hold a log-sum-exp of -1e38)."""
    B, N, H, W, D = q.shape
    at = torch.arange(H * W)
    dy = at[None] // W - at[:, None] // W + ks - 1
    dx = at[None] % W - at[:, None] % W + ks - 1
    s = q.flatten(2, 3) @ k.flatten(2, 3).transpose(-1, -2) * scale
    s = s + rpb[:, dy.clamp(0, 2 * ks - 2), dx.clamp(0, 2 * ks - 2)]
    p = s.masked_fill(~O.neighbour_mask(H, W, ks), float("-inf")).softmax(-1)
    return (p @ v.flatten(2, 3)).view(q.shape)


def _both(x, ks, scale):
    """(O, dQ, dK, dV, dRPB) of the kernels and of the reference; x = (q, k, v, rpb, dO)."""
    from e_natten_amd import natten2d
    xg = [t.cuda().requires_grad_(True) for t in x[:4]]
    o = natten2d(*xg[:3], ks, scale, rpb=xg[3])
    got = [t.detach().cpu().double() for t in (o, *torch.autograd.grad(o, xg, x[4].cuda()))]
    xr = [t.double().requires_grad_(True) for t in x[:4]]
    o_ref = _dense(*xr, ks, scale)
    return got, [t.detach() for t in (o_ref, *torch.autograd.grad(o_ref, xr, x[4].double()))]


def _rpb(heads, ks, seed=5):
    return torch.randn(heads, 2 * ks - 1, 2 * ks - 1, generator=torch.Generator().manual_seed(seed))


NAMES = ("O", "dQ", "dK", "dV", "dRPB")


@pytest.mark.parametrize("shape,ks,dtype", [
    ((1, 2, 26, 24, 32), 5, BF16),
    ((1, 2, 20, 21, 128), 9, BF16),
    ((1, 2, 26, 29, 64), 11, BF16),
    ((1, 2, 24, 24, 32), 7, F16),
])
def test_bias_of_the_lowest_value(shape, ks, dtype):
    # head 0: every entry is the lowest finite value, which absorbs the logits: uniform probabilities.
    # head 1: the query itself and what follows it are masked out that way; the first query then
    # has nothing else
    ensure_built()
    print("case lowest bias", shape, dtype, "k=%d" % ks, flush=True)
    q, k, v, g = make_inputs(shape, dtype, seed=73)
    rpb = _rpb(2, ks).to(dtype)
    rpb[0] = torch.finfo(dtype).min
    rpb.view(2, -1)[1, (2 * ks - 1) ** 2 // 2:] = torch.finfo(dtype).min
    got, ref = _both((q, k, v, rpb, g), ks, shape[-1] ** -0.5)
    for name, x, r in zip(NAMES, got, ref):
        norm = ((x - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        # (bfloat16 as in test_bias.  Float16's lowest value leaves logits of -65504 their last 8 bits:
        # in float32 they are rounded to 2^-8, a probability by 1.1e-3 in the mean)
        assert norm <= (4e-3 if dtype == BF16 else 2e-3), (name, norm)


def test_gradients_beyond_float16():
    # dS of some 1e5, whose 16-bit terms would be an infinity and its negative, under a small softmax
    # scale: the gradients of q and k themselves are in range (that of the bias is not)
    ensure_built()
    q, k, v, g = make_inputs((1, 2, 24, 20, 64), F16, seed=43)
    got, ref = _both((q, k, v * 200, _rpb(2, 3).to(F16), g * 200), 3, 2.0 ** -10)
    for name, x, r in zip(NAMES[:4], got, ref):
        norm = ((x - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        assert norm <= 5e-4, (name, norm)  # (as in test_bias)


@pytest.mark.parametrize("shape,ks", [((1, 2, 28, 24, 32), 7), ((1, 1, 26, 28, 64), 13), ((1, 1, 20, 24, 128), 9)])
def test_float16_with_small_upstream_gradients(shape, ks):
    # dS of 1e-6 and less, which two float16 terms alone do not hold
    ensure_built()
    print("case small gradients", shape, ks, flush=True)
    q, k, v, g = make_inputs(shape, torch.float32, seed=59)
    x = [t.to(F16) for t in (q, k, v, _rpb(shape[1], ks), g * 1e-4)]
    got, ref = _both(x, ks, shape[-1] ** -0.5)
    for name, x, r in list(zip(NAMES, got, ref))[1:4]:
        norm = ((x - r).norm() / r.norm()).item()
        rounding = ((r.to(F16).double() - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e, of the result's rounding alone %.2e" % (norm, rounding), flush=True)
        assert norm <= 1.05 * rounding, (name, norm, rounding)


@pytest.mark.parametrize("which", ["k", "v", "dO"])
@pytest.mark.parametrize("shape,ks,dtype", [
    ((1, 2, 29, 24, 32), 5, BF16),    # inner tiles and border
    ((1, 1, 26, 28, 64), 13, F16),    # two waves per block of keys, one halo in LDS at a time
    ((1, 1, 20, 21, 128), 9, BF16),
    ((1, 1, 22, 21, 128), 11, F16),   # frame body only
])
def test_values_that_are_not_finite_stay_in_their_windows(shape, ks, dtype, which):
    # a NaN in one pixel of k, v or dO: only what the windows connect with it may be touched, though rows
    # outside a window are staged beside it
    ensure_built()
    print("case not finite", which, shape, dtype, "k=%d" % ks, flush=True)
    H, W = shape[2:4]
    at = 12 * W + 9
    q, k, v, g = make_inputs(shape, dtype, seed=79)
    rpb, scale = _rpb(shape[1], ks).to(dtype), shape[-1] ** -0.5
    _, ref = _both((q, k, v, rpb, g), ks, scale)
    {"k": k, "v": v, "dO": g}[which].flatten(2, 3)[:, :, at] = float("nan")
    got, _ = _both((q, k, v, rpb, g), ks, scale)
    mask = O.neighbour_mask(H, W, ks)
    only = torch.zeros(H * W, dtype=torch.bool)
    only[at] = True
    queries = only if which == "dO" else mask[:, at]   # queries with a gradient that is touched
    keys = mask[queries].any(0)                        # the keys that these see
    none = torch.zeros_like(only)
    pairs = (mask & queries[:, None]).nonzero()
    entries = torch.zeros(2 * ks - 1, 2 * ks - 1, dtype=torch.bool)
    entries[pairs[:, 1] // W - pairs[:, 0] // W + ks - 1, pairs[:, 1] % W - pairs[:, 0] % W + ks - 1] = True
    touched = (none if which == "dO" else queries, queries, keys, none if which == "v" else keys, entries.flatten())
    for name, x, r, t in zip(NAMES, got, ref, touched):
        x, r = ((y.flatten(2, 3) if name != "dRPB" else y.flatten(1)[None, :, :, None]) for y in (x, r))
        assert x[:, :, t].isnan().all(), name
        x, r = x[:, :, ~t], r[:, :, ~t]
        if r.numel() == 0:
            continue
        norm = ((x - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        assert norm <= (4e-3 if dtype == BF16 else 5e-4), (name, norm)  # (as in test_bias)


@pytest.mark.parametrize("shape,kernel,dtype", [
    ((5, 3, 17, 21, 32), (7, 7), BF16),     # the tiles' sums, more rows than threads of an entry, and a remainder
    ((1, 2, 9, 8, 64), (5, 5), F16),        # fewer rows than threads
    ((2, 2, 12, 13, 20), (5, 5), BF16),     # the general kernels: head_dim
    ((2, 2, 11, 14, 32), (3, 7), F16),      # ... rectangular windows
    ((1, 2, 10, 12, 32), (3, 3), torch.float32)])
def test_gradient_in_the_tensors_type(shape, kernel, dtype):
    # the native binding has the sums written in the tensors' type, the Python Function converts float32 ones
    ensure_built()
    from e_natten_amd import natten2d, ops
    print("case bias gradient", shape, kernel, dtype, flush=True)
    assert ops.NATIVE_BINDING
    q, k, v, g = (t.cuda() for t in make_inputs(shape, dtype, seed=3))
    rpb = torch.randn(shape[1], 2 * kernel[0] - 1, 2 * kernel[1] - 1, generator=torch.Generator().manual_seed(7)).to(dtype).cuda()
    scale = shape[-1] ** -0.5
    both = []
    for call in (lambda r: natten2d(q, k, v, kernel, scale, rpb=r),
                 lambda r: ops.Natten2dWindow.apply(q, k, v, r, kernel, (False, False), scale)):
        r = rpb.clone().requires_grad_(True)
        both.append(torch.autograd.grad(call(r), r, g)[0])
    assert both[0].dtype == dtype and torch.equal(*both)


@pytest.mark.parametrize("shape,ks,dtype", [
    ((70, 2, 8, 8, 32), 7, BF16),     # one tile to an image, more images than threads of an entry
    ((33, 3, 13, 9, 32), 5, F16),     # four
    ((2, 2, 64, 64, 32), 3, F16),     # as many as threads
    ((2, 1, 67, 65, 32), 3, BF16)])   # more
def test_sums_over_the_tiles_of_many_images(shape, ks, dtype):
    test_bias(shape, ks, dtype, "plain")
