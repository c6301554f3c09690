"""The float32 matrix-core backward, dV and dK in one launch and one after the other: every built head
dim and kernel size on images with partial tiles, and a workspace that is aligned to its floats only."""
import pytest
import torch

from _util import assert_close, ensure_built, make_inputs, oracle_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,ks,hw", [
    (32, 3, (19, 13)), (32, 5, (22, 30)), (32, 7, (33, 17)), (32, 7, (7, 9)), (64, 3, (16, 21)), (64, 5, (27, 20)),
    (64, 7, (18, 23)), (128, 3, (13, 18)), (128, 5, (21, 19)), (128, 7, (20, 15)),
    # both ends of an axis clamp the windows of one wave's keys
    (128, 5, (21, 12)), (32, 5, (12, 12)), (64, 5, (17, 11)), (32, 5, (11, 13)), (64, 7, (17, 14)), (32, 7, (14, 14)), (128, 7, (14, 14)), (32, 3, (6, 6))])
def test_backward(D, ks, hw):
    from e_natten_amd import _lib as L
    lib = ensure_built()
    B, N, (H, W) = 2, 3, hw
    print("case float32", D, ks, hw, flush=True)
    q, k, v, g = make_inputs((B, N, H, W, D), torch.float32, seed=D + ks, q_scale=D ** -0.5)
    qd, kd, vd, gd = (t.cuda() for t in (q, k, v, g))
    o, dq, dk, dv = (torch.full_like(qd, float("nan")) for _ in range(4))
    lse = torch.empty((B, N, H, W), device="cuda")
    ws = torch.full((lib.enatten2d_bwd_workspace_bytes(B, N, H, W, D, ks, L.F32) // 4 + 1,), float("nan"), device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    rc = lib.enatten2d_fwd(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), o.data_ptr(), lse.data_ptr(),
                           B, N, H, W, D, ks, L.F32, None, None, None, None, 1.0, st)
    assert rc == 0, L.last_error()
    rc = lib.enatten2d_bwd(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), o.data_ptr(), gd.data_ptr(), lse.data_ptr(),
                           dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr() + 4, B, N, H, W, D, ks, L.F32,
                           None, None, None, None, None, 1.0, st)
    assert rc == 0, L.last_error()
    torch.cuda.synchronize()
    ref = oracle_all(q, k, v, g, ks, small=True)
    assert_close((o.cpu(), dq.cpu(), dk.cpu(), dv.cpu()), (ref[0], ref[2], ref[3], ref[4]), torch.float32, "d%d k%d" % (D, ks))


@pytest.mark.parametrize("D,ks,hw", [
    # blocks of 2x2 pixels cut by the image's edge, windows clamped at one end and at both, axes of k .. 2k pixels
    (32, 3, (3, 5)), (64, 3, (6, 4)), (128, 3, (9, 11)), (32, 5, (5, 6)), (64, 5, (9, 10)), (128, 5, (10, 23)), (128, 5, (8, 8)),
    (32, 7, (13, 14)), (64, 7, (14, 31)), (128, 7, (7, 8)), (128, 7, (13, 22)), (64, 7, (25, 17))])
def test_views_of_one_projection(D, ks, hw):
    from e_natten_amd import kernel_path, natten2d
    ensure_built()
    assert kernel_path(D, ks, torch.float32) == "mfma"
    B, N, (H, W) = 2, 2, hw
    print("case float32 views", D, ks, hw, flush=True)
    q, k, v, g = make_inputs((B, N, H, W, D), torch.float32, seed=3 * D + ks, q_scale=D ** -0.5)
    x = torch.stack([t.permute(0, 2, 3, 1, 4) for t in (q, k, v)], dim=3).cuda().requires_grad_(True)  # [B, H, W, 3, N, D]
    up = g.permute(0, 2, 3, 1, 4).contiguous().cuda().permute(0, 3, 1, 2, 4)
    o = natten2d(*(t.movedim(3, 1) for t in x.unbind(3)), ks)
    o.backward(up)
    torch.cuda.synchronize()
    ref = oracle_all(q, k, v, g, ks, small=True)
    got = [x.grad[:, :, :, i].permute(0, 3, 1, 2, 4).cpu() for i in range(3)]
    assert_close((o.detach().cpu(), *got), (ref[0], ref[2], ref[3], ref[4]), torch.float32, "d%d k%d" % (D, ks))


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("ks", [3, 5, 7])
def test_infinite_results(D, ks):
    """Results that are infinite by the operator's arithmetic leave as the infinity, not as NaN.  (A query or key that shares a
    2x2 block with one that sees the value, but does not see it itself, may get NaN: its weight, zero, meets the infinity.)"""
    from e_natten_amd import natten2d
    ensure_built()
    print("case float32 infinities", D, ks, flush=True)
    H, W, r, c = 24, 24, 11, 11  # (windows and tiles away from the border)
    shape, inf = (1, 1, H, W, D), float("inf")
    near = torch.zeros(H, W, dtype=torch.bool)
    near[r - ks // 2:r + ks // 2 + 1, c - ks // 2:c + ks // 2 + 1] = True  # sees (r, c), and is seen from there

    def run(q, k, v, g):
        ins = [t.cuda().requires_grad_(True) for t in (q, k, v)]
        o = natten2d(*ins, ks)
        return [t.detach().cpu()[0, 0] for t in (o, *torch.autograd.grad(o, ins, g.cuda()))]

    # one infinite value, one infinite element of the upstream gradient
    q, k, v, g = make_inputs(shape, torch.float32, seed=D + ks, q_scale=D ** -0.5)
    plain = run(q, k, v, g)
    for sign in (1, -1):
        v2, g2 = v.clone(), g.clone()
        v2[0, 0, r, c, 5] = g2[0, 0, r, c, D - 3] = sign * inf
        o, dv = run(q, k, v2, g)[0], run(q, k, v, g2)[3]
        assert (o[near][:, 5] == sign * inf).all() and (dv[near][:, D - 3] == sign * inf).all()
        for got, ref, ch in ((o, plain[0], 5), (dv, plain[3], D - 3)):
            keep = torch.arange(D) != ch
            assert torch.equal(got[..., keep], ref[..., keep])
            assert got[..., ch][~near].isnan().sum() <= 2 * ks + 1 and torch.equal(
                got[..., ch][~near & ~got[..., ch].isnan()], ref[..., ch][~near & ~got[..., ch].isnan()])
    # finite inputs whose gradients overflow: all logits zero (q has channel 2 only, k channel 1), dP = 1e38 for one pair
    q, k, v, g = (torch.zeros(shape) for _ in range(4))
    q[0, 0, r, c, 2] = k[0, 0, r, c, 1] = 1e8
    v[0, 0, r, c, 0] = g[0, 0, r, c, 0] = 1e19
    got = run(q, k, v, g)
    ref = oracle_all(q, k, v, g, ks, small=True)
    ref = [ref[i][0, 0].float() for i in (0, 2, 3, 4)]  # (float64 until here)
    assert ref[1].isinf().sum() == 1 and ref[2].isinf().sum() == ks * ks
    for name, x, y in zip(("O", "dQ", "dK", "dV"), got, ref):
        assert torch.equal(x.isinf(), y.isinf()) and torch.equal(x[x.isinf()], y[y.isinf()]), name
        assert torch.allclose(x[x.isfinite()], y[x.isfinite()], rtol=1e-5, atol=0), name


@pytest.mark.parametrize("D,ks,hw", [(32, 3, (9, 10)), (64, 3, (12, 17)), (128, 5, (14, 11)), (32, 5, (10, 16)), (64, 7, (13, 19)), (128, 7, (15, 8))])
def test_one_infinite_gradient_anywhere(D, ks, hw):
    """An infinite element of the upstream gradient at every place of an image, one in a head: every key that its query sees
    has an infinite dV, and of the others none that is 4 or more pixels away from such a key has NaN (the blocks of keys of a
    wave are walked over the same queries)."""
    from e_natten_amd import natten2d
    ensure_built()
    print("case float32 infinity anywhere", D, ks, hw, flush=True)
    H, W = hw
    n = H * W
    one = torch.arange(n)
    q, k, v, g = (t.expand(1, n, H, W, D).contiguous() for t in make_inputs((1, 1, H, W, D), torch.float32, seed=D + ks, q_scale=D ** -0.5))
    g.view(n, n, D)[one, one, 7] = float("inf")
    ins = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    dv = torch.autograd.grad(natten2d(*ins, ks), ins, g.cuda())[2].cpu()[0, ..., 7]
    first = lambda i, L: min(max(i - ks // 2, 0), L - ks)
    for at in range(n):
        r, c = first(at // W, H), first(at % W, W)
        assert (dv[at, r:r + ks, c:c + ks] == float("inf")).all(), (at // W, at % W)
        far = torch.ones(H, W, dtype=torch.bool)
        far[max(r - 3, 0):r + ks + 3, max(c - 3, 0):c + ks + 3] = False
        assert dv[at][far].isfinite().all(), (at // W, at % W)


@pytest.mark.parametrize("ks,W,D", [(3, 65536, 32), (3, 65537, 32), (5, 65600, 64), (7, 70001, 32), (3, 70001, 128)])
def test_wide_images(ks, W, D):
    """Images on both sides of the width from which the dK/dV pass has 64-bit places: views of [.., W, H, D] tensors, whose
    strides between rows and columns are both small.  Every width is on the matrix-core kernels."""
    from e_natten_amd import natten2d
    lib = ensure_built()
    print("case float32 wide", ks, W, D, flush=True)
    q, k, v, g = make_inputs((1, 1, ks + 1, W, D), torch.float32, seed=W, q_scale=D ** -0.5)
    swap = lambda t: t.transpose(2, 3).contiguous().cuda().transpose(2, 3)
    ins = [swap(t).requires_grad_(True) for t in (q, k, v)]
    lib.enatten_profile_enable(1)
    o = natten2d(*ins, ks)
    got = [t.detach().cpu() for t in (o, *torch.autograd.grad(o, ins, swap(g)))]
    lib.enatten_profile_enable(0)
    names = [lib.enatten_profile_kernel_name(i) for i in range(3)]
    assert names == [b"fwd_mfma_f32", b"bwd_dq_mfma_f32", b"bwd_dkdv_mfma_f32"], names
    ref = oracle_all(q, k, v, g, ks)
    assert_close(got, (ref[0], *ref[2:]), torch.float32, "d%d k%d W %d" % (D, ks, W))
