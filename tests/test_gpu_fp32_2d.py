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
