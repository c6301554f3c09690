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
