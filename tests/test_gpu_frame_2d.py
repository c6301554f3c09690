"""The border (frame) tiles of the dK/dV pass: many images whose tiles are counted from another start
in each, blocks of queries of every width, and head dims below 64 with the largest windows."""
import pytest
import torch

from _util import O, assert_close, ensure_built, make_inputs, oracle_all, run_capi, run_gpu

pytestmark = pytest.mark.gpu
BF, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("shape,ks,dtype", [
    ((7, 9, 26, 26, 64), 9, BF),     # 16 tiles per image, 64 workgroups per XCD: whole images apart
    ((5, 7, 28, 28, 64), 13, F16),   # the same with two waves per block of keys
    ((3, 50, 24, 17, 32), 3, BF),    # 9 tiles per image
    ((1, 3, 61, 43, 64), 7, BF),     # inner tiles too; 11 and 14 queries side by side
    ((1, 2, 37, 50, 32), 5, F16), ((1, 2, 35, 27, 128), 11, BF), ((2, 1, 41, 29, 96), 9, F16),
])
def test_border_tiles(shape, ks, dtype):
    ensure_built()
    print("case border", shape, dtype, "k=%d" % ks, flush=True)
    q, k, v, g = make_inputs(shape, dtype, seed=7)
    o, _, dq, dk, dv = run_capi(q, k, v, g, ks, shape[-1] ** -0.5)
    ref = oracle_all(q, k, v, g, ks, shape[-1] ** -0.5)
    assert_close((o, dq, dk, dv), (ref[0], ref[2], ref[3], ref[4]), dtype, "border k%d" % ks)


@pytest.mark.parametrize("hw,ks,D", [((19, 21), 5, 64), ((26, 23), 9, 64), ((29, 30), 7, 32), ((31, 27), 13, 64)])
def test_logits_far_below_zero(hw, ks, D):
    # all logits near -300: exp(0 - lse) overflows, so what stands beside a rectangle's queries must not count
    ensure_built()
    print("case far below zero", hw, ks, D, flush=True)
    q, k, v, g = make_inputs((1, 2, *hw, D), BF, seed=11)
    q, k = (1 + 0.02 * q.float()).to(BF), (-300 / D + 0.02 * k.float()).to(BF)
    got = run_gpu(q, k, v, g, ks)
    ref = oracle_all(q, k, v, g, ks, small=True)
    assert all(torch.isfinite(t.float()).all() for t in got)
    # (dS of nearly equal keys cancel in dQ, and of nearly equal queries in dK: 16-bit weights say little there)
    for x, r in ((got[0], ref[0]), (got[3], ref[4])):
        assert O.rel_err(x, r) <= 2e-2


@pytest.mark.parametrize("which", ["dO", "q"])
@pytest.mark.parametrize("hw,D,ks,dtype", [
    ((26, 23), 64, 7, BF), ((26, 21), 48, 3, BF), ((30, 27), 64, 11, F16), ((22, 23), 128, 3, F16), ((27, 25), 96, 7, BF),
    ((25, 27), 128, 11, BF)])
def test_values_that_are_not_finite_stay_in_their_blocks_of_keys(hw, D, ks, dtype, which):
    """A NaN in one query, another one in each head: dK and dV of the 4x4 blocks of keys that its window
    does not meet are finite, though the query may stand right beside those that a block's waves walk."""
    ensure_built()
    print("case one query not finite", which, hw, D, ks, flush=True)
    (H, W), heads, row = hw, 16, 9
    q, k, v, g = make_inputs((1, heads, H, W, D), dtype, seed=23)
    for h in range(heads):
        {"dO": g, "q": q}[which][0, h, row, 4 + h] = float("nan")
    _, _, dk, dv = run_gpu(q, k, v, g, ks, D ** -0.5)
    for h in range(heads):
        keys = O.neighbour_mask(H, W, ks)[row * W + 4 + h].reshape(H, W)
        blocks = torch.nn.functional.max_pool2d(keys.float()[None], 4, ceil_mode=True)[0] > 0
        blocks = blocks.repeat_interleave(4, 0).repeat_interleave(4, 1)[:H, :W]
        for name, x in (("dK", dk), ("dV", dv)):
            nan = ~x[0, h].float().isfinite().all(-1)
            assert nan[keys].all(), (name, h)
            assert not (nan & ~blocks).any(), (name, h, (nan & ~blocks).nonzero().tolist())


@pytest.mark.parametrize("D,ks,hw,dtype", [
    (40, 11, (43, 38), BF), (48, 13, (50, 44), BF), (56, 13, (13, 28), F16), (48, 11, (24, 120), F16)])
def test_largest_windows_below_head_dim_64(D, ks, hw, dtype):
    """The second part's sums lie over rows whose channels from D on have to be zero for the next tile:
    a workgroup has several tiles here."""
    from e_natten_amd import natten2d
    ensure_built()
    B, N = (6, 8) if hw[0] * hw[1] < 2000 else (4, 8)
    print("case below 64", D, ks, hw, dtype, flush=True)
    q, k, v, g = make_inputs((B, N, *hw, D), dtype, seed=D)
    k, v = k + 2, v + 2  # (means that cancel in dQ and dS, which rounded weights would show)
    scale = D ** -0.5
    ref = oracle_all(q, k, v, g, ks, scale)
    for x, r in zip(run_gpu(q, k, v, g, ks, scale), (ref[0], *ref[2:])):
        # the rounding of the results, 2^-9 or 2^-12 of an element at most, and no more: no 16-bit weights
        assert ((x.double() - r.double()).norm() / r.double().norm()).item() <= (2.0 ** -9 if dtype == BF else 2.0 ** -12)
    # views of a projection, and the sub-grids of a dilated call: the same values at twice the distance
    if min(hw) < 2 * ks:
        return
    x = torch.stack([t.permute(0, 2, 3, 1, 4) for t in (q, k, v)], dim=3).cuda()
    qg, kg, vg = (t.permute(0, 3, 1, 2, 4).requires_grad_(True) for t in x.unbind(3))
    gg = g.cuda()
    grads = torch.autograd.grad(natten2d(qg, kg, vg, ks, scale, 2), (qg, kg, vg), gg)
    for r in range(2):
        for c in range(2):
            at = (slice(None), slice(None), slice(r, None, 2), slice(c, None, 2))
            sub = [t.detach()[at].contiguous().requires_grad_(True) for t in (qg, kg, vg)]
            want = torch.autograd.grad(natten2d(*sub, ks, scale), sub, gg[at].contiguous())
            assert all(torch.equal(a[at], b) for a, b in zip(grads, want))


@pytest.mark.parametrize("shape,dtype", [
    ((8, 8, 32, 32), BF), ((1, 41, 40, 40), BF), ((1, 41, 40, 40), F16),  # 1024 and 1025 tiles: the build for three waves, and for four
    ((1, 45, 37, 43), F16), ((2, 1, 166, 252), BF)])                     # ... cut tiles, nearly all tiles inner
def test_four_waves_at_head_dim_32(shape, dtype):
    ensure_built()
    shape = (*shape, 32)
    print("case four waves", shape, dtype, flush=True)
    q, k, v, g = make_inputs(shape, dtype, seed=5)
    o, _, dq, dk, dv = run_capi(q, k, v, g, 5, 32 ** -0.5)
    ref = oracle_all(q, k, v, g, 5, 32 ** -0.5)
    assert_close((o, dq, dk, dv), (ref[0], ref[2], ref[3], ref[4]), dtype, "four waves")
