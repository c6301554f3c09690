"""1D windows of any length on the matrix cores, causal and centred, against the dense-mask oracle."""
import pytest
import torch

from _util import BF16_REL, O, ensure_built, make_inputs

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("shape,ks,causal,dtype,layout", [
    ((1, 2, 65, 32), 2, True, BF16, "plain"),      # smallest window with a gradient (on the general kernels)
    ((2, 1, 64, 64), 64, True, F16, "plain"),      # plain causal attention of one tile
    ((1, 3, 200, 128), 33, True, BF16, "proj"),    # band edges inside the steps of 32 keys
    ((1, 2, 300, 128), 300, True, F16, "plain"),   # window = sequence
    ((2, 2, 131, 40), 16, True, BF16, "proj"),     # head_dim below a built one
    ((1, 2, 17, 8), 5, True, F16, "plain"),        # shorter than one step of keys
    ((4, 128, 130, 32), 70, True, BF16, "plain"),  # more tiles than workgroups at a time, the last one cut
    ((4, 128, 200, 128), 100, True, F16, "proj"),
    ((2, 90, 330, 128), 256, True, F16, "plain"),  # two groups of queries per wave in the forward, the last tile cut
    ((2, 90, 330, 128), 257, False, BF16, "proj"),
    ((2, 90, 310, 128), 300, True, BF16, "proj"),  # ... its second group of some waves past the end
    ((1, 2, 257, 64), 51, False, BF16, "proj"),    # centred: clamped windows at both ends
    ((2, 1, 129, 128), 129, False, F16, "plain"),  # window = sequence: plain attention
    ((8, 64, 160, 64), 97, False, BF16, "plain"),  # more tiles than workgroups at a time
    # the smallest windows of every head_dim: on the general kernels below these, in the backward or both
    ((1, 2, 140, 64), 2, True, F16, "proj"),
    ((1, 2, 140, 48), 5, True, BF16, "plain"),     # only the backward here
    ((1, 2, 140, 48), 6, True, BF16, "proj"),
    ((1, 2, 140, 56), 2, True, F16, "plain"),      # neither
    ((1, 2, 140, 32), 4, True, BF16, "plain"),
    ((1, 2, 140, 32), 3, True, F16, "proj"),       # neither
    ((1, 2, 140, 24), 8, True, BF16, "proj"),
    ((1, 2, 140, 16), 6, True, F16, "plain"),      # only the forward here
    ((1, 2, 140, 8), 12, True, BF16, "proj"),
])
def test_band_windows(shape, ks, causal, dtype, layout):
    ensure_built()
    from e_natten_amd import natten1d
    print("case band", shape, dtype, "k=%d" % ks, "causal" if causal else "centred", layout, flush=True)
    q, k, v, g = make_inputs(shape, dtype, seed=31)
    scale = shape[-1] ** -0.5
    if layout == "proj":
        qkv = torch.stack([t.permute(0, 2, 1, 3) for t in (q, k, v)], dim=2).cuda()
        qg, kg, vg = (t.permute(0, 2, 1, 3).requires_grad_(True) for t in qkv.unbind(2))
    else:
        qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = natten1d(qg, kg, vg, ks, scale, 1, causal)
    got = (o, *torch.autograd.grad(o, (qg, kg, vg), g.cuda()))
    # (a sample of the heads: every head is the same computation on other data)
    heads = slice(0, None, max(1, shape[1] // 4))
    qr, kr, vr = (t[-1:, heads].double().requires_grad_(True) for t in (q, k, v))
    o_ref = O.natten2d_window_dense_mask(qr.unsqueeze(2), kr.unsqueeze(2), vr.unsqueeze(2), (1, ks),
                                         (False, causal), scale).squeeze(2)
    ref = (o_ref.detach(), *torch.autograd.grad(o_ref, (qr, kr, vr), g[-1:, heads].double()))
    for name, x, r in zip(("O", "dQ", "dK", "dV"), got, ref):
        x = x.detach()[-1:, heads].cpu()
        err = O.rel_err(x, r)
        # P and dS are carried to 16 bits or more: what is left is the rounding of the results
        # (2^-9 of an element for bfloat16, 2^-12 for float16) and of O in delta
        norm = ((x.double() - r).norm() / r.norm()).item()
        print("   ", name, "max-abs / max %.2e" % err, "2-norm %.2e" % norm, flush=True)
        assert err <= BF16_REL, (name, err)
        assert norm <= (4e-3 if dtype == BF16 else 5e-4), (name, norm)
    assert torch.equal(o, natten1d(qg, kg, vg, ks, scale, 1, causal))


@pytest.mark.parametrize("shape,ks,causal,dtype", [
    ((1, 64, 500, 128), 90, True, BF16),    # 512 tiles: blocks of 64 keys
    ((1, 57, 560, 128), 90, True, BF16),    # 513: blocks of 32
    ((1, 57, 513, 128), 31, False, F16),    # ... a last tile of one query
    ((1, 57, 560, 72), 33, True, F16),
    ((1, 64, 500, 72), 33, True, F16),
    ((2, 52, 600, 128), 511, True, F16),
    ((2, 52, 600, 128), 512, True, F16),    # two groups of queries per wave
    ((2, 52, 577, 128), 513, False, BF16),  # ... the second group of the last tile past the end
])
def test_blocks_of_the_forward(shape, ks, causal, dtype):
    ensure_built()
    from e_natten_amd import natten1d
    print("case blocks", shape, dtype, "k=%d" % ks, flush=True)
    q, k, v, _ = make_inputs(shape, dtype, seed=37)
    scale = shape[-1] ** -0.5
    o = natten1d(q.cuda(), k.cuda(), v.cuda(), ks, scale, 1, causal)[-1:, ::16].cpu()
    qr, kr, vr = (t[-1:, ::16].double().unsqueeze(2) for t in (q, k, v))
    ref = O.natten2d_window_dense_mask(qr, kr, vr, (1, ks), (False, causal), scale).squeeze(2)
    norm = ((o.double() - ref).norm() / ref.norm()).item()
    print("    O 2-norm %.2e" % norm, flush=True)
    assert norm <= (4e-3 if dtype == BF16 else 5e-4), norm  # (as in test_band_windows)


@pytest.mark.parametrize("ks,causal,d,dtype", [(33, True, 64, BF16), (51, False, 128, F16), (70, True, 40, F16)])
def test_values_that_are_not_finite_stay_in_their_windows(ks, causal, d, dtype):
    # a NaN in v at one position: only queries that see it, and the keys that such queries see, may
    # be touched (in a causal sequence nothing before it), though rows outside a window are staged
    ensure_built()
    from e_natten_amd import natten1d
    print("case not finite", ks, causal, d, dtype, flush=True)
    T, pos, scale = 260, 140, d ** -0.5
    q, k, v, g = make_inputs((1, 2, T, d), dtype, seed=41)
    qr, kr, vr = (t.double().requires_grad_(True) for t in (q, k, v))
    o_ref = O.natten2d_window_dense_mask(qr.unsqueeze(2), kr.unsqueeze(2), vr.unsqueeze(2), (1, ks),
                                         (False, causal), scale).squeeze(2)
    ref = (o_ref.detach(), *torch.autograd.grad(o_ref, (qr, kr, vr), g.double()))
    vbad = v.clone()
    vbad[:, :, pos] = float("nan")
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, vbad))
    o = natten1d(qg, kg, vg, ks, scale, 1, causal)
    got = [t.detach().cpu() for t in (o, *torch.autograd.grad(o, (qg, kg, vg), g.cuda()))]
    start = lambda t: max(0, t - ks + 1) if causal else min(max(t - ks // 2, 0), T - ks)
    windows = [range(start(t), t + 1 if causal else start(t) + ks) for t in range(T)]
    sees = torch.tensor([pos in w for w in windows])
    reached = torch.zeros(T, dtype=torch.bool)
    for w in (w for w in windows if pos in w):
        reached[w.start:w.stop] = True
    assert got[0][:, :, sees].isnan().all() and got[1][:, :, sees].isnan().all()
    assert got[2][:, :, reached].isnan().all()
    for name, x, r, touched in zip(("O", "dQ", "dK", "dV"), got, ref,
                                   (sees, sees, reached, torch.zeros(T, dtype=torch.bool))):
        x, r = x[:, :, ~touched].double(), r[:, :, ~touched]
        norm = ((x - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        assert norm <= (4e-3 if dtype == BF16 else 5e-4), (name, norm)  # (as in test_band_windows)


def test_gradients_of_logits_beyond_float16():
    # dS of some 1e5, whose 16-bit terms would be an infinity and its negative, under a small
    # softmax scale: the gradients of q and k themselves are in range
    ensure_built()
    from e_natten_amd import natten1d
    q, k, v, g = make_inputs((1, 2, 130, 64), F16, seed=43)
    v, g, scale = v * 200, g * 200, 2.0 ** -10
    qr, kr, vr = (t.double().requires_grad_(True) for t in (q, k, v))
    o_ref = O.natten2d_window_dense_mask(qr.unsqueeze(2), kr.unsqueeze(2), vr.unsqueeze(2), (1, 3),
                                         (False, True), scale).squeeze(2)
    ref = torch.autograd.grad(o_ref, (qr, kr, vr), g.double())
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    got = torch.autograd.grad(natten1d(qg, kg, vg, 3, scale, 1, True), (qg, kg, vg), g.cuda())
    for name, x, r in zip(("dQ", "dK", "dV"), got, ref):
        norm = ((x.cpu().double() - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        assert norm <= 5e-4, (name, norm)  # (as in test_band_windows)


def _against_oracle(x, ks, causal, scale):
    """(O, dQ, dK, dV) of the kernels and of the dense-mask oracle; x = (q, k, v, dO)."""
    from e_natten_amd import natten1d
    xg = [t.cuda().requires_grad_(True) for t in x[:3]]
    o = natten1d(*xg, ks, scale, 1, causal)
    got = [t.detach().cpu().double() for t in (o, *torch.autograd.grad(o, xg, x[3].cuda()))]
    xr = [t.double().requires_grad_(True) for t in x[:3]]
    o_ref = O.natten2d_window_dense_mask(*(t.unsqueeze(2) for t in xr), (1, ks), (False, causal), scale).squeeze(2)
    return got, (o_ref.detach(), *torch.autograd.grad(o_ref, xr, x[3].double()))


@pytest.mark.parametrize("shape,ks,causal,dtype", [
    ((1, 2, 300, 64), 128, True, BF16),
    ((1, 2, 300, 128), 101, False, F16),
    ((2, 1, 200, 40), 5, True, F16),
    ((1, 2, 260, 32), 70, True, BF16),
])
def test_keys_and_values_with_a_common_component(shape, ks, causal, dtype):
    # dP is then large against its spread over a window, and an error of delta, which the whole
    # window shares, is multiplied by the common component of the keys
    ensure_built()
    print("case common component", shape, ks, causal, dtype, flush=True)
    q, k, v, g = make_inputs(shape, torch.float32, seed=53)
    got, ref = _against_oracle([t.to(dtype) for t in (q, k + 2, v + 2, g)], ks, causal, shape[-1] ** -0.5)
    for name, x, r in zip(("O", "dQ", "dK", "dV"), got, ref):
        norm = ((x - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        assert norm <= (4e-3 if dtype == BF16 else 5e-4), (name, norm)  # (as in test_band_windows)


@pytest.mark.parametrize("shape,ks", [((1, 2, 600, 64), 128), ((1, 2, 400, 128), 300), ((1, 2, 200, 32), 5)])
def test_float16_with_small_upstream_gradients(shape, ks):
    # dS of 1e-6 and less, which two float16 terms alone do not hold
    ensure_built()
    print("case small gradients", shape, ks, flush=True)
    q, k, v, g = make_inputs(shape, torch.float32, seed=59)
    got, ref = _against_oracle([t.to(F16) for t in (q, k, v, g * 1e-4)], ks, True, shape[-1] ** -0.5)
    for name, x, r in zip(("dQ", "dK", "dV"), got[1:], ref[1:]):
        norm = ((x - r).norm() / r.norm()).item()
        rounding = ((r.to(F16).double() - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e, of the result's rounding alone %.2e" % (norm, rounding), flush=True)
        assert norm <= 1.05 * rounding, (name, norm, rounding)


@pytest.mark.parametrize("dtype,size", [(BF16, 1e16), (F16, 4096.0)])
def test_logits_far_from_zero(dtype, size):
    # logits of -1e32 (float16: -1.7e7) that are equal over a window: the probabilities are uniform
    ensure_built()
    q, k, v, g = make_inputs((1, 2, 150, 64), dtype, seed=61)
    q, k = torch.zeros_like(q), torch.zeros_like(k)
    q[..., 0], k[..., 0] = size, -size
    from e_natten_amd import natten1d
    x = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    o = natten1d(*x, 40, 1.0, 1, True)
    dv = torch.autograd.grad(o, x, g.cuda())[2]
    p = O.axis_window_mask(150, 40, True).double()
    p = p / p.sum(1, keepdim=True)
    for name, got, r in (("O", o, p @ v.double()), ("dV", dv, p.T @ g.double())):
        norm = ((got.detach().cpu().double() - r).norm() / r.norm()).item()
        print("   ", name, dtype, "2-norm %.2e" % norm, flush=True)
        assert norm <= (4e-3 if dtype == BF16 else 5e-4), (name, norm)  # (as in test_band_windows)


@pytest.mark.parametrize("shape,ks,causal,dtype,layout", [
    ((2, 52, 600, 128), 512, True, F16, "plain"),   # the second group of the last tile cut
    ((2, 52, 577, 128), 513, False, BF16, "proj"),  # ... past the end, but for one query
    ((2, 52, 640, 128), 600, True, BF16, "proj"),   # whole tiles
])
def test_two_groups_of_queries(shape, ks, causal, dtype, layout):
    # two groups of queries per wave in the forward, from 512 keys on: the gradients need its log-sum-exp as well (windows of 256 to
    # 300 keys, above, are walked with one group in blocks of 32 keys)
    test_band_windows(shape, ks, causal, dtype, layout)


@pytest.mark.parametrize("shape,ks,causal,dtype,layout", [
    ((4, 24, 512, 48), 33, True, F16, "plain"),    # 768 tiles: no budget of four waves per SIMD in the dK/dV pass
    ((1, 71, 700, 48), 101, False, F16, "proj"),   # 781: four
    ((4, 24, 449, 40), 20, True, F16, "proj"),     # 768, the last of a sequence with one key
])
def test_tiles_of_the_key_pass(shape, ks, causal, dtype, layout):
    test_band_windows(shape, ks, causal, dtype, layout)
