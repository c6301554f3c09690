"""Head dims between 32 and 64 with 11x11 and 13x13 windows: probabilities and dS in two 16-bit terms where the
general kernels have float32."""
import pytest
import torch

from _util import O, ensure_built, make_inputs
from test_gpu_bias_2d import NAMES, _dense, _rpb

pytestmark = pytest.mark.gpu
BF, F16 = torch.bfloat16, torch.float16


def _both(q, k, v, g, rpb, ks, scale):
    """(O, dQ, dK, dV[, dRPB]) of the kernels and of float64; rpb: a table or None."""
    from e_natten_amd import natten2d
    x = [t for t in (q, k, v, rpb) if t is not None]
    xg = [t.cuda().requires_grad_(True) for t in x]
    o = natten2d(*xg[:3], ks, scale, rpb=None if rpb is None else xg[3])
    got = [t.detach().cpu().double() for t in (o, *torch.autograd.grad(o, xg, g.cuda()))]
    xr = [t.double().requires_grad_(True) for t in x]
    table = torch.zeros(q.shape[1], 2 * ks - 1, 2 * ks - 1, dtype=torch.double) if rpb is None else xr[3]
    o_ref = _dense(*xr[:3], table, ks, scale)
    return got, [t.detach() for t in (o_ref, *torch.autograd.grad(o_ref, xr, g.double()))]


@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("D,ks,hw,dtype", [(40, 13, (27, 30), BF), (48, 11, (32, 29), BF), (56, 11, (26, 37), F16),
                                           (48, 13, (32, 32), F16)])
def test_common_components_cancel(D, ks, hw, dtype, biased):
    # keys and values far from zero: a window's dS sum to zero, and what they fall short of that reaches dQ 32 times.
    # Besides the rounding of the results there is what float32 leaves of dO . V of some 1e4 (2^-10 in 1e2, the
    # deviation): 1% of float16's rounding
    ensure_built()
    print("case common components", D, ks, hw, dtype, biased, flush=True)
    q, k, v, g = make_inputs((1, 2, *hw, D), torch.float32, seed=D + ks)
    q, k, v, g = q.to(dtype), (k + 32).to(dtype), (v + 32).to(dtype), (g + 8).to(dtype)
    got, ref = _both(q, k, v, g, _rpb(2, ks).to(dtype) if biased else None, ks, D ** -0.5)
    for name, x, r in list(zip(NAMES, got, ref))[:4]:
        norm = ((x - r).norm() / r.norm()).item()
        rounding = ((r.to(dtype).double() - r).norm() / r.norm()).item()
        print("   ", name, "2-norm %.2e, of the result's rounding alone %.2e" % (norm, rounding), flush=True)
        assert norm <= 1.02 * rounding, (name, norm, rounding)


@pytest.mark.parametrize("which", ["q", "k", "v", "dO"])
@pytest.mark.parametrize("D,ks,hw,dtype", [
    (48, 11, (43, 38), BF), (40, 13, (44, 44), F16),   # inner tiles and border
    (40, 13, (20, 27), BF), (56, 11, (19, 24), F16),   # border tiles only
])
def test_values_that_are_not_finite_stay_in_their_windows(D, ks, hw, dtype, which):
    """A NaN in one pixel, without a bias: what its windows connect with it is NaN, all else as without it."""
    ensure_built()
    print("case not finite", which, D, ks, hw, dtype, flush=True)
    H, W = hw
    at = (H // 2) * W + 9
    scale = D ** -0.5
    q, k, v, g = make_inputs((1, 2, H, W, D), dtype, seed=31)
    clean, _ = _both(q, k, v, g, None, ks, scale)
    {"q": q, "k": k, "v": v, "dO": g}[which].flatten(2, 3)[:, :, at] = float("nan")
    got, _ = _both(q, k, v, g, None, ks, scale)
    mask = O.neighbour_mask(H, W, ks)
    only = torch.zeros(H * W, dtype=torch.bool)
    only[at] = True
    queries = only if which in ("q", "dO") else mask[:, at]   # queries with a gradient that is touched
    keys = mask[queries].any(0)                               # the keys that these see
    none = torch.zeros_like(only)
    touched = (none if which == "dO" else queries, queries, keys, none if which == "v" else keys)
    for name, x, c, t in zip(NAMES, got, clean, touched):
        x, c = x.flatten(2, 3), c.flatten(2, 3)
        assert x[:, :, t].isnan().all(), name
        x, c = x[:, :, ~t], c[:, :, ~t]
        if c.numel() == 0:
            continue
        # (keys and queries beside the NaN are summed again, in another order and in float32: the rounding of results)
        norm = ((x - c).norm() / c.norm()).item()
        print("   ", name, "2-norm %.2e" % norm, flush=True)
        assert norm <= (2.0 ** -9 if dtype == BF else 2.0 ** -12), (name, norm)
