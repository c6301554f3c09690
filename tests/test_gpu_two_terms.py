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
