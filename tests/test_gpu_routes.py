"""Calls that the kernels for causal, long, dilated, biased and small calls take, against the general
kernels, over the orders, strides, types and sizes that they accept or have to leave to others."""
import random

import pytest
import torch

from _util import ensure_built

pytestmark = pytest.mark.gpu
LAYOUTS = ("plain", "proj", "one batch", "one head", "off by 4", "off by 8", "axes swapped", "channels first")


def _tensor(shape, dtype, layout, gen):
    """N(0, 1) values; whatever the layout, a tensor of the given shape on the GPU."""
    B, N, *ext, d = shape
    new = lambda *s: torch.randn(s, generator=gen, device="cuda", dtype=dtype)
    if layout == "proj":
        return new(B, *ext, 3, N, d).unbind(len(ext) + 1)[1].movedim(len(ext) + 1, 1)
    if layout == "one batch":
        return new(1, N, *ext, d).expand(shape)
    if layout == "one head":
        return new(B, 1, *ext, d).expand(shape)
    if layout.startswith("off"):
        by = int(layout[-1])
        return new(B, N, *ext, d + by)[..., by:]
    if layout == "axes swapped":
        return new(B, N, *ext[::-1], d).movedim(-2, 2) if len(ext) == 2 else new(B, *ext, N, d).movedim(-2, 1)
    if layout == "channels first":
        return new(B, N, d, *ext).movedim(2, -1)
    return new(*shape)


def _draw(kind, rng):
    """(shape, call of q, k, v, rpb, kernel_size if there is a bias)"""
    from e_natten_amd import natten1d, natten2d
    d = rng.choice((8, 16, 24, 32, 32, 40, 48, 64, 64, 72, 96, 128, 128, 20, 136))
    scale = d ** -0.5
    if kind in ("causal", "long"):
        T = max(60 if kind == "long" else 1, int(2 ** rng.uniform(4, 10.5)))
        k = min(T, int(2 ** rng.uniform(1, 8.5))) if kind == "causal" else rng.randrange(51, min(T, 401) + 1, 2)
        shape = (rng.randint(1, 4), rng.randint(1, 6), T, d)
        return shape, lambda q, k_, v, r: natten1d(q, k_, v, k, scale, 1, kind == "causal"), None, "k=%d" % k
    k, dil = rng.choice((3, 5, 7, 7, 9, 11, 13)), rng.randint(2, 5) if kind == "dilated" else 1
    side = lambda: rng.randint(k, max(k, 16)) if kind == "small" else rng.randint(k * dil, max(k * dil + 1, min(3 * k * dil, 90)))
    images = (rng.randint(8, 16), rng.randint(8, 24)) if kind == "small" else (rng.randint(1, 3), rng.randint(1, 6))
    return ((*images, side(), side(), d), lambda q, k_, v, r: natten2d(q, k_, v, k, scale, dil, rpb=r),
            k if kind == "bias" else None, "k=%d dilation=%d" % (k, dil))


@pytest.mark.parametrize("kind", ["causal", "long", "dilated", "bias", "small"])
def test_against_the_general_kernels(kind):
    from e_natten_amd import _lib
    lib = ensure_built()
    rng = random.Random(kind)
    for it in range(24):
        dtype = rng.choice((torch.bfloat16, torch.float16))
        shape, f, bias, what = _draw(kind, rng)
        layouts = [rng.choice(LAYOUTS) for _ in range(4)]
        gen = torch.Generator(device="cuda").manual_seed(it)
        q, k, v, g = (_tensor(shape, dtype, l, gen) for l in layouts)
        if it % 3 == 0:  # (a common component of keys and values)
            k, v = k + 1.5, v + 1.5
        ins = [t.detach().requires_grad_(True) for t in (q, k, v)]
        if bias:
            ins.append(torch.randn((shape[1], 2 * bias - 1, 2 * bias - 1), generator=gen, device="cuda",
                                   dtype=dtype).requires_grad_(True))
        print("case", kind, it, shape, dtype, what, layouts, flush=True)
        res = []
        for path in (0, _lib.PATH_SIMT):
            lib.enatten_set_path(path)
            try:
                o = f(*ins[:3], ins[3] if bias else None)
                res.append([t.detach().double() for t in (o, *torch.autograd.grad(o, ins, g))])
            finally:
                lib.enatten_set_path(0)
        # A rounding of a whole tensor is 1.7e-3 of it in 2-norm (float16: an eighth).  Causal, long and
        # biased calls carry P and dS to 16 bits and more: at most some results are rounded the other way.
        # Dilated and small ones round P and dS once, under keys of rms 1.8 (sqrt(2 * 3.2) * 1.7e-3 = 4.3e-3)
        # and round the results, on both sides
        bound = 8e-3 if kind in ("dilated", "small") else 1.7e-3
        for name, a, b in zip(("O", "dQ", "dK", "dV", "dRPB"), *res):
            norm = ((a - b).norm() / b.norm()).item()
            assert norm <= (bound if dtype == torch.bfloat16 else bound / 8), (name, norm)
