"""The order of the border tiles (csrc/frame_order.h), compiled for the CPU: every tile once, and no
workgroup of the dK/dV pass is given more work than in the plain order."""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

from _util import ROOT

SOURCE = """#include "frame_order.h"
extern "C" int order(int n, int per_img, int step, int plain, int *image, int *place) {
    const enatten::FrameOrder o = plain ? enatten::FrameOrder{0, 1} : enatten::frame_order(per_img, step, n);
    for (int t = 0; t < n; t++) {
        const enatten::FramePlace p = enatten::frame_place(t, per_img, o);
        image[t] = p.image;
        place[t] = p.place;
    }
    return o.turn;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "order.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "e_natten_amd", "csrc"),
                           str(d / "order.cpp"), "-o", str(d / "order.so")])
    return ctypes.CDLL(str(d / "order.so"))


def walk(lib, n, per_img, step, plain=False):
    """(turn, image of each tile, its place)"""
    image, place = np.empty(n, np.int32), np.empty(n, np.int32)
    turn = lib.order(n, per_img, step, int(plain), *(x.ctypes.data_as(ctypes.c_void_p) for x in (image, place)))
    return turn, image, place


@pytest.mark.parametrize("per_img", [1, 2, 3, 4, 9, 15, 16, 24, 25, 60, 64, 128, 240, 4096, 4097])
def test_every_tile_once(lib, per_img):
    for step in (1, 5, 7, 32, 45, 64, 96, 120, per_img // 2 or 1, per_img, 2 * per_img):
        n = (200 * step // per_img + 2) * per_img
        _, image, place = walk(lib, n, per_img, step)
        assert (image == np.arange(n) // per_img).all() and place.min() >= 0
        assert np.array_equal(np.sort(image.astype(np.int64) * per_img + place), np.arange(n)), (per_img, step)


def spans(L, k, side):
    """Per tile of one axis: (length of the longest run of queries that one 4-key part has) by block."""
    out = []
    for r0 in range(0, L, 8):
        lo = lambda i: 0 if i < k else i - k // 2
        hi = lambda i: L if i >= L - k else i + k // 2 + 1
        blocks = []
        for b in range(lo(r0), hi(min(r0 + 8, L) - 1), side):
            blocks.append([max(0, min(hi(min(w + 4, L) - 1), b + side) - max(lo(w), b)) for w in (r0, r0 + 4) if w < L])
        out.append(blocks)
    return out


def frame_costs(H, W, k, side, parts):
    """Cost of each border tile in the numbering of frame_tile: 2 per block of queries and 1 per step of the
    block's busiest wave."""
    rows, cols = spans(H, k, side), spans(W, k, side)
    first = (k + 7) // 8
    ni_r, ni_c = (H - k) // 8 - first, (W - k) // 8 - first
    inner = lambda r, c: ni_r > 0 and ni_c > 0 and first <= r < first + ni_r and first <= c < first + ni_c
    return np.array([sum(2 + max(-(-p * -(-q // 4) // (8 * parts)) for p in a for q in b) for a in rows[r] for b in cols[c])
                     for r in range(len(rows)) for c in range(len(cols)) if not inner(r, c)]), max(ni_r, 0) * max(ni_c, 0)


def busiest(costs, place, step):
    """The dearest walk: each of 8 runs of tiles is dealt out with stride `step`."""
    per = -(-len(place) // 8)
    return max(costs[place[x + s:min(x + per, len(place)):step]].sum()
               for x in range(0, len(place), per) for s in range(min(step, per)))


def test_no_workgroup_has_more_than_in_the_plain_order(lib):
    rng = random.Random(3)
    # (kernel_size, side of a block of queries, parts of a block, workgroups per CU)
    bodies = [(3, 10, 1, 3), (5, 12, 1, 3), (7, 14, 1, 2), (9, 16, 1, 2), (11, 22, 2, 1), (13, 23, 2, 1), (13, 12, 1, 2)]
    sizes = [(26, 26, 128, 9), (26, 26, 700, 9), (28, 28, 128, 13), (32, 32, 128, 9), (24, 24, 700, 9), (34, 34, 128, 11),
             (36, 36, 128, 13), (34, 50, 128, 11), (62, 34, 128, 11), (26, 52, 128, 13), (60, 24, 128, 13)]
    turned = 0
    for i in range(400):
        if i < len(sizes):
            H, W, images, k = sizes[i]
            body = next(b for b in bodies if b[0] == k)
        else:
            body = rng.choice(bodies)
            H, W = (rng.randint(max(14, body[0]), 72) for _ in range(2))
            images = rng.choice((rng.randint(1, 16) * 8, rng.randint(1, 300)))
        k, side, parts, wgs = body
        costs, inner = frame_costs(H, W, k, side, parts)
        per_img, n = len(costs), len(costs) * images
        share = n / (n + inner * images / 2)  # (two inner tiles cost about one border tile)
        step = max(1, min(-(-n // 8), round(32 * wgs * share)))
        if n > 30000:
            continue
        turn, _, place = walk(lib, n, per_img, step)
        period = per_img // np.gcd(per_img, step)
        units = n / (8 * period * step)
        long = period == 1 or units >= 2 and (period <= 4 or units == int(units) or period <= 8 and units >= 3)
        assert (turn != 0) == (per_img >= 3 and period < per_img and long), (per_img, step)
        if turn:
            turned += 1
            new, old = (busiest(costs, x, step) for x in (place, walk(lib, n, per_img, step, plain=True)[2]))
            assert new <= old, (H, W, images, k, step, new, old)
    assert turned >= 30
    for (H, W, images, k), body, gain in (((26, 26, 128, 9), bodies[3], 1.5), ((28, 28, 128, 13), bodies[5], 1.8)):
        costs, _ = frame_costs(H, W, k, *body[1:3])
        n, step = len(costs) * images, 32 * body[3]
        new, old = (busiest(costs, walk(lib, n, len(costs), step, plain)[2], step) for plain in (False, True))
        assert gain * new <= old, (H, W, new, old)
