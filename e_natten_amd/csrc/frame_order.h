// Which border (frame) tiles a workgroup of the dK/dV pass takes.  Integers only, without HIP: the host
// chooses, the kernel walks, and tests compile it for the CPU.
#ifndef ENATTEN_FRAME_ORDER_H
#define ENATTEN_FRAME_ORDER_H

#ifdef __HIPCC__
#define ENATTEN_HD __host__ __device__ inline
#else
#define ENATTEN_HD inline
#endif

namespace enatten {

// Frame tiles are numbered image by image, `per_img` to an image, and a workgroup takes every `step`-th.
// A tile's cost depends on its place in the image (those of the second ring from the border have up to
// four blocks of queries, those of a corner one).  Where `step` is a multiple of per_img a workgroup would get
// the same place of every image, and those with the dearest end last: there the places of an image are counted
// from a start that moves on by `turn` from one of a workgroup's tiles to the next.  The same where `step` is
// half a multiple (two places) on walks of twelve tiles and more; over 1700 sizes whose tiles were charged their
// blocks and steps the busiest workgroup then never has more than in the plain order, on shorter walks up
// to 1.43 times as much.  Everywhere else the plain order brings a workgroup to a third of the places or more, and
// another is as often worse as better (34x34 d64 k11, 25 tiles, step 32: busiest workgroup 1.12 times the mean in
// the plain order, 1.09 to 1.33 in those that reach every place, up to 2.09 in the others).
// dK/dV pass, bf16, plain -> turned, us: 700 images of 26x26 d64 k9 (16 tiles, step 64) 491 -> 255, 128 images of
// 28x28 k13 (step 32) 224 -> 109.  Left plain: 128 images of 34x34 k11 118 (with steps of 15 tiles of 25 162),
// 62x34 k11 167 (214), 60x24 k13 147 (179).

// 0 for the plain order; `ntiles` tiles on eight runs
inline int frame_turn(int per_img, int step, long long ntiles) {
    if (per_img < 3 || 2 * step % per_img != 0 || (step % per_img != 0 && ntiles < 96ll * step)) return 0;
    // what a workgroup moves on by, from tile to tile: about 5/8 of the places, without a common factor,
    // so that it comes to all of them
    int on = per_img * 5 / 8;
    for (;; on++) {
        int a = per_img, b = on;
        while (b) { const int r = a % b; a = b; b = r; }
        if (a == 1) break;
    }
    return (on + per_img - step % per_img) % per_img;
}

struct FramePlace {
    int image, place;
};
// (a rotation of the places of each image; with a turn per_img <= 2 step, so the products stay within an int)
ENATTEN_HD FramePlace frame_place(int t, int per_img, int step, int turn) {
    FramePlace p;
    p.image = t / per_img;
    p.place = t - p.image * per_img;
    if (turn) p.place = (p.place + p.image * per_img / step % per_img * turn) % per_img;
    return p;
}

}  // namespace enatten

#endif  // ENATTEN_FRAME_ORDER_H
