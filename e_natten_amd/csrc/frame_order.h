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
// four blocks of queries, those of a corner one).  Where `step` is a multiple of per_img, or of half of it, a
// workgroup would get one place of every image, or two, and those with the dearest end last: there the
// places of an image are counted from a start that moves on by `turn` with every `unit` tiles, `unit` being the first
// multiple of step that is one of per_img.  Within a unit a workgroup then has the places that it has in the plain
// order, and in the next unit those of another workgroup, so whole units are never dearer than in the plain order;
// parts of one may be, so the two places are turned on walks of two units and more.  Everywhere else the plain order brings
// a workgroup to a third of the places or more, and another is as often worse as better (34x34 d64 k11, 25
// tiles, step 32: busiest workgroup 1.12 times the mean in the plain order, 1.09 to 1.33 in those that move on
// by a number without a common factor, up to 2.09 in the others).
// dK/dV pass, bf16, plain -> turned, us: 700 images of 26x26 d64 k9 (16 tiles, step 64) 491 -> 255, 128 images of
// 28x28 k13 (step 32) 224 -> 109.  Left plain: 128 images of 34x34 k11 118 (with steps of 15 tiles of 25 162),
// 62x34 k11 167 (214), 60x24 k13 147 (179).
struct FrameOrder {
    int turn, unit;  // turn 0: the plain order
};
// `ntiles` tiles, an eighth of them to each XCD
inline FrameOrder frame_order(int per_img, int step, long long ntiles) {
    const int unit = step % per_img == 0 ? step : 2 * step;
    if (per_img < 3 || unit % per_img != 0 || (unit != step && ntiles < 16ll * unit)) return {0, 1};
    // about 5/8 of the workgroups that differ in their places, without a common factor, so that it comes to all
    const int others = unit == step ? per_img : per_img / 2;
    int turn = others * 5 / 8;
    for (;; turn++) {
        int a = others, b = turn;
        while (b) { const int r = a % b; a = b; b = r; }
        if (a == 1) break;
    }
    return {turn, unit};
}

struct FramePlace {
    int image, place;
};
// (a rotation of the places of each image; per_img is at most unit where there is a turn, so the product stays
// within an int)
ENATTEN_HD FramePlace frame_place(int t, int per_img, FrameOrder o) {
    FramePlace p;
    p.image = t / per_img;
    p.place = t - p.image * per_img;
    if (o.turn) p.place = (p.place + p.image * per_img / o.unit % per_img * o.turn) % per_img;
    return p;
}

}  // namespace enatten

#endif  // ENATTEN_FRAME_ORDER_H
