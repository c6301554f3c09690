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
// four blocks of queries, those of a corner one).  In the plain order a workgroup gets the same per_img / gcd(step,
// per_img) places of every image, and those with the dearest end last: where they are few, the places of an image are
// counted from a start that moves on by `turn` with every `unit` tiles, `unit` being the first multiple of step that is
// one of per_img.  Within a unit a workgroup then has the places that it has in the plain order, and in the next
// unit those of another workgroup, so whole units are never dearer than in the plain order.  Parts of one may be, so
// two to four places are turned on walks of two units and more, five to eight on three, and any number on whole
// units: a cost model of 3000 walks finds none dearer with that (some by 2% with five to eight places on two units, or
// with more).  One place: 0.54 to 1 of the busiest workgroup's cost, two 0.64 to 1, three and four 0.70 to 1,
// five to eight 0.74 to 1.
// dK/dV pass, bf16, plain -> turned, us: one place, 700 images of 26x26 d64 k9 (16 tiles, step 64) 491 -> 255, 128 images of
// 28x28 k13 (step 32) 224 -> 109; four, 16 images of 128x128 d128 k13 (256 tiles, step 64) 226 -> 213, k11 213 -> 207.  Left
// plain: 128 images of 34x34 d64 k11 (25 tiles, step 32) 118 (with steps of 15 tiles of 25 162).
struct FrameOrder {
    int turn, unit;  // turn 0: the plain order
};
// `ntiles` tiles, an eighth of them to each XCD
inline FrameOrder frame_order(int per_img, int step, long long ntiles) {
    auto gcd = [](int a, int b) {
        while (b) { const int r = a % b; a = b; b = r; }
        return a;
    };
    const int others = gcd(step, per_img), places = per_img / others;  // `others` workgroups differ in their places
    const long long unit = (long long)places * step;
    if (per_img < 3 || others < 2 || ntiles < 8 * unit * (places == 1 ? 0 : 2) ||
        (places > 4 && ntiles % (8 * unit) && (places > 8 || ntiles < 24 * unit)))
        return {0, 1};
    // about 5/8 of them, without a common factor, so that it comes to all
    int turn = others * 5 / 8;
    while (gcd(others, turn) != 1) turn++;
    return {turn, (int)unit};
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
