// Host build of the star classifier for tests of fields with infinities: a vertex's lower slots lie in
// the grid, and its star code is that of a finite field with the same order.
#include <cstdint>
#include "gradient.h"

using namespace dmtz;

template <class T>
static i64 check(const T* f, const T* finite, i64 W, i64 H, i64 D) {
    Dims d{W, H, D};
    i64 bad = 0;
    for (i64 v = 0; v < W * H * D; v++) {
        i64 x, y, z;
        vxyz(d, v, x, y, z);
        LowerStar a, b;
        star_of(f, d, v, a);
        star_of(finite, d, v, b);
        for (int k = 0; k < 14; k++)
            bad += ((a.L >> k) & 1u) && !inb(d, x + DIR[k][0], y + DIR[k][1], z + DIR[k][2]);
        StarCode ca, cb;
        encode_star(a, ca);
        encode_star(b, cb);
        for (int k = 0; k < 4; k++) bad += ca.w[k] != cb.w[k];
    }
    return bad;
}

extern "C" int64_t ic_check_f32(const float* f, const float* g, int64_t W, int64_t H, int64_t D) {
    return check<float>(f, g, W, H, D);
}
extern "C" int64_t ic_check_f64(const double* f, const double* g, int64_t W, int64_t H, int64_t D) {
    return check<double>(f, g, W, H, D);
}
