// Host build of a wave's tile (star_planes.h tile_words) for tests: the rows, sides and clamped loads of
// every lane of every tile, classified, against the classifier of one vertex.
#include <cstdint>
#include <vector>
#include "gradient.h"
#include "mismatch.h"
#include "star_planes.h"

using namespace dmtz;

struct Collect {
    uint64_t w[4][32];
    uint64_t clo[32], ilo[32];
    uint32_t chi[32], ihi[32];
    void code(int k, const uint32_t* lo, const uint32_t* hi) {
        for (int r = 0; r < 32; r++) w[k][r] = (uint64_t)hi[r] << 32 | lo[r];
    }
    void masks_lo(const uint32_t* c0, const uint32_t* c1, const uint32_t* i0, const uint32_t* i1) {
        for (int r = 0; r < 32; r++) {
            clo[r] = (uint64_t)c1[r] << 32 | c0[r];
            ilo[r] = (uint64_t)i1[r] << 32 | i0[r];
        }
    }
    void masks_hi(const uint32_t* c2, const uint32_t* i2) {
        for (int r = 0; r < 32; r++) {
            chi[r] = c2[r];
            ihi[r] = i2[r];
        }
    }
};

template <class T>
static i64 check(const T* f, i64 W, i64 H, i64 D) {
    Dims d{W, H, D};
    const Step64 st(d);
    const i64 N = W * H * D;
    i64 bad = 0;
    for (i64 base = 0; base < N; base += PLANE_TILE)
        for (i64 v0 = base; v0 < base + 64; v0++) {
            StarWords sw;
            tile_words(f, d, st, N, v0, sw);
            Collect c;
            classify_words(sw, c);
            for (int row = 0; row < PLANE_ROWS && v0 + 64 * row < N; row++) {
                const int b = 31 - row;
                LowerStar ls;
                star_of(f, d, v0 + 64 * row, ls);
                StarCode sc;
                encode_star(ls, sc);
                uint64_t clo, ilo;
                uint32_t chi, ihi;
                crit_mask(ls, clo, chi);
                member_mask(ls, ilo, ihi);
                for (int k = 0; k < 4; k++) bad += sc.w[k] != c.w[k][b];
                bad += (clo != c.clo[b]) + (ilo != c.ilo[b]) + (chi != c.chi[b]) + (ihi != c.ihi[b]);
            }
        }
    return bad;
}

extern "C" int64_t tc_check_f32(const float* f, int64_t W, int64_t H, int64_t D) { return check<float>(f, W, H, D); }
extern "C" int64_t tc_check_f64(const double* f, int64_t W, int64_t H, int64_t D) { return check<double>(f, W, H, D); }
