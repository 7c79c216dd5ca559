// Host build of star_planes.h for tests: codes and masks of every vertex, 32 at a time, against
// lower_star.h.
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
    const i64 N = W * H * D;
    i64 bad = 0;
    for (i64 v0 = 0; v0 < N; v0 += 32) {
        StarWords sw{};
        uint32_t side[6] = {0, 0, 0, 0, 0, 0};
        for (int r = 0; r < 32; r++) {
            T val[15];
            const i64 v = v0 + r < N ? v0 + r : N - 1;
            i64 x, y, z;
            vxyz(d, v, x, y, z);
            const bool in[6] = {x > 0, x < W - 1, y > 0, y < H - 1, z > 0, z < D - 1};
            for (int k = 0; k < 6; k++) side[k] = (side[k] << 1) | (uint32_t)in[k];
            gather_star(f, d, v, val);
            for (int k = 0; k < 14; k++)  // outside the grid: any finite value
                if (!inb(d, x + DIR[k][0], y + DIR[k][1], z + DIR[k][2])) val[k] = (T)(k % 3) - 1;
            add_vertex(val, sw);
        }
        finish(sw, side);
        Collect c;
        classify_words(sw, c);
        for (int r = 0; r < 32 && v0 + r < N; r++) {
            const int b = 31 - r;
            LowerStar ls;
            star_of(f, d, v0 + r, ls);
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

extern "C" int64_t sp_check_f32(const float* f, int64_t W, int64_t H, int64_t D) { return check<float>(f, W, H, D); }
extern "C" int64_t sp_check_f64(const double* f, int64_t W, int64_t H, int64_t D) { return check<double>(f, W, H, D); }
