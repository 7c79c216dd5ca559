// Host build of rules.h for tests: every rule on every mismatched cell, against the rule of repair.h
// (which the host check compares with the oracle).
#include <cstdint>
#include <set>
#include <vector>
#include "repair.h"
#include "rules.h"

using namespace dmtz;

struct SetSink {
    std::set<i64>* s;
    void operator()(i64 v) const { s->insert(v); }
};

// out: records, records sent to the general rule, records whose edit sets differ. With every != 0
// each cell critical in one field only is a record at its owner in g, as in the correction.
template <class T>
static void check(const T* f, const T* g, i64 W, i64 H, i64 D, double eps, int edit_type, const uint8_t* counter,
                  i64* out) {
    Dims d{W, H, D};
    Counts c = make_counts(d);
    std::vector<StarCode> cf(c.N), cg(c.N);
    for (i64 v = 0; v < c.N; v++) {
        LowerStar ls;
        star_of(f, d, v, ls);
        encode_star(ls, cf[v]);
        star_of(g, d, v, ls);
        encode_star(ls, cg[v]);
    }
    FieldGrad<T> F(f, cf.data(), d, c);
    int32_t off[15];
    for (int s = 0; s < 14; s++) off[s] = (int32_t)(DIR[s][0] + DIR[s][1] * W + DIR[s][2] * W * H);
    off[14] = 0;
    for (i64 v = 0; v < c.N; v++) {
        uint64_t flo, lo;
        uint32_t fhi, hi;
        local_crit(F, v, flo, fhi);
        owner_mismatch(cg[v], flo, fhi, lo, hi);
        for (int lc = 0; lc < LC_COUNT; lc++) {
            if (!lc_bit(lo, hi, lc)) continue;
            std::set<i64> want, got;
            SetSink ws{&want}, gs{&got};
            Repair<T, SetSink> R(f, cf.data(), g, cg.data(), d, c, counter, eps, 1.0, edit_type, ws);
            LocalRules<T, SetSink> L{f, cf.data(), g, cg.data(), counter, &RT, off, d, c, eps, edit_type, gs};
            const i64 id = local_cell_id(d, c, v, lc);
            bool done = true;
            switch (lc_type(lc)) {
                case 0: R.fix_minimum(id); done = L.template run<0>((uint32_t)v, lc); break;
                case 1: R.fix_saddle(id); done = L.template run<1>((uint32_t)v, lc); break;
                case 2: R.fix_2saddle(id); done = L.template run<2>((uint32_t)v, lc); break;
                default: R.fix_maximum(id); done = L.template run<3>((uint32_t)v, lc);
            }
            out[0]++;
            if (!done) {
                out[1]++;
                out[2] += !got.empty();  // nothing may be emitted before the general rule runs
            } else {
                out[2] += got != want;
            }
        }
    }
}

extern "C" void rc_check_f32(const float* f, const float* g, int64_t W, int64_t H, int64_t D, double eps, int et,
                             const uint8_t* counter, int64_t* out) {
    check<float>(f, g, W, H, D, eps, et, counter, out);
}
extern "C" void rc_check_f64(const double* f, const double* g, int64_t W, int64_t H, int64_t D, double eps, int et,
                             const uint8_t* counter, int64_t* out) {
    check<double>(f, g, W, H, D, eps, et, counter, out);
}
