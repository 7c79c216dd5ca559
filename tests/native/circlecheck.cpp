// Host build of walls.h for tests: every chain of a field pair followed to its end, against
// Repair::wall_walk.
#include <cstdint>
#include <vector>
#include "walls.h"

using namespace dmtz;

// out: chains, those that run in a circle, the most steps of one, disagreements
template <class T>
static void check(const T* f, const T* g, i64 W, i64 H, i64 D, i64* out) {
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
    const FieldGrad<T> F(f, cf.data(), d, c);
    int32_t off[15];
    for (int s = 0; s < 14; s++) off[s] = (int32_t)(DIR[s][0] + DIR[s][1] * W + DIR[s][2] * W * H);
    off[14] = 0;
    NullSink none;
    const LocalRules<T, NullSink> R{f, cf.data(), g, cg.data(), nullptr, &RT, off, d, c, 0.0, 0, none};
    const WallGraph<T> G{R, &WT};
    Repair<T, NullSink> S(f, cf.data(), g, cg.data(), d, c, nullptr, 0, 0, 0, none);
    std::vector<uint8_t> open(12 * c.N, 0);
    std::vector<uint32_t> queue;
    auto add = [&](typename WallGraph<T>::At t) {
        const uint32_t id = G.face_id(t);
        if (!open[id]) {
            open[id] = 1;
            queue.push_back(id);
        }
    };
    for (i64 v = 0; v < c.N; v++)
        G.mismatched_edges((uint32_t)v, [&](typename WallGraph<T>::At e) { G.faces_of(e, add); });
    for (size_t k = 0; k < queue.size(); k++) G.leading_to(G.face_at(queue[k]), add);
    for (i64 v = 0; v < c.N; v++) {
        uint64_t lo, ilo;
        uint32_t hi, ihi;
        code_masks(cf[v], lo, hi, ilo, ihi);
        for (int lc = LC_TRI; lc < LC_TET; lc++) {
            if (!(((lo & ilo) >> lc) & 1)) continue;
            const typename WallGraph<T>::At t{(uint32_t)v, lc - LC_TRI};
            if (!open[G.face_id(t)]) continue;
            typename WallGraph<T>::At e{0, 0};
            i64 steps = 0, want = -1;
            const int s = G.follow(t, e, [&](uint32_t x) { return open[x] != 0; }, steps);
            out[0]++;
            out[2] = steps > out[2] ? steps : out[2];
            std::vector<uint32_t> buf(2 * (1u << 10) + 2);
            const bool over = S.wall_walk(local_cell_id(d, c, v, lc), buf.data(), buf.data() + (1u << 10), 1u << 10, want);
            if (s == 0) out[1]++;
            out[3] += s < 0 || over || want < 0 || (s == 1 && R.edge_number(e) != want);
        }
    }
}

extern "C" void wc_follow_f32(const float* f, const float* g, int64_t W, int64_t H, int64_t D, int64_t* out) {
    check<float>(f, g, W, H, D, out);
}
extern "C" void wc_follow_f64(const double* f, const double* g, int64_t W, int64_t H, int64_t D, int64_t* out) {
    check<double>(f, g, W, H, D, out);
}
