// Host build of pairs.h for tests: the pair words and the walks over them against the pairing
// lookups and walks of gradient.h and repair.h (which the host check compares with the oracle).
#include <cstdint>
#include <vector>
#include "pairs.h"
#include "repair.h"
#include "mismatch.h"

using namespace dmtz;

struct Nothing {
    void operator()(i64) const {}
};

template <class T>
static i64 check(const T* f, const T* g, i64 W, i64 H, i64 D) {
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
    const FieldGrad<T> F(f, cf.data(), d, c), G(g, cg.data(), d, c);
    Repair<T, Nothing> R(f, cf.data(), g, cg.data(), d, c, nullptr, 0, 0, 0, Nothing{});
    std::vector<uint32_t> pf(c.N), pg(c.N);
    i64 step[14];
    for (uint32_t s = 0; s < 14; s++) step[s] = slot_step(d, s);
    i64 bad = 0;
    for (i64 v = 0; v < c.N; v++) {
        i64 x, y, z;
        vxyz(d, v, x, y, z);
        pf[v] = pair_word(f, cf.data(), d, v, x, y, z);
        pg[v] = pair_word(g, cg.data(), d, v, x, y, z);
    }
    for (i64 v = 0; v < c.N; v++) {
        i64 x, y, z;
        vxyz(d, v, x, y, z);
        const bool cube = x < W - 1 && y < H - 1 && z < D - 1;
        const uint32_t s = pw_slot(pf[v]);
        bad += F.pv(v) != (s == PW_NO_SLOT ? -1 : F.edge_of(v, (int)s));
        const uint32_t m = pair_mismatch(pf[v], pg[v]);
        bad += ((m & MIS_SLOT) != 0) != (F.pv(v) != -1 && F.pv(v) != G.pv(v));
        for (int t = 0; t < 6; t++) {
            const uint32_t out = pw_out(pf[v], t);
            if (!cube) {
                bad += out != PW_NONE;
                continue;
            }
            TetAt a{v, (int)x, (int)y, (int)z, t};
            const i64 id = tet_id_at(d, a);
            bad += id != tet_id_of_vertex(d, v, t);
            i64 w[3], face = -1;
            if (out != PW_NONE) {
                int n = 0;
                for (int k = 0; k < 4; k++)
                    if (k != (int)out) w[n++] = corner_vidx(d, x, y, z, PT.corner[t][k]);
                face = tri_id3(d, c, w[0], w[1], w[2]);
                i64 q0, q1;  // the tet across that face
                R.cofacets(face, q0, q1);
                cross_face(d, a, PT.across[4 * t + out]);
                bad += (a.v < 0 ? -1 : tet_id_at(d, a)) != (q0 == id ? q1 : q0);
                bad += a.v >= 0 && a.v != vidx(d, a.x, a.y, a.z);
            }
            bad += F.pt(id) != face;
            bad += (((m >> t) & 1u) != 0) != (F.pt(id) != G.pt(id));
        }
        bool ovf = false;
        bad += paired_min(pf.data(), step, v, c.N, ovf) != R.f_min_label(v, c.N, ovf);
        i64 t1 = -1, t2 = -1;
        bad += g_min_of(pf.data(), pg.data(), step, v, t1, c.N, ovf) != R.g_min_walk(v, t2, c.N, ovf);
        bad += t1 != t2 || ovf;
        // cofacets of every star triangle, and the walks from them
        uint64_t elo;
        uint32_t ehi;
        local_cells_exist(d, v, elo, ehi);
        for (int t = 0; t < 36; t++) {
            if (!((elo >> (LC_TRI + t)) & 1)) continue;
            const i64 tri = local_cell_id(d, c, v, LC_TRI + t);
            i64 q[2];
            R.cofacets(tri, q[0], q[1]);
            int n = 0;
            for (int k = 0; k < 2; k++) {
                const TetAt a = start_tet(d, v, (int)x, (int)y, (int)z, PT.start[t][k]);
                if (a.v < 0) continue;
                const i64 id = q[n++];
                bad += tet_id_at(d, a) != id;
                bool found, o2 = false;
                i64 dv;
                TetAt div = a;
                R.as_walk(id, c.N, found, dv, o2);
                bad += path_mismatch(d, pf.data(), pg.data(), PT.across, a, c.N, div, ovf) != found;
                bad += found && tet_id_at(d, div) != dv;
                const i64 h = paired_max(d, pg.data(), PT.across, a, c.N, ovf), want = R.paired_max(id, 1, c.N, o2);
                bad += (h < 0 ? -1 : tet_id_of_vertex(d, h / 8, (int)(h % 8))) != want;
                bad += ovf || o2;
            }
            bad += n < 2 && q[n] != -1;
        }
        // the edges v records in the descending check
        uint64_t lo;
        uint32_t hi;
        for (int s2 = 0; s2 < 14; s2++) {
            if (!((elo >> (LC_EDGE + s2)) & 1)) continue;
            const i64 w = v + step[s2];
            i64 rec;
            const bool has = R.ds_geometry(local_cell_id(d, c, v, LC_EDGE + s2), rec) && rec == v;
            const bool mine = (m & MIS_SLOT) && (w < v || !(pair_mismatch(pf[w], pg[w]) & MIS_SLOT));
            bad += has != mine;
            bad += (w < v) != ((s2 & 1) != 0);
        }
        (void)lo;
        (void)hi;
    }
    return bad;
}

extern "C" int64_t pc_check_f32(const float* f, const float* g, int64_t W, int64_t H, int64_t D) {
    return check<float>(f, g, W, H, D);
}
extern "C" int64_t pc_check_f64(const double* f, const double* g, int64_t W, int64_t H, int64_t D) {
    return check<double>(f, g, W, H, D);
}
