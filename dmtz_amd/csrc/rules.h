// The critical-cell repair rules (fix_minimum / fix_saddle / fix_2saddle / fix_maximum,
// main_3d.cu:2554-4303) over cells kept in the frame of a vertex.
//
// repair.h states the rules over global simplex ids, as the reference does: every pairing lookup
// decodes an id, compares the cell's vertices and encodes the partner's id, some hundred 64-bit
// instructions each, and the rules' code grows to a hundred thousand instructions. Here a cell is
// (vertex, local index): its partner is read from the code of its highest vertex and is a cell in that
// vertex's frame, its other vertices are at fixed index offsets, and moving a cell to another
// vertex's frame is a table lookup. What is left of a rule is its comparisons and two to five
// dependent reads.
//
// The reference tells the kinds of a partner apart by testing whether the id, taken as one kind
// after the other, is paired back (an edge id, a tet id and a vertex id are plain numbers). The
// pairing codes name the kind, and the two agree except where numbers of different kinds collide:
//   - a face whose number is a vertex number, paired with a tet whose number, taken as an edge's,
//     is an edge at that vertex (face_taken_as_vertex);
//   - an edge paired with a vertex whose number, taken as a face's, is a face of the tet that has
//     the edge's number (vertex_taken_as_face).
// A rule that meets such a collision returns false before it emits anything, and the record takes the
// rule of repair.h. The host check compares both on every record of fields and grids where
// collisions do occur.
#pragma once
#include "edit.h"
#include "mismatch.h"

namespace dmtz {

struct alignas(4) RuleTables {
    uint8_t tri_i[36], tri_j[36];  // star triangles: the two other vertices' slots
    uint8_t tri_k[36][2];          // slots completing a star tet, and the tets
    uint8_t tri_q[36][2];
    uint8_t tri_at[36][2];         // the triangle seen from the vertex in slot tri_i, tri_j
    uint8_t tri_own[36], tri_mask[36];  // the vertex's corner in the triangle's cube, the triangle's corners
    uint8_t tet_s[24][3];          // star tets: slots
    uint8_t tet_face[24][3];       // the face (star triangle) that leaves out tet_s[q][c]
    uint8_t tet_at[24][3];         // the tet seen from the vertex in slot tet_s[q][c]
    uint8_t tet_own[24], tet_type[24];
    uint8_t tri_of[14][14];
    uint8_t adj_n[14], adj_l[14][6];
    uint8_t pad[2];
};
static_assert(sizeof(RuleTables) % 4 == 0 && sizeof(RuleTables) / 4 <= 256, "loaded by one word per thread of a block");

namespace detail {
constexpr void cube_of(const int* sl, int n, int& own, uint32_t& mask) {  // vertices 0 and DIR[sl[k]]
    int mn[3] = {0, 0, 0};
    for (int k = 0; k < n; k++)
        for (int a = 0; a < 3; a++) mn[a] = DIR[sl[k]][a] < mn[a] ? DIR[sl[k]][a] : mn[a];
    own = -mn[0] - 2 * mn[1] - 4 * mn[2];
    mask = 1u << own;
    for (int k = 0; k < n; k++)
        mask |= 1u << ((DIR[sl[k]][0] - mn[0]) + 2 * (DIR[sl[k]][1] - mn[1]) + 4 * (DIR[sl[k]][2] - mn[2]));
}
constexpr RuleTables make_rule_tables() {
    RuleTables r{};
    for (int t = 0; t < 36; t++) {
        const int i = ST.tri_i[t], j = ST.tri_j[t];
        r.tri_i[t] = (uint8_t)i;
        r.tri_j[t] = (uint8_t)j;
        for (int c = 0; c < 2; c++) {
            r.tri_k[t][c] = ST.tri_k[t][c];
            r.tri_q[t][c] = ST.tri_q[t][c];
        }
        r.tri_at[t][0] = (uint8_t)(SP.at_w[i][LC_TRI + t] - LC_TRI);
        r.tri_at[t][1] = (uint8_t)(SP.at_w[j][LC_TRI + t] - LC_TRI);
        const int sl[2] = {i, j};
        int own = 0;
        uint32_t mask = 0;
        cube_of(sl, 2, own, mask);
        r.tri_own[t] = (uint8_t)own;
        r.tri_mask[t] = (uint8_t)mask;
    }
    for (int q = 0; q < 24; q++) {
        const int sl[3] = {ST.tet_s[q][0], ST.tet_s[q][1], ST.tet_s[q][2]};
        for (int c = 0; c < 3; c++) {
            r.tet_s[q][c] = (uint8_t)sl[c];
            r.tet_face[q][c] = ST.tet_f[q][2 - c];
            r.tet_at[q][c] = (uint8_t)(SP.at_w[sl[c]][LC_TET + q] - LC_TET);
        }
        int own = 0;
        uint32_t mask = 0;
        cube_of(sl, 3, own, mask);
        r.tet_own[q] = (uint8_t)own;
        for (int k = 0; k < 6; k++)
            if (TET_MASK[k] == mask) r.tet_type[q] = (uint8_t)k;
    }
    for (int i = 0; i < 14; i++) {
        for (int j = 0; j < 14; j++) r.tri_of[i][j] = (uint8_t)(ST.tri_of[i][j] < 0 ? 0 : ST.tri_of[i][j]);
        r.adj_n[i] = ST.adj_n[i];
        for (int k = 0; k < 6; k++) r.adj_l[i][k] = ST.adj_l[i][k];
    }
    return r;
}
}  // namespace detail

constexpr RuleTables RT = detail::make_rule_tables();

// tb and off (the index offset of every slot, off[14] = 0) lie in LDS on the device.
template <class T, class Sink, class Code = const StarCode*>
struct LocalRules {
    const T* f;
    Code cf;
    const T* g;
    Code cg;
    const uint8_t* counter;
    const RuleTables* tb;
    const int32_t* off;
    const Dims& d;
    const Counts& c;
    double eps;
    int edit_type;
    Sink& sink;

    DMTZ_HD uint32_t at(uint32_t v, int slot) const { return v + (uint32_t)off[slot]; }
    static DMTZ_HD bool up(const T* x, uint32_t a, uint32_t b) {  // a above b
        const T va = x[a], vb = x[b];
        return va > vb || (va == vb && a > b);
    }
    static DMTZ_HD bool up(T va, T vb, uint32_t a, uint32_t b) { return va > vb || (va == vb && a > b); }
    DMTZ_HD bool fa(uint32_t a, uint32_t b) const { return up(f, a, b); }
    DMTZ_HD bool ga(uint32_t a, uint32_t b) const { return up(g, a, b); }
    DMTZ_HD void tgt(uint32_t v) { sink((i64)v); }

    struct At {  // a cell in the frame of its vertex v
        uint32_t v;
        int l;
    };
    // The cell in the frame of its highest vertex in field x.
    DMTZ_HD At edge_owner(const T* x, At e) const {
        const uint32_t w = at(e.v, e.l);
        return up(x, w, e.v) ? At{w, e.l ^ 1} : e;
    }
    DMTZ_HD At tri_owner(const T* x, At t) const {
        const uint32_t a = at(t.v, tb->tri_i[t.l]), b = at(t.v, tb->tri_j[t.l]);
        const T xv = x[t.v], xa = x[a], xb = x[b];
        At r = t;
        T m = xv;
        if (up(xa, m, a, r.v)) {
            r = At{a, tb->tri_at[t.l][0]};
            m = xa;
        }
        if (up(xb, m, b, r.v)) r = At{b, tb->tri_at[t.l][1]};
        return r;
    }
    DMTZ_HD At tet_owner(const T* x, At q) const {
        uint32_t w[3];
        T xw[3];
        for (int k = 0; k < 3; k++) {
            w[k] = at(q.v, tb->tet_s[q.l][k]);
            xw[k] = x[w[k]];
        }
        At r = q;
        T m = x[q.v];
        for (int k = 0; k < 3; k++)
            if (up(xw[k], m, w[k], r.v)) {
                r = At{w[k], tb->tet_at[q.l][k]};
                m = xw[k];
            }
        return r;
    }
    // Partner fields at the owner: edge: 14 = the owner, < 14 = the triangle completed by that slot,
    // 15 = none; triangle: 0 / 1 = edge to tri_i / tri_j, 2 / 3 = tet through tri_k[0] / [1], 7 = none;
    // tet: the slot its face leaves out, 3 = none.
    static DMTZ_HD int slot_of(const Code& cd, uint32_t v) { return partner_slot_of(cd, (i64)v); }
    static DMTZ_HD int edge_code(const Code& cd, At e) { return partner_edge_of(cd, (i64)e.v, e.l); }
    static DMTZ_HD int tri_code(const Code& cd, At t) { return partner_tri_of(cd, (i64)t.v, t.l); }
    static DMTZ_HD int tet_code(const Code& cd, At q) { return partner_tet_of(cd, (i64)q.v, q.l); }

    DMTZ_HD i64 tri_number(At t) const {
        i64 x, y, z;
        vxyz(d, (i64)t.v, x, y, z);
        const int o = tb->tri_own[t.l];
        return tri_id_local(d, c, x - (o & 1), y - ((o >> 1) & 1), z - (o >> 2), tb->tri_mask[t.l]);
    }
    DMTZ_HD i64 tet_number(At q) const {
        i64 x, y, z;
        vxyz(d, (i64)q.v, x, y, z);
        const int o = tb->tet_own[q.l];
        return 6 * ((z - (o >> 2)) * (d.W - 1) * (d.H - 1) + (y - ((o >> 1) & 1)) * (d.W - 1) + (x - (o & 1))) +
               tb->tet_type[q.l];
    }
    DMTZ_HD i64 edge_number(At e) const {
        i64 x, y, z;
        vxyz(d, (i64)e.v, x, y, z);
        // edge_id_dir with a run-time slot: the anchor is the smaller corner on every axis
        const int s = e.l;
        return EdgeBlocks(d).start(s >> 1) + edge_within(d, s >> 1, x - (DIR[s][0] < 0), y - (DIR[s][1] < 0), z - (DIR[s][2] < 0));
    }
    // Whether triangles outside the xy planes can have a vertex's number (they come after those).
    DMTZ_HD bool tiny() const { return c.foff[1] < c.N; }

    // Face t, paired with tet q: is t's number a vertex of the edge that has q's number?
    DMTZ_HD bool face_taken_as_vertex(At t, At q) const {
        if (!tiny() && (0xF0u & tb->tri_mask[t.l]) != 0) return false;  // not in an xy plane: number >= N
        const i64 p = tri_number(t);
        if (p >= c.N) return false;
        i64 a, b;
        edge_verts(d, c, tet_number(q), a, b);
        return p == a || p == b;
    }
    // Edge e, paired with vertex u: is the face that has u's number a face of the tet that has e's?
    DMTZ_HD bool vertex_taken_as_face(uint32_t u, At e) const {
        const i64 n = edge_number(e);
        if (n >= c.T) return false;
        if (!tiny()) {  // an xy face: its cube is the one above it or below it
            const i64 cube = n / 6, sq = u / 2;
            if (cube != sq && cube != sq - (d.W - 1) * (d.H - 1)) return false;
        }
        i64 w[3], q[4];
        tri_verts(d, c, (i64)u, w[0], w[1], w[2]);
        tet_verts(d, n, q[0], q[1], q[2], q[3]);
        bool in = true;
        for (int k = 0; k < 3; k++) in = in && (w[k] == q[0] || w[k] == q[1] || w[k] == q[2] || w[k] == q[3]);
        return in;
    }

    static DMTZ_HD void sort3(uint32_t& a, uint32_t& b, uint32_t& e) {  // descending
        uint32_t t;
        if (a < b) { t = a; a = b; b = t; }
        if (a < e) { t = a; a = e; e = t; }
        if (b < e) { t = b; b = e; e = t; }
    }
    DMTZ_HD void tri_vertices(At t, uint32_t& a, uint32_t& b, uint32_t& e) const {  // descending
        a = t.v;
        b = at(t.v, tb->tri_i[t.l]);
        e = at(t.v, tb->tri_j[t.l]);
        sort3(a, b, e);
    }
    DMTZ_HD double delta(uint32_t v) const {
        if (edit_type == 1) return halving_delta(eps, counter[v]);
        return EditArith<T>::delta0(f[v], g[v], eps);
    }
    DMTZ_HD bool slot_in_grid(uint32_t v, int slot) const {
        i64 x, y, z;
        vxyz(d, (i64)v, x, y, z);
        return inb(d, x + DIR[slot][0], y + DIR[slot][1], z + DIR[slot][2]);
    }

    // fix_minimum main_3d.cu:2554-2586
    DMTZ_HD bool minimum(uint32_t v) {
        const int s = slot_of(cf, v);
        tgt(s == 15 ? v : at(v, s));
        return true;
    }

    // fix_saddle main_3d.cu:2588-3037; edge a of v, v its owner in g
    DMTZ_HD bool saddle(uint32_t v, int a) {
        const uint32_t w = at(v, a), v1 = v > w ? v : w, v2 = v > w ? w : v;
        const At e = edge_owner(f, At{v, a});
        const int nib = edge_code(cf, e);
        if (nib == 14) {  // :2602-2641
            const uint32_t o = e.v == v ? w : v;
            const int s = slot_of(cg, e.v);
            if (s != 15 && ga(o, at(e.v, s))) tgt(o);
        } else if (nib < 14) {  // :2643-2827
            const uint32_t v3 = at(e.v, nib);
            const T f1 = f[v1], f2 = f[v2], f3 = f[v3], g1 = g[v1], g2 = g[v2], g3 = g[v3];
            const bool v1e = up(g1, g3, v1, v3), v2e = up(g2, g3, v2, v3);
            const bool o1 = up(f1, f3, v1, v3), o2 = up(f2, f3, v2, v3);
            if ((v1e && v2e) || (o1 && o2)) {
                tgt(v3);
                return true;
            }
            const At p{e.v, tb->tri_of[e.l][nib]};
            const At pg = tri_owner(g, p);
            const int cc = tri_code(cg, pg);
            if (cc < 2) {  // :2719-2799
                const At q{pg.v, cc == 0 ? tb->tri_i[pg.l] : tb->tri_j[pg.l]};
                const uint32_t qo = at(q.v, q.l), b3 = at(pg.v, cc == 0 ? tb->tri_j[pg.l] : tb->tri_i[pg.l]);
                const uint32_t a1 = q.v > qo ? q.v : qo, a2 = q.v > qo ? qo : q.v;
                const uint32_t fv = (a1 != v1 && a1 != v2) ? a1 : a2;
                if (fa(a2, b3) && fa(a1, b3)) {
                    const At qf = edge_owner(f, q);
                    const int nq = edge_code(cf, qf);
                    if (nq < 14) {
                        tgt(at(qf.v, nq));
                        return true;
                    }
                    if (nq == 14 && vertex_taken_as_face(qf.v, q)) return false;
                }
                if (fabs_d(delta(fv)) > 0) tgt(fv);
            } else {
                if (cc < 4 && face_taken_as_vertex(pg, At{pg.v, tb->tri_q[pg.l][cc - 2]})) return false;
                if (o1 && !v1e) tgt(v3);
                else tgt(!v2e ? v3 : v2);
            }
        } else {  // false negative :2830-3036
            const int ng = edge_code(cg, At{v, a});
            if (ng == 14) {
                tgt(v);
            } else if (ng < 14) {
                const uint32_t v3 = at(v, ng);
                const bool v1e = ga(v2, v3), v2e = ga(v1, v3);  // :2886-2887
                const bool or1 = fa(v2, v3), or2 = fa(v1, v3);
                if (v1e == v2e) {
                    if (v1e != or1) tgt(v2);
                    if (v2e != or2) tgt(v1);
                } else {  // lowest f-vertex of the edge's link between its ends (:2942-3003)
                    const int sl = v1 == v ? a : a ^ 1;
                    i64 x, y, z;
                    vxyz(d, (i64)v1, x, y, z);
                    bool any = false;
                    uint32_t best = 0;
                    for (int k = 0; k < tb->adj_n[sl]; k++) {
                        const int s = tb->adj_l[sl][k];
                        if (!inb(d, x + DIR[s][0], y + DIR[s][1], z + DIR[s][2])) continue;
                        const uint32_t n = at(v1, s);
                        if (fa(v1, n) != fa(v2, n) && (!any || fa(best, n))) {
                            best = n;
                            any = true;
                        }
                    }
                    if (any) {
                        tgt(best);
                    } else {
                        tgt(v1);
                        tgt(v2);
                    }
                }
            }
        }
        return true;
    }

    // fix_2saddle main_3d.cu:3039-3983; triangle t of v, v its owner in g
    DMTZ_HD bool saddle2(uint32_t v, int t) {
        const At m = tri_owner(f, At{v, t});
        const int cc = tri_code(cf, m);
        if (cc < 2) {  // :3057-3223
            const At p{m.v, cc == 0 ? tb->tri_i[m.l] : tb->tri_j[m.l]};
            const uint32_t po = at(p.v, p.l), v3 = at(m.v, cc == 0 ? tb->tri_j[m.l] : tb->tri_i[m.l]);
            const uint32_t v1 = p.v > po ? p.v : po, v2 = p.v > po ? po : p.v;
            const T f1 = f[v1], f2 = f[v2], f3 = f[v3], g1 = g[v1], g2 = g[v2], g3 = g[v3];
            const bool v1e = up(g2, g3, v2, v3), v2e = up(g1, g3, v1, v3);
            const bool o1 = up(f2, f3, v2, v3), o2 = up(f1, f3, v1, v3);
            // v3 below both in g: the edge's face in f is this one, whose third vertex is v3
            uint32_t r = v3;
            if (o1 != o2 && v1e != v2e) {
                const At pg = up(g1, g2, v1, v2) == (p.v == v1) ? p : At{po, p.l ^ 1};
                const int nib = edge_code(cg, pg);
                if (nib < 14) {
                    const uint32_t w3 = at(pg.v, nib);
                    const T f4 = f[w3], g4 = g[w3];
                    if (up(g2, g4, v2, w3) && up(g1, g4, v1, w3)) {
                        const bool oe1 = up(f2, f4, v2, w3), oe2 = up(f1, f4, v1, w3);
                        if (oe1 != oe2) r = oe1 ? v1 : v2;
                    }
                } else if (nib == 14 && vertex_taken_as_face(pg.v, p)) {
                    return false;
                }
            }
            tgt(r);
        } else if (cc < 4) {  // :3226-3477
            const At p{m.v, tb->tri_q[m.l][cc - 2]};
            if (face_taken_as_vertex(m, p)) return false;
            const uint32_t a = at(m.v, tb->tri_i[m.l]), b = at(m.v, tb->tri_j[m.l]);
            const uint32_t v4 = at(m.v, tb->tri_k[m.l][cc - 2]);
            const T f4 = f[v4];
            if (up(f[a], f4, a, v4) && up(f[b], f4, b, v4) && up(f[m.v], f4, m.v, v4)) {
                tgt(v4);
                return true;
            }
            const At pg = tet_owner(g, p);
            const int ct = tet_code(cg, pg);
            if (ct == 3) {
                tgt(v4);
                return true;
            }
            const At w{pg.v, tb->tet_face[pg.l][ct]};
            uint32_t w1, w2, w3;
            tri_vertices(w, w1, w2, w3);
            const T g4 = g[v4];
            const bool gall = up(g[w3], g4, w3, v4) && up(g[w2], g4, w2, v4) && up(g[w1], g4, w1, v4);
            const bool hall = up(f[w3], f4, w3, v4) && up(f[w2], f4, w2, v4) && up(f[w1], f4, w1, v4);
            if (!gall && !hall) {
                const At wf = tri_owner(f, w);
                const int ci = tri_code(cf, wf);
                if (ci < 2) {  // :3288, the face's vertex off the edge
                    tgt(at(wf.v, ci == 0 ? tb->tri_j[wf.l] : tb->tri_i[wf.l]));
                } else if (ci < 4) {  // :3302
                    if (face_taken_as_vertex(wf, At{wf.v, tb->tri_q[wf.l][ci - 2]})) return false;
                    // the tet's vertices in descending order, where :3307-3309 put the face's
                    // vertex at the place of the fourth: w3 is dropped when the new one is above w2
                    const uint32_t x = at(wf.v, tb->tri_k[wf.l][ci - 2]);
                    tgt(w1);
                    tgt(w2);
                    tgt(x);
                    if (x < w2) tgt(w3);
                }
            } else {
                tgt(w1);
                tgt(w2);
                tgt(w3);
            }
        } else {  // false negative :3480-3981
            const int cq = tri_code(cg, At{v, t});
            if (cq < 2) {  // :3488-3610
                const At q{v, cq == 0 ? tb->tri_i[t] : tb->tri_j[t]};
                const At qf = edge_owner(f, q);
                const int nib = edge_code(cf, qf);
                if (nib < 14) {
                    tgt(at(qf.v, nib));
                } else if (nib == 14) {
                    if (vertex_taken_as_face(qf.v, q)) return false;
                    tgt(v);
                    tgt(at(v, q.l));
                }
            } else if (cq < 4) {  // :3613-3980
                const At q{v, tb->tri_q[t][cq - 2]};
                if (face_taken_as_vertex(At{v, t}, q)) return false;
                uint32_t v1, v2, v3;
                tri_vertices(At{v, t}, v1, v2, v3);
                const uint32_t v4 = at(v, tb->tri_k[t][cq - 2]);
                if (ga(v3, v4) && ga(v2, v4) && ga(v1, v4)) {
                    if (!fa(v3, v4)) tgt(v3);
                    else if (!fa(v2, v4)) tgt(v2);
                    else if (!fa(v1, v4)) tgt(v1);
                    return true;
                }
                const At qf = tet_owner(f, q);
                const int ct = tet_code(cf, qf);
                bool all = ct != 3 && tri_number(At{qf.v, tb->tet_face[qf.l][ct]}) < c.T;  // :3937: a face id
                uint32_t best = 0;
                bool any = false;
                if (!all) {  // get_smallest_vertex main_3d.cu:2115-2194
                    for (int k = 0; k < 2; k++) {
                        const int s = tb->tri_k[t][k];
                        if (!slot_in_grid(v, s)) continue;
                        const uint32_t n = at(v, s);
                        if ((int)fa(v1, n) + (int)fa(v2, n) + (int)fa(v3, n) == 2 && (!any || fa(best, n))) {
                            best = n;
                            any = true;
                        }
                    }
                    all = !any;
                }
                if (all) {
                    tgt(v1);
                    tgt(v2);
                    tgt(v3);
                } else {
                    tgt(best);
                }
            }
        }
        return true;
    }

    // fix_maximum main_3d.cu:3985-4303; tet q of v, v its owner in g
    DMTZ_HD bool maximum(uint32_t v, int q) {
        const At m = tet_owner(f, At{v, q});
        const int ct = tet_code(cf, m);
        uint32_t v1, v2, v3;
        if (ct < 3) {
            const At p{m.v, tb->tet_face[m.l][ct]};
            tri_vertices(p, v1, v2, v3);
            const uint32_t v4 = at(m.v, tb->tet_s[m.l][ct]);
            if (fa(v1, v4) && fa(v2, v4) && fa(v3, v4)) {
                tgt(v4);
                return true;
            }
            const At pg = tri_owner(g, p);
            const int cc = tri_code(cg, pg);
            if (cc < 2) {
                tgt(pg.v);  // the higher end of the edge in g: the face's owner
            } else if (cc < 4) {
                if (face_taken_as_vertex(pg, At{pg.v, tb->tri_q[pg.l][cc - 2]})) return false;
                tgt(v4);
            }
            return true;
        }
        const int cg_ = tet_code(cg, At{v, q});
        if (cg_ == 3) return true;  // critical in both fields: not a mismatch
        const At p{v, tb->tet_face[q][cg_]};
        tri_vertices(p, v1, v2, v3);
        const uint32_t v4 = at(v, tb->tet_s[q][cg_]);
        const bool o1 = fa(v1, v4), o2 = fa(v2, v4), o3 = fa(v3, v4);
        const bool gall = ga(v1, v4) && ga(v2, v4) && ga(v3, v4), oall = o1 && o2 && o3;
        if (!gall || oall) {
            const At pf = tri_owner(f, p);
            const int ci = tri_code(cf, pf);
            if (ci < 2) {
                const At e{pf.v, ci == 0 ? tb->tri_i[pf.l] : tb->tri_j[pf.l]};
                if (!gall) {
                    tgt(pf.v);
                    tgt(at(e.v, e.l));
                } else {  // the reference takes the edge's number for a tet's
                    i64 t1, t2, t3, t4;
                    tet_verts(d, edge_number(e), t1, t2, t3, t4);
                    i64 w = t4;
                    if (t1 != v1 && t1 != v2 && t1 != v3) w = t1;
                    else if (t2 != v1 && t2 != v2 && t2 != v3) w = t2;
                    else if (t3 != v1 && t3 != v2 && t3 != v3) w = t3;
                    if (w >= 0 && w < c.N) sink(w);
                }
                return true;
            }
            if (ci < 4) {
                const uint32_t x = at(pf.v, tb->tri_k[pf.l][ci - 2]);
                if (!gall) {
                    if (face_taken_as_vertex(pf, At{pf.v, tb->tri_q[pf.l][ci - 2]})) return false;
                    tgt(v1);
                    tgt(v2);
                    tgt(v3);
                }
                tgt(x);
                return true;
            }
            if (gall) return true;
        }
        if (!o1) tgt(v1);
        if (!o2) tgt(v2);
        if (!o3) tgt(v3);
        return true;
    }

    // The rule of a record (vertex v, local cell lc); TYPE is its cell type.
    template <int TYPE>
    DMTZ_HD bool run(uint32_t v, int lc) {
        if (TYPE == 0) return minimum(v);
        if (TYPE == 1) return saddle(v, lc - LC_EDGE);
        if (TYPE == 2) return saddle2(v, lc - LC_TRI);
        return maximum(v, lc - LC_TET);
    }
};

}  // namespace dmtz
