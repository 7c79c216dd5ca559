// 2-saddle walls (get_false_ds_wall main_3d.cu:5064-5133) from the mismatched edges backwards.
//
// Repair::wall_walk searches every wall depth first for its first mismatched edge, a serial walk with
// a visited set of its own per f-critical face; near convergence nearly all walls hold none and are
// searched to their end. Whether a search meets a mismatch does not depend on its order, so the
// faces from which one is reached ("open" faces) are found once for all walls, backwards: the faces
// of the mismatched edges, then, from each open face paired with an edge, that edge's other faces.
// A search that enters only open faces meets the same first mismatch (the others hold none), and it
// never turns back: every open face has a mismatched edge of its own or leads on to an open face, and
// of several the search takes the one pushed last. What is left of a walk is that chain.
//
// As in rules.h, the reference compares partners as plain numbers: a vertex and a face with one
// number count as equal partners, and an edge paired with a vertex leads on to the face that has the
// vertex's number if that face is paired with the tet that has the edge's number. Such links can close
// a circle (about one chain in 150 thousand over random fields of a few dozen vertices); a face whose
// chain comes back to itself takes the search of repair.h.
#pragma once
#include "repair.h"
#include "rules.h"

namespace dmtz {

// Faces by anchor (the smallest corner's vertex): 12 kinds per vertex, as 12 v + kind.
struct alignas(4) WallTables {
    uint8_t kind[36];       // of star triangle t
    uint8_t corner[12];     // a corner of each kind and the star triangle there
    uint8_t tri[12];
};
namespace detail {
constexpr WallTables make_wall_tables() {
    WallTables w{};
    int n = 0;
    uint32_t masks[12] = {};
    for (int b = 0; b < 4; b++)
        for (int k = 0; k < 6; k++)
            if (TRI_MASK[b][k]) masks[n++] = TRI_MASK[b][k];
    for (int t = 0; t < 36; t++)
        for (int k = 0; k < 12; k++)
            if (masks[k] == RT.tri_mask[t]) {
                w.kind[t] = (uint8_t)k;
                w.corner[k] = RT.tri_own[t];
                w.tri[k] = (uint8_t)t;
            }
    return w;
}
}  // namespace detail
constexpr WallTables WT = detail::make_wall_tables();

struct NullSink {
    DMTZ_HD void operator()(i64) const {}
};

template <class T, class Code = const StarCode*>
struct WallGraph {
    using Rules = LocalRules<T, NullSink, Code>;
    using At = typename Rules::At;
    const Rules& r;
    const WallTables* wt;

    DMTZ_HD i64 corner_offset(int k) const { return (k & 1) + ((k >> 1) & 1) * r.d.W + (k >> 2) * r.d.W * r.d.H; }
    DMTZ_HD uint32_t face_id(At t) const {
        return (uint32_t)((i64)t.v - corner_offset(r.tb->tri_own[t.l])) * 12u + wt->kind[t.l];
    }
    DMTZ_HD At face_at(uint32_t id) const {
        const int k = (int)(id % 12u);
        return At{(uint32_t)((i64)(id / 12u) + corner_offset(wt->corner[k])), wt->tri[k]};
    }
    // The face / edge with a number of the reference.
    DMTZ_HD At face_of_number(i64 n) const {
        i64 a, b, e;
        tri_verts(r.d, r.c, n, a, b, e);
        return At{(uint32_t)a, ST.tri_of[slot_between(r.d, a, b)][slot_between(r.d, a, e)]};
    }
    DMTZ_HD At edge_of_number(i64 n) const {
        i64 a, b;
        edge_verts(r.d, r.c, n, a, b);
        return At{(uint32_t)a, slot_between(r.d, a, b)};
    }

    // An edge's partner in f, when f pairs it, against its partner in g.
    enum Kind { NONE, MISMATCH, FACE, VERTEX };
    DMTZ_HD Kind partner(At e, At& p) const {
        const At ef = r.edge_owner(r.f, e);
        const int nf = Rules::edge_code(r.cf, ef);
        if (nf == 15) return NONE;
        const At eg = r.edge_owner(r.g, e);
        const int ng = Rules::edge_code(r.cg, eg);
        bool same;
        if (nf == 14) p = At{ef.v, 0};
        else p = At{ef.v, r.tb->tri_of[ef.l][nf]};
        if (ng == 15) same = false;
        else if (nf == 14 && ng == 14) same = ef.v == eg.v;
        else if (nf < 14 && ng < 14) same = r.at(ef.v, nf) == r.at(eg.v, ng);
        else if (nf == 14) same = r.tri_number(At{eg.v, r.tb->tri_of[eg.l][ng]}) == (i64)ef.v;
        else same = r.tri_number(p) == (i64)eg.v;
        return !same ? MISMATCH : (nf == 14 ? VERTEX : FACE);
    }

    // The faces around edge e: fn(face).
    template <class Fn>
    DMTZ_HD void faces_of(At e, Fn fn) const {
        i64 x, y, z;
        vxyz(r.d, (i64)e.v, x, y, z);
        for (int k = 0; k < r.tb->adj_n[e.l]; k++) {
            const int s = r.tb->adj_l[e.l][k];
            if (inb(r.d, x + DIR[s][0], y + DIR[s][1], z + DIR[s][2])) fn(At{e.v, r.tb->tri_of[e.l][s]});
        }
    }

    // The mismatched edges that v owns in f (every edge f pairs has one owner): fn(edge).
    template <class Fn>
    DMTZ_HD void mismatched_edges(uint32_t v, Fn fn) const {
        const uint64_t wf = code_word(r.cf, (i64)v, 0), lf = code_word(r.cf, (i64)v, 1) & 0x3FFFull;
        // the same lower slots and partners in g: every edge v owns in f has the same owner and partner
        if (((wf ^ code_word(r.cg, (i64)v, 0)) << 8) == 0 && lf == (code_word(r.cg, (i64)v, 1) & 0x3FFFull)) return;
        for (uint32_t m = (uint32_t)lf; m; m &= m - 1) {
            const At e{v, __builtin_ctz(m)};
            At p;
            if (partner(e, p) == MISMATCH) fn(e);
        }
    }

    // The faces that lead on to face t: fn(face).
    template <class Fn>
    DMTZ_HD void leading_to(At t, Fn fn) const {
        const At o = r.tri_owner(r.f, t);
        const int cc = Rules::tri_code(r.cf, o);
        if (cc >= 4) return;
        At e;
        if (cc < 2) {
            e = At{o.v, cc == 0 ? r.tb->tri_i[o.l] : r.tb->tri_j[o.l]};
        } else {  // paired with a tet: an edge of the tet's number, paired with the vertex of t's
            const At q{o.v, r.tb->tri_q[o.l][cc - 2]};
            if (!r.face_taken_as_vertex(o, q)) return;
            e = edge_of_number(r.tet_number(q));
            const At ef = r.edge_owner(r.f, e);
            if (Rules::edge_code(r.cf, ef) != 14 || (i64)ef.v != r.tri_number(o)) return;
        }
        const uint32_t self = face_id(t);
        faces_of(e, [&](At p) {
            if (face_id(p) != self) fn(p);
        });
    }

    // One step of the chain from open face t: the mismatched edge in e (returns 1), the next open face in
    // t (returns 0), or nothing (returns -1: t is not open). open(id): the face is open.
    template <class Open>
    DMTZ_HD int chain_step(At& t, At& e, Open open) const {
        const uint32_t vi = r.at(t.v, r.tb->tri_i[t.l]), vj = r.at(t.v, r.tb->tri_j[t.l]);
        const int li = r.tb->tri_at[t.l][0];  // t seen from vi: back to v, and on to vj
        const int back = r.tb->tri_i[t.l] ^ 1;
        const int on = r.tb->tri_i[li] == back ? r.tb->tri_j[li] : r.tb->tri_i[li];
        // edges by the vertex they leave out, smallest index first: (v1,v2), (v1,v3), (v2,v3)
        At es[3] = {{t.v, r.tb->tri_i[t.l]}, {t.v, r.tb->tri_j[t.l]}, {vi, on}};
        uint32_t left[3] = {vj, vi, t.v};
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2 - a; b++)
                if (left[b] > left[b + 1]) {
                    const uint32_t x = left[b];
                    left[b] = left[b + 1];
                    left[b + 1] = x;
                    const At y = es[b];
                    es[b] = es[b + 1];
                    es[b + 1] = y;
                }
        const uint32_t self = face_id(t);
        bool any = false;
        At next = t;
        for (int k = 0; k < 3; k++) {
            At p;
            const Kind kind = partner(es[k], p);
            if (kind == MISMATCH) {
                e = es[k];
                return 1;
            }
            if (kind == VERTEX) {
                if (!r.vertex_taken_as_face(p.v, es[k])) continue;
                const FieldGrad<T, Code> F(r.f, r.cf, r.d, r.c);
                if (F.pf((i64)p.v) != r.edge_number(es[k])) continue;
                p = face_of_number((i64)p.v);
            } else if (kind == NONE) {
                continue;
            }
            const uint32_t id = face_id(p);
            if (id != self && open(id)) {
                next = p;
                any = true;
            }
        }
        if (!any) return -1;
        t = next;
        return 0;
    }

    // The chain from open face t to its end: 1 with the mismatched edge in e, -1 from a face that is not
    // open, 0 when it runs in a circle. The next face depends on the face alone, so a chain that meets the
    // face it was at 1, 2, 4, 8, ... steps before never ends; one that ends is followed however long it
    // is. n receives the number of steps.
    template <class Open>
    DMTZ_HD int follow(At t, At& e, Open open, i64& n) const {
        uint32_t mark = face_id(t);
        i64 next = 1;
        for (n = 1;; n++) {
            const int s = chain_step(t, e, open);
            if (s != 0) return s;
            const uint32_t id = face_id(t);
            if (id == mark) return 0;
            if (n == next) {
                mark = id;
                next *= 2;
            }
        }
    }
};

}  // namespace dmtz
