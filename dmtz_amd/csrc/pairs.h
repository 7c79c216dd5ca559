// Pair words: the pairings that separatrix walks follow, four bytes per vertex.
//
// A walk along a V-path asks one question per step: which face is this tet paired with (ascending
// paths, is_false main_3d.cu:4437-4497, get_paired_id :4499-4537), or which edge is this vertex
// paired with (descending paths, main_3d.cu:4613-4687, 4961-5062). Answered from the star codes, a
// step decodes a global id, compares four values to find the tet's owner and reads the owner's
// code: two dependent reads and some hundred instructions. The pair word of vertex v answers both
// kinds of question with one 4-byte read:
//   bits 3t .. 3t+2   tet of type t of the cube anchored at v: which of its four corners (in
//                     increasing corner order) its paired face leaves out, 4 = unpaired or no cube
//   bits 18 .. 21     slot of the edge v is paired with, 15 = none (a minimum)
// Words are built by one dense pass over the codes, and a walk then moves from tet to tet through
// a 24-entry table (the tet across the face opposite each corner).
#pragma once
#include "gradient.h"

namespace dmtz {

constexpr uint32_t PW_NONE = 4;       // a tet without a paired face
constexpr int PW_SLOT_SHIFT = 18;     // the vertex's steepest slot
constexpr uint32_t PW_NO_SLOT = 15;

struct PairTables {
    uint8_t corner[6][4];     // corners of tet type t, increasing (so by increasing vertex index)
    uint8_t lq_shift[6][4];   // the owner at corner position p: bit position of the tet's field in code word 1
    uint8_t out_of[6][4][4];  // the owner at position p, field value c: position of the left-out corner
    // across[4 t + p]: the tet across the face opposite corner position p of type t.
    // bits 0-2 its type, bits 3-4 the axis to move along (3: same cube), bit 5 the direction (1: up)
    uint8_t across[24];
    // start[t][k]: cofacet tet k (in the reference's search order, main_3d.cu:4380-4426) of star
    // triangle t of a vertex v: bits 0-2 type, bits 3-5 v's corner number in the tet's cube
    uint8_t start[36][2];
};

namespace detail {
constexpr int corner_slot(int a, int b) {  // slot of corner b seen from corner a of one cube
    const int dx = (b & 1) - (a & 1), dy = ((b >> 1) & 1) - ((a >> 1) & 1), dz = ((b >> 2) & 1) - ((a >> 2) & 1);
    return ST.slot_of[(dx + 1) * 9 + (dy + 1) * 3 + (dz + 1)];
}
constexpr int tet_of_slots(int a, int b, int c) {
    const uint32_t key = (1u << a) | (1u << b) | (1u << c);
    for (int q = 0; q < 24; q++)
        if (((1u << ST.tet_s[q][0]) | (1u << ST.tet_s[q][1]) | (1u << ST.tet_s[q][2])) == key) return q;
    return -1;
}
constexpr int tet_type_of_mask(uint32_t m) {
    for (int k = 0; k < 6; k++)
        if (TET_MASK[k] == m) return k;
    return -1;
}

constexpr PairTables make_pair_tables() {
    PairTables r{};
    for (int t = 0; t < 6; t++) {
        int n = 0;
        for (int k = 0; k < 8; k++)
            if ((TET_MASK[t] >> k) & 1) r.corner[t][n++] = (uint8_t)k;
        for (int p = 0; p < 4; p++) {
            int slot[4] = {-1, -1, -1, -1}, o[3] = {0, 0, 0}, m = 0;
            for (int j = 0; j < 4; j++)
                if (j != p) {
                    slot[j] = corner_slot(r.corner[t][p], r.corner[t][j]);
                    o[m++] = j;
                }
            const int q = tet_of_slots(slot[o[0]], slot[o[1]], slot[o[2]]);
            r.lq_shift[t][p] = (uint8_t)(14 + 2 * q);
            for (int c = 0; c < 3; c++)
                for (int j = 0; j < 4; j++)
                    if (j != p && slot[j] == ST.tet_s[q][c]) r.out_of[t][p][c] = (uint8_t)j;
            r.out_of[t][p][3] = (uint8_t)PW_NONE;
            // the tet across the face opposite corner p: the only other tet of the surrounding
            // cubes with the face's three corners
            uint32_t face = 0;
            for (int j = 0; j < 4; j++)
                if (j != p) face |= 1u << r.corner[t][j];
            uint8_t found = 0xFF;
            for (int k = 0; k < 6; k++)
                if (k != t && (TET_MASK[k] & face) == face) found = (uint8_t)(k | (3 << 3));
            for (int axis = 0; axis < 3; axis++)
                for (int up = 0; up < 2; up++) {
                    // the face lies in the plane of that side; its corners in the next cube
                    uint32_t moved = 0;
                    bool ok = true;
                    for (int k = 0; k < 8; k++)
                        if ((face >> k) & 1) {
                            ok = ok && ((k >> axis) & 1) == up;
                            moved |= 1u << (k ^ (1 << axis));
                        }
                    if (!ok) continue;
                    for (int k = 0; k < 6; k++)
                        if ((TET_MASK[k] & moved) == moved) found = (uint8_t)(k | (axis << 3) | (up << 5));
                }
            r.across[4 * t + p] = found;
        }
    }
    for (int t = 0; t < 36; t++) {
        // the triangle's vertex of largest index, from which the search starts
        const int sl[3] = {14, ST.tri_i[t], ST.tri_j[t]};
        int base = 0;
        for (int k = 1; k < 3; k++)
            if (TB[sl[k]] > TB[sl[base]]) base = k;
        int off[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
        for (int k = 0; k < 3; k++)
            for (int a = 0; a < 3; a++) off[k][a] = sl[k] == 14 ? 0 : DIR[sl[k]][a];
        int s[2] = {0, 0}, n = 0;
        for (int k = 0; k < 3; k++)
            if (k != base)
                s[n++] = ST.slot_of[(off[k][0] - off[base][0] + 1) * 9 + (off[k][1] - off[base][1] + 1) * 3 +
                                    (off[k][2] - off[base][2] + 1)];
        const int lt = ST.tri_of[s[0]][s[1]];
        for (int c = 0; c < 2; c++) {
            const int k4 = ST.tri_k[lt][c];
            int v[4][3] = {};
            for (int k = 0; k < 3; k++)
                for (int a = 0; a < 3; a++) v[k][a] = off[k][a];
            for (int a = 0; a < 3; a++) v[3][a] = off[base][a] + DIR[k4][a];
            int mn[3] = {v[0][0], v[0][1], v[0][2]};
            for (int k = 1; k < 4; k++)
                for (int a = 0; a < 3; a++) mn[a] = v[k][a] < mn[a] ? v[k][a] : mn[a];
            uint32_t mask = 0;
            for (int k = 0; k < 4; k++)
                mask |= 1u << ((v[k][0] - mn[0]) + 2 * (v[k][1] - mn[1]) + 4 * (v[k][2] - mn[2]));
            const int own = (-mn[0]) + 2 * (-mn[1]) + 4 * (-mn[2]);
            r.start[t][c] = (uint8_t)(tet_type_of_mask(mask) | (own << 3));
        }
    }
    return r;
}
}  // namespace detail

constexpr PairTables PT = detail::make_pair_tables();

// Fields of the pair word of the six tets of the cube with corner values val[8] and corner codes'
// second words w1[8]. Ties between corners go to the larger index, the later corner.
template <class T>
DMTZ_HD uint32_t cube_pairs(const T* val, const uint64_t* w1) {
    uint32_t word = 0;
#pragma unroll
    for (int t = 0; t < 6; t++) {
        T mv = val[PT.corner[t][0]];
        uint64_t mw = w1[PT.corner[t][0]];
        uint32_t p = 0;
#pragma unroll
        for (int j = 1; j < 4; j++) {
            const T x = val[PT.corner[t][j]];
            const bool up = x >= mv;
            mv = up ? x : mv;
            mw = up ? w1[PT.corner[t][j]] : mw;
            p = up ? (uint32_t)j : p;
        }
        uint32_t shifts = 0;
        uint64_t outs = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            shifts |= (uint32_t)PT.lq_shift[t][j] << (8 * j);
#pragma unroll
            for (int c = 0; c < 4; c++) outs |= (uint64_t)PT.out_of[t][j][c] << (12 * j + 3 * c);
        }
        const uint32_t c = (uint32_t)(mw >> ((shifts >> (8 * p)) & 63u)) & 3u;
        word |= ((uint32_t)(outs >> (12 * p + 3 * c)) & 7u) << (3 * t);
    }
    return word;
}
constexpr uint32_t PW_NO_CUBE = PW_NONE * 0x9249u;  // six unpaired tets

// Pair word of vertex v (coordinates x, y, z) from a field and its star codes.
template <class T, class Code>
DMTZ_HD uint32_t pair_word(const T* fld, const Code& code, const Dims& d, i64 v, i64 x, i64 y, i64 z) {
    uint32_t word = PW_NO_CUBE;
    if (x < d.W - 1 && y < d.H - 1 && z < d.D - 1) {
        T val[8];
        uint64_t w1[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const i64 u = v + (k & 1) + ((k >> 1) & 1) * d.W + ((k >> 2) & 1) * d.W * d.H;
            val[k] = fld[u];
            w1[k] = code_word(code, u, 1);
        }
        word = cube_pairs(val, w1);
    }
    return word | (uint32_t)partner_slot_of(code, v) << PW_SLOT_SHIFT;
}

DMTZ_HD uint32_t pw_out(uint32_t word, int type) { return (word >> (3 * type)) & 7u; }
DMTZ_HD uint32_t pw_slot(uint32_t word) { return (word >> PW_SLOT_SHIFT) & 15u; }

// Where the pairings of f and g differ at v: bits 0-5 the tets of v's cube, bit 6 the vertex's edge
// when f pairs the vertex (an ascending path of f compares its tets, a descending one its
// vertices, and neither compares an unpaired cell of f: main_3d.cu:4453, 4849-4861).
DMTZ_HD uint32_t pair_mismatch(uint32_t wf, uint32_t wg) {
    uint32_t x = wf ^ wg;
    x |= (x >> 1) | (x >> 2);
    uint32_t m = 0;
#pragma unroll
    for (int t = 0; t < 6; t++) m |= ((x >> (3 * t)) & 1u) << t;
    const uint32_t sf = pw_slot(wf);
    return m | (uint32_t)(sf != PW_NO_SLOT && sf != pw_slot(wg)) << 6;
}
constexpr uint32_t MIS_SLOT = 1u << 6;

// A tet: the vertex its cube is anchored at, with its coordinates, and its type. v < 0: no tet.
struct TetAt {
    i64 v;
    int x, y, z, type;
};

DMTZ_HD i64 tet_id_at(const Dims& d, const TetAt& a) {
    return 6 * ((i64)a.z * (d.W - 1) * (d.H - 1) + (i64)a.y * (d.W - 1) + a.x) + a.type;
}
// The tet of a type in the cube anchored at v.
DMTZ_HD i64 tet_id_of_vertex(const Dims& d, i64 v, int type) {
    i64 x, y, z;
    vxyz(d, v, x, y, z);
    return 6 * (z * (d.W - 1) * (d.H - 1) + y * (d.W - 1) + x) + type;
}

// Cofacet tet k of star triangle lt of vertex v at (x, y, z); entry = PT.start[lt][k].
DMTZ_HD TetAt start_tet(const Dims& d, i64 v, int x, int y, int z, uint32_t entry) {
    TetAt a;
    const int own = (int)(entry >> 3);
    a.type = (int)(entry & 7u);
    a.x = x - (own & 1);
    a.y = y - ((own >> 1) & 1);
    a.z = z - ((own >> 2) & 1);
    const bool in = a.x >= 0 && a.y >= 0 && a.z >= 0 && a.x < d.W - 1 && a.y < d.H - 1 && a.z < d.D - 1;
    a.v = in ? v - (own & 1) - ((own >> 1) & 1) * d.W - ((own >> 2) & 1) * d.W * d.H : -1;
    return a;
}

// Move to the tet across the face that leaves out corner position out of a; entry =
// PT.across[4 * a.type + out]. a.v = -1 when the face lies on the grid's boundary.
DMTZ_HD void cross_face(const Dims& d, TetAt& a, uint32_t entry) {
    a.type = (int)(entry & 7u);
    const uint32_t axis = (entry >> 3) & 3u;
    if (axis == 3u) return;
    const int s = (entry & 32u) ? 1 : -1;
    a.x += axis == 0u ? s : 0;
    a.y += axis == 1u ? s : 0;
    a.z += axis == 2u ? s : 0;
    const bool in = a.x >= 0 && a.y >= 0 && a.z >= 0 && a.x < d.W - 1 && a.y < d.H - 1 && a.z < d.D - 1;
    const i64 st = axis == 0u ? 1 : (axis == 1u ? d.W : d.W * d.H);
    a.v = in ? a.v + s * st : -1;
}

// The ascending path of the field with pair words pw from tet a, one step: false when the tet is
// unpaired (the path ends at it); otherwise moves a across the paired face (a.v = -1: off the
// grid) and returns true. (The face's other chain tests of main_3d.cu:4466-4489 always hold: a
// tet and its face are paired in one step of the gradient, each with the other.)
DMTZ_HD bool ascend(const Dims& d, const uint32_t* pw, const uint8_t* across, TetAt& a) {
    const uint32_t out = pw_out(pw[a.v], a.type);
    if (out == PW_NONE) return false;
    cross_face(d, a, across[4 * a.type + (int)out]);
    return true;
}

// The same tet as a number that is equal for equal tets, -1 for no tet.
DMTZ_HD i64 tet_handle(const TetAt& a) { return a.v < 0 ? -1 : a.v * 8 + a.type; }

// get_paired_id (main_3d.cu:4499-4537): the tet reached from a along pw's ascending path, as a
// handle; -1 when the path leaves the grid or a is no tet.
DMTZ_HD i64 paired_max(const Dims& d, const uint32_t* pw, const uint8_t* across, TetAt a, i64 cap, bool& overflow) {
    i64 n = 0;
    bool more = a.v >= 0;
    while (more) {
        more = ascend(d, pw, across, a) && a.v >= 0;
        if (more && ++n > cap) {
            overflow = true;
            more = false;
        }
    }
    return tet_handle(a);
}

// is_false (main_3d.cu:4437-4497): the first tet of f's ascending path from a whose f and g
// partners differ, in div; false when there is none.
DMTZ_HD bool path_mismatch(const Dims& d, const uint32_t* pf, const uint32_t* pg, const uint8_t* across, TetAt a,
                           i64 cap, TetAt& div, bool& overflow) {
    i64 n = 0;
    bool more = a.v >= 0, found = false;
    while (more) {
        const uint32_t out = pw_out(pf[a.v], a.type);
        if (out == PW_NONE) {
            more = false;
        } else if (out != pw_out(pg[a.v], a.type)) {
            div = a;
            found = true;
            more = false;
        } else {
            cross_face(d, a, across[4 * a.type + (int)out]);
            more = a.v >= 0;
            if (more && ++n > cap) {
                overflow = true;
                more = false;
            }
        }
    }
    return found;
}

// get_orginal_saddle_min_pairs (main_3d.cu:4613-4687): the minimum reached from vertex v. step[s] =
// slot_step of slot s.
DMTZ_HD i64 paired_min(const uint32_t* pw, const i64* step, i64 v, i64 cap, bool& overflow) {
    i64 n = 0;
    for (uint32_t s = pw_slot(pw[v]); s != PW_NO_SLOT && !overflow; s = pw_slot(pw[v])) {
        v += step[s];
        if (++n > cap) overflow = true;
    }
    return v;
}

// One endpoint of get_false_ds_vpath_connectivity (main_3d.cu:4961-5062): the minimum g's
// descending path reaches from v; trouble (kept when already set) = the first vertex on it whose
// f and g edges differ.
DMTZ_HD i64 g_min_of(const uint32_t* pf, const uint32_t* pg, const i64* step, i64 v, i64& trouble, i64 cap,
                     bool& overflow) {
    i64 n = 0;
    for (uint32_t s = pw_slot(pg[v]); s != PW_NO_SLOT && !overflow; s = pw_slot(pg[v])) {
        if (trouble == -1 && pw_slot(pf[v]) != s) trouble = v;
        v += step[s];
        if (++n > cap) overflow = true;
    }
    return v;
}

}  // namespace dmtz
