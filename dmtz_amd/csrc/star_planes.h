// The lower-star classifier (lower_star.h) over bit planes: 32 vertices per lane at once.
//
// lower_star.h evaluates the five passes for one vertex with masks over its 14 slots; most of its
// five thousand instructions handle one bit each. Here a 32-bit word holds one condition for 32
// vertices: from the comparisons of each vertex's 15 values on, every step is a bitwise operation on
// such words, and the star codes and masks are transposed back to one vertex per word at the end.
// About 22 thousand instructions for 2048 vertices of a wave instead of 5 thousand for 64.
//
// The passes are those of lower_star.h, cell by cell, in the same order; see there for their meaning.
// A triangle's state is three words: any (paired), b0 and b1 (the low bits of its code), from which
// the T0 claims are read back; a tet is left out at the slot completing the triangle that claims it.
#pragma once
#include <cstring>
#include <utility>

#include "lower_star.h"

namespace dmtz {

constexpr int N_PAIRS = 91;  // pairs of slots i < j
constexpr int pair_index(int i, int j) { return i * 13 - i * (i - 1) / 2 + (j - i - 1); }

// Comparison words of 32 vertices. p[pair_index(i, j)] holds the strict comparison that decides
// whether n_i is below n_j: n_i < n_j, or n_j < n_i where the index order breaks ties towards n_i
// (TB[i] < TB[j]); l[i] the same for n_i and the centre until finish() turns it into "n_i is in the
// grid and below the centre".
struct StarWords {
    uint32_t p[N_PAIRS];
    uint32_t l[14];

    // n_j below n_i
    DMTZ_HD uint32_t bel(int i, int j) const {
        const int a = i < j ? i : j, b = i < j ? j : i;
        const uint32_t q = p[pair_index(a, b)];
        return ((TB[a] < TB[b]) == (a == j)) ? ~q : q;
    }
};

DMTZ_HD float fma_of(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
DMTZ_HD double fma_of(double a, double b, double c) { return __builtin_fma(a, b, c); }

// The sign bit of a - b: a < b (a, b finite, neither -0; subnormal differences are kept).
DMTZ_HD uint32_t sign_word(float a, float b) {
    const float x = a - b;
    uint32_t u;
    memcpy(&u, &x, 4);
    return u;
}
DMTZ_HD uint32_t sign_word(double a, double b) {
    const double x = a - b;
    uint64_t u;
    memcpy(&u, &x, 8);
    return (uint32_t)(u >> 32);
}
// The words move up by one bit and take the comparison in: one subtraction and one funnel shift.
DMTZ_HD uint32_t push_sign(uint32_t w, uint32_t sign) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_alignbit(w, sign, 31);
#else
    return (w << 1) | (sign >> 31);
#endif
}

namespace detail {
template <int I, int J>
struct WordLoop {
    template <class T>
    DMTZ_HD static void run(const T* val, StarWords& w) {
        uint32_t& x = w.p[pair_index(I, J)];
        x = push_sign(x, TB[I] < TB[J] ? sign_word(val[J], val[I]) : sign_word(val[I], val[J]));
        if constexpr (J + 1 < 14) WordLoop<I, J + 1>::run(val, w);
        else if constexpr (I + 2 < 14) WordLoop<I + 1, I + 2>::run(val, w);
    }
};
template <int I>
struct WordCentreLoop {
    template <class T>
    DMTZ_HD static void run(const T* val, StarWords& w) {
        w.l[I] = push_sign(w.l[I], TB[I] < TB[14] ? sign_word(val[14], val[I]) : sign_word(val[I], val[14]));
        if constexpr (I + 1 < 14) WordCentreLoop<I + 1>::run(val, w);
    }
};

// The same two for values of which some are infinite or NaN: their differences have no sign to go by, so
// the bits are the comparisons of lower_star.h (below).
template <int I, int J>
struct WordLoopAny {
    template <class T>
    DMTZ_HD static void run(const T* val, StarWords& w) {
        uint32_t& x = w.p[pair_index(I, J)];
        x = (x << 1) | (uint32_t)(below<T, I, J>(val) != (TB[I] < TB[J]));
        if constexpr (J + 1 < 14) WordLoopAny<I, J + 1>::run(val, w);
        else if constexpr (I + 2 < 14) WordLoopAny<I + 1, I + 2>::run(val, w);
    }
};
template <int I>
struct WordCentreLoopAny {
    template <class T>
    DMTZ_HD static void run(const T* val, StarWords& w) {
        w.l[I] = (w.l[I] << 1) | (uint32_t)(below<T, I, 14>(val) != (TB[I] < TB[14]));
        if constexpr (I + 1 < 14) WordCentreLoopAny<I + 1>::run(val, w);
    }
};

// fn(0), ..., fn(N - 1) with compile-time arguments: the passes below are too long for the unroller,
// and an index that is not a constant would put their words into memory.
#if defined(__HIPCC__)
#define DMTZ_INLINE_LAMBDA __attribute__((always_inline))
#else
#define DMTZ_INLINE_LAMBDA
#endif
template <class Fn, int... I>
DMTZ_HD void each_of(std::integer_sequence<int, I...>, Fn fn) {
    (fn(std::integral_constant<int, I>{}), ...);
}
template <int N, class Fn>
DMTZ_HD void each(Fn fn) {
    each_of(std::make_integer_sequence<int, N>{}, fn);
}

template <int S>
DMTZ_HD void transpose_step(uint32_t* a) {
    constexpr uint32_t m = S == 16 ? 0x0000ffffu : S == 8 ? 0x00ff00ffu : S == 4 ? 0x0f0f0f0fu : S == 2 ? 0x33333333u : 0x55555555u;
#pragma unroll
    for (int k = 0; k < 32; k++)
        if (!(k & S)) {
            const uint32_t x = a[k], y = a[k + S];
            a[k] = (x & m) | ((y << S) & ~m);
            a[k + S] = ((x >> S) & m) | (y & ~m);
        }
}
}  // namespace detail

// Shift the comparisons of one more vertex's values into the words (the last vertex is bit 0). The
// values are finite; a slot outside the grid may hold any of them.
template <class T>
DMTZ_HD void add_vertex(const T* val, StarWords& w) {
    T v[15];
#pragma unroll
    for (int k = 0; k < 15; k++) v[k] = val[k] + (T)0;  // -0 to +0: equal values have no sign
    detail::WordLoop<0, 1>::run(v, w);
    detail::WordCentreLoop<0>::run(v, w);
}

// The same for any values, by comparisons.
template <class T>
DMTZ_HD void add_vertex_any(const T* val, StarWords& w) {
    detail::WordLoopAny<0, 1>::run(val, w);
    detail::WordCentreLoopAny<0>::run(val, w);
}

// After the last vertex: side[2 a] and side[2 a + 1] say for which vertices the grid goes on down and
// up axis a; slots outside it are below nothing.
DMTZ_HD void finish(StarWords& w, const uint32_t* side) {
#pragma unroll
    for (int k = 0; k < 14; k++) {
        uint32_t x = TB[k] < TB[14] ? ~w.l[k] : w.l[k];
#pragma unroll
        for (int a = 0; a < 3; a++)
            if (DIR[k][a] != 0) x &= side[2 * a + (DIR[k][a] > 0)];
        w.l[k] = x;
    }
}

constexpr int PLANE_ROWS = 32;
constexpr i64 PLANE_TILE = 64 * PLANE_ROWS;

// 64 vertices further in coordinates: at most one carry per axis.
struct Step64 {
    int x, y, z;
    DMTZ_HD explicit Step64(const Dims& d)
        : x((int)(64 % d.W)), y((int)(64 / d.W % d.H)), z((int)(64 / (d.W * d.H))) {}
};

// The comparison words of one lane of a wave's tile: lane l of the tile at vertex base takes the vertices
// v0 + 64 b, v0 = base + l. The next row's values are loaded while a row is compared; a neighbour's
// index is only kept inside the field, since finish() drops the slots outside the grid. The tile's values
// gather in a sum of zeros, which an infinity or a NaN makes a NaN: a lane that met one takes its rows
// again with comparisons (15 multiply-adds a row, 2 % of the pass's instructions).
template <class T>
DMTZ_HD void tile_words(const T* fld, const Dims& d, const Step64& st, i64 n, i64 v0, StarWords& w) {
    const int W = (int)d.W, H = (int)d.H, D = (int)d.D, last = (int)(n - 1);
    i64 x64, y64, z64;
    vxyz(d, v0 <= last ? v0 : last, x64, y64, z64);
    int x = (int)x64, y = (int)y64, z = (int)z64;
    uint32_t v = (uint32_t)v0;  // v0 < n + PLANE_TILE < 2^32
    int32_t off[14];
#pragma unroll
    for (int k = 0; k < 14; k++) off[k] = (int32_t)slot_step(d, k);
    uint32_t side[6] = {0, 0, 0, 0, 0, 0};
    auto load = [&](T* val) {
        const uint32_t u = v < (uint32_t)last ? v : (uint32_t)last;
#pragma unroll
        for (int k = 0; k < 14; k++) {
            uint32_t q;
            if (k & 1) {  // odd slots lead down
                const int t = (int)u + off[k];
                q = t < 0 ? 0u : (uint32_t)t;
            } else {
                const uint32_t t = u + (uint32_t)off[k];
                q = t < (uint32_t)last ? t : (uint32_t)last;
            }
            val[k] = fld[q];
        }
        val[14] = fld[u];
        v += 64;
    };
    T zero = 0;
    auto sides = [&]() {
        side[0] = (side[0] << 1) | (uint32_t)(x > 0);
        side[1] = (side[1] << 1) | (uint32_t)(x < W - 1);
        side[2] = (side[2] << 1) | (uint32_t)(y > 0);
        side[3] = (side[3] << 1) | (uint32_t)(y < H - 1);
        side[4] = (side[4] << 1) | (uint32_t)(z > 0);
        side[5] = (side[5] << 1) | (uint32_t)(z < D - 1);
        x += st.x;
        const int cx = x >= W;
        x -= cx ? W : 0;
        y += st.y + cx;
        const int cy = y >= H;
        y -= cy ? H : 0;
        z += st.z + cy;
    };
#pragma unroll
    for (int k = 0; k < N_PAIRS; k++) w.p[k] = 0;
#pragma unroll
    for (int k = 0; k < 14; k++) w.l[k] = 0;
    T cur[15], nxt[15];
    load(cur);
#pragma unroll 1
    for (int b = 0; b < PLANE_ROWS; b++) {
        load(nxt);  // past the last row: not used
        sides();
        add_vertex(cur, w);
#pragma unroll
        for (int k = 0; k < 15; k++) {
            zero = fma_of(cur[k], (T)0, zero);
            cur[k] = nxt[k];
        }
    }
    if (__builtin_expect(zero != zero, 0)) {
        v = (uint32_t)v0;
#pragma unroll 1
        for (int b = 0; b < PLANE_ROWS; b++) {  // 32 bits are pushed: nothing of the words before is left
            load(cur);
            add_vertex_any(cur, w);
        }
    }
    finish(w, side);
}

// 32 x 32 bit transpose in place: bit p of a[r] becomes bit r of a[p].
DMTZ_HD void transpose32(uint32_t* a) {
    detail::transpose_step<16>(a);
    detail::transpose_step<8>(a);
    detail::transpose_step<4>(a);
    detail::transpose_step<2>(a);
    detail::transpose_step<1>(a);
}

namespace detail {
// Word 2 + K of the star codes, from the triangles' state.
template <int K>
DMTZ_HD void tri_planes(const uint32_t* any, const uint32_t* b0, const uint32_t* b1, uint32_t* lo, uint32_t* hi) {
#pragma unroll
    for (int b = 0; b < 64; b++) {
        const int t = 21 * K + b / 3;
        uint32_t x = 0;
        if (b < 63 && t < 36) x = (b % 3 == 0 ? b0[t] : b % 3 == 1 ? b1[t] : 0u) | ~any[t];
        if (b < 32) lo[b] = x;
        else hi[b - 32] = x;
    }
    transpose32(lo);
    transpose32(hi);
}
}  // namespace detail

// The classification of 32 vertices. out receives, per vertex (index = bit of the words):
//   code(k, lo, hi)              halves of word k of the star code (lo[32], hi[32])
//   masks_lo(c0, c1, i0, i1)     owned critical cells (c) and members (i), cells 0-31 and 32-50
//   masks_hi(c2, i2)             the same for the tets
// in the order code(0), code(1), code(2), code(3), masks_lo, masks_hi.
template <class Out>
DMTZ_HD void classify_words(const StarWords& w, Out& out) {
    const uint32_t* L = w.l;
    // V: one-hot steepest slot
    uint32_t S[14], any_below = 0;
    detail::each<14>([&](auto k_) DMTZ_INLINE_LAMBDA {
        constexpr int k = decltype(k_)::value;
        uint32_t m = L[k];
#pragma unroll
        for (int j = 0; j < 14; j++)
            if (j != k) m &= ~(L[j] & w.bel(k, j));
        S[k] = m;
        any_below |= L[k];
    });
    const uint32_t none = ~any_below;

    // The lowest candidates of edge a among its link: E0 below n_a, E1 above it.
    auto lowest = [&](auto a_, bool e1, uint32_t* m) DMTZ_INLINE_LAMBDA {
        constexpr int a = decltype(a_)::value;
        uint32_t c[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int x = 0; x < 6; x++)
            if (x < ST.adj_n[a]) {
                const int k = ST.adj_l[a][x];
                c[x] = L[k] & (e1 ? ~w.bel(a, k) : w.bel(a, k));
            }
#pragma unroll
        for (int x = 0; x < 6; x++) {
            m[x] = c[x];
#pragma unroll
            for (int y = 0; y < 6; y++)
                if (y != x && x < ST.adj_n[a] && y < ST.adj_n[a]) m[x] &= ~(c[y] & w.bel(ST.adj_l[a][x], ST.adj_l[a][y]));
        }
    };

    uint32_t any[36], b0[36], b1[36];
#pragma unroll
    for (int t = 0; t < 36; t++) any[t] = b0[t] = b1[t] = 0;
    uint32_t pe[14];  // edges paired in E0, then with the centre or in any pass
    detail::each<14>([&](auto a_) DMTZ_INLINE_LAMBDA {
        constexpr int a = decltype(a_)::value;
        uint32_t m[6];
        lowest(a_, false, m);
        const uint32_t on = L[a] & ~S[a];
        pe[a] = 0;
#pragma unroll
        for (int x = 0; x < 6; x++)
            if (x < ST.adj_n[a]) {
                const int t = ST.adj_t[a][x];
                const uint32_t sel = m[x] & on;
                pe[a] |= sel;
                any[t] |= sel;
                if (ST.tri_j[t] == a) b0[t] |= sel;
            }
    });

    // T0
    detail::each<36>([&](auto t_) DMTZ_INLINE_LAMBDA {
        constexpr int t = decltype(t_)::value;
        const int i = ST.tri_i[t], j = ST.tri_j[t], k0 = ST.tri_k[t][0], k1 = ST.tri_k[t][1];
        const uint32_t c0 = L[k0] & w.bel(i, k0) & w.bel(j, k0), c1 = L[k1] & w.bel(i, k1) & w.bel(j, k1);
        const uint32_t fr = L[i] & L[j] & ~any[t];
        const uint32_t p1 = fr & c1 & (~c0 | w.bel(k0, k1)), p0 = fr & c0 & ~p1;
        b0[t] |= p1;
        b1[t] = p0 | p1;
        any[t] |= p0 | p1;
    });

    // E1, and the edges' partner nibbles (15 = none, 14 = the centre, else the slot of E0 or E1)
    uint32_t lo[32], hi[32];
#pragma unroll
    for (int k = 0; k < 32; k++) lo[k] = hi[k] = 0;
    detail::each<14>([&](auto a_) DMTZ_INLINE_LAMBDA {
        constexpr int a = decltype(a_)::value;
        uint32_t m0[6], m1[6];
        lowest(a_, false, m0);
        lowest(a_, true, m1);
        const uint32_t on0 = L[a] & ~S[a], on1 = on0 & ~pe[a];
        uint32_t nib[4] = {0, S[a], S[a], S[a]}, paired = S[a] | pe[a];
#pragma unroll
        for (int x = 0; x < 6; x++)
            if (x < ST.adj_n[a]) {
                const int k = ST.adj_l[a][x], t = ST.adj_t[a][x];
                const uint32_t s1 = m1[x] & on1 & ~any[t];
                const uint32_t s = (m0[x] & on0) | s1;
                any[t] |= s1;  // the triangle's other edge cannot choose it: n_k is above n_a
                if (ST.tri_j[t] == a) b0[t] |= s1;
                paired |= s1;
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if ((k >> q) & 1) nib[q] |= s;
            }
        pe[a] = paired;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t x = nib[q] | ~paired;
            if (a < 8) lo[4 * a + q] = x;
            else hi[4 * (a - 8) + q] = x;
        }
    });
    detail::each<4>([&](auto q_) DMTZ_INLINE_LAMBDA {
        constexpr int q = decltype(q_)::value;
        uint32_t x = none;
#pragma unroll
        for (int k = 0; k < 14; k++)
            if ((k >> q) & 1) x |= S[k];
        hi[24 + q] = x;
    });
    transpose32(lo);
    transpose32(hi);
    out.code(0, lo, hi);

    // T1; q0, q1, q2: the tet leaves out that slot of tet_s[q]
    uint32_t qc[24][3];
#pragma unroll
    for (int q = 0; q < 24; q++)
#pragma unroll
        for (int c = 0; c < 3; c++) qc[q][c] = 0;
    auto claim = [&](int t, int x, uint32_t p) DMTZ_INLINE_LAMBDA {
        const int q = ST.tri_q[t][x], k = ST.tri_k[t][x];
#pragma unroll
        for (int c = 0; c < 3; c++)
            if (ST.tet_s[q][c] == k) qc[q][c] |= p;
    };
    detail::each<36>([&](auto t_) DMTZ_INLINE_LAMBDA {
        constexpr int t = decltype(t_)::value;
        claim(t, 0, b1[t] & ~b0[t]);
        claim(t, 1, b1[t] & b0[t]);
    });
    uint32_t qt0[24];
#pragma unroll
    for (int q = 0; q < 24; q++) qt0[q] = qc[q][0] | qc[q][1] | qc[q][2];
    detail::each<36>([&](auto t_) DMTZ_INLINE_LAMBDA {
        constexpr int t = decltype(t_)::value;
        const int i = ST.tri_i[t], j = ST.tri_j[t], k0 = ST.tri_k[t][0], k1 = ST.tri_k[t][1];
        const uint32_t c0 = L[k0] & (w.bel(i, k0) ^ w.bel(j, k0)), c1 = L[k1] & (w.bel(i, k1) ^ w.bel(j, k1));
        const uint32_t fr = L[i] & L[j] & ~any[t];
        const uint32_t pick1 = c1 & (~c0 | w.bel(k0, k1)), pick0 = c0 & ~pick1;
        const uint32_t p1 = fr & pick1 & ~qt0[ST.tri_q[t][1]], p0 = fr & pick0 & ~qt0[ST.tri_q[t][0]];
        claim(t, 0, p0);
        claim(t, 1, p1);
        b0[t] |= p1;
        b1[t] |= p0 | p1;
        any[t] |= p0 | p1;
    });

    // word 1: L, then two bits per tet (3 = unpaired)
    uint32_t qany[24];
#pragma unroll
    for (int k = 0; k < 14; k++) lo[k] = L[k];
    detail::each<24>([&](auto q_) DMTZ_INLINE_LAMBDA {
        constexpr int q = decltype(q_)::value;
        qany[q] = qc[q][0] | qc[q][1] | qc[q][2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int bit = 14 + 2 * q + c;
            const uint32_t x = qc[q][1 + c] | ~qany[q];
            if (bit < 32) lo[bit] = x;
            else hi[bit - 32] = x;
        }
    });
    hi[30] = hi[31] = 0;
    transpose32(lo);
    transpose32(hi);
    out.code(1, lo, hi);

    // words 2 and 3: three bits per triangle (7 = unpaired)
    detail::tri_planes<0>(any, b0, b1, lo, hi);
    out.code(2, lo, hi);
    detail::tri_planes<1>(any, b0, b1, lo, hi);
    out.code(3, lo, hi);

    // masks over the local cells
    uint32_t i0[32], i1[32];
    detail::each<64>([&](auto lc_) DMTZ_INLINE_LAMBDA {
        constexpr int lc = decltype(lc_)::value;
        uint32_t in = 0, crit = 0;
        if (lc == LC_VERT) {
            in = ~0u;
            crit = none;
        } else if (lc < LC_TRI) {
            in = L[lc - LC_EDGE];
            crit = in & ~pe[lc - LC_EDGE];
        } else if (lc < LC_TET) {
            const int t = lc - LC_TRI;
            in = L[ST.tri_i[t]] & L[ST.tri_j[t]];
            crit = in & ~any[t];
        }
        if (lc < 32) {
            lo[lc] = crit;
            i0[lc] = in;
        } else {
            hi[lc - 32] = crit;
            i1[lc - 32] = in;
        }
    });
    transpose32(lo);
    transpose32(hi);
    transpose32(i0);
    transpose32(i1);
    out.masks_lo(lo, hi, i0, i1);
    detail::each<32>([&](auto q_) DMTZ_INLINE_LAMBDA {
        constexpr int q = decltype(q_)::value;
        lo[q] = i0[q] = 0;
        if (q < 24) {
            i0[q] = L[ST.tet_s[q][0]] & L[ST.tet_s[q][1]] & L[ST.tet_s[q][2]];
            lo[q] = i0[q] & ~qany[q];
        }
    });
    transpose32(lo);
    transpose32(i0);
    out.masks_hi(lo, i0);
}

}  // namespace dmtz
