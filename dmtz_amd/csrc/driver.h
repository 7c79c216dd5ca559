// driver.h: device kernels, the context and the host driver of the topology-correction path,
// shared by the library's translation units (dmtz_core.hip: contexts; dmtz_f32.hip and
// dmtz_f64.hip: the entry points of include/dmtz.h per field type). Everything here has internal
// linkage, so each unit compiles the templates it instantiates.
//
// MI355X (gfx950) implementation of the DMTz topology-correction path behind include/dmtz.h.
//
// Device work (one HIP stream per context):
//   k_code, k_code_g, k_code_planes
//                 lower star of every vertex -> 32-byte star code (the gradient of
//                 main_3d.cu:1930-2316 restricted to each vertex's lower star), a thread per vertex
//                 or, on large grids, over bit planes
//   k_critf_gather  f-critical status of the 75 local cells of every vertex (once per run)
//   k_detect      mismatch records from the g star codes and the f-critical masks
//                 (get_false_* main_3d.cu:2492-2550), 4 typed lists
//   k_fix_cp      repair rules over a record list -> edit set (main_3d.cu:2554-4303)
//   k_apply, k_apply_marked
//                 epsilon-checked edit of the edit set (applyDeltaBuffer1 main_3d.cu:1122-1164),
//                 listed or marked
//   k_dirty (or k_dirty_mark + k_dirty_collect), k_code_list_g
//                 re-evaluation of the g star codes around the vertices whose value changed
//   k_fcrit       f-critical cells (for separatrix checks and filtration)
//   k_pairs, k_as_walk, k_mism_full / k_mism_marked, k_as_bad + k_as_list, k_ds_list
//                 separatrix checks, geometry (main_3d.cu:4437-4497, 4837-4959)
//   k_labels, k_as_branch + k_as_combine, k_ds_branch + k_ds_combine
//                 separatrix checks, connectivity (main_3d.cu:4499-4835, 4961-5062)
//   k_wall_seeds, k_wall_level, k_wall_levels, k_wall_chain, k_ds_wall
//                 2-saddle walls (main_3d.cu:5064-5133)
//   k_fix_paths   separatrix and wall repairs (main_3d.cu:5135-5413)
//   k_pin         filtration (main_3d.cu:2405-2490)
//   k_zone_cells, k_zone, k_snap_boxes, k_tie_mark, k_tie_raise, k_freeze_all
//                 the optional finisher at stalls (no counterpart in the reference)
// Host: the sweep loop of main_3d.cu:6784-7149; per-sweep counts are read back like the
// reference's cudaMemcpyFromSymbol calls (main_3d.cu:6918-6921, 6989-6992, 7096-7143).
//
// Records: a mismatched (or f-critical) cell is stored as (vertex << 7) | local cell, where the
// vertex is the cell's owner in g (in f for f-critical lists) and the local cell numbers the 75
// cells around a vertex (lower_star.h). Lists are filled with wave-aggregated atomics: the set is
// deterministic, the order is not, and every consumer is order independent.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <hipcub/hipcub.hpp>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <algorithm>
#include <atomic>
#include <thread>
#include <vector>

#include "../../include/dmtz.h"
#include "mismatch.h"
#include "pairs.h"
#include "repair.h"
#include "rules.h"
#include "star_planes.h"
#include "walls.h"

using namespace dmtz;
typedef unsigned long long ull;

namespace {

enum : int {
    K_MIN = 0, K_S1 = 1, K_S2 = 2, K_MAX = 3,  // record lists per cell type
    K_TGT = 4,                                  // edit set size
    K_DS = 5, K_AS = 6,                         // separatrix mismatch lists
    K_MOVED = 7,                                // edits that changed a value or a counter
    K_FC0 = 8,                                  // f-critical lists per type: 8..11
    K_WALK = 12,                                // capped walks
    K_CHG = 13, K_DIRTY = 14,                   // changed vertices, dirty stars
    K_FINISH = 15,                              // finisher tie-repair marks
    K_STARS = 16,                               // star codes re-evaluated from dirty lists
    K_DSW = 17,                                 // 2-saddle wall mismatch list
    K_WOVF = 18,                                // wall walks that outgrew their visited set
    K_ASNEXT = 19,                              // next face of the work-stealing path walk
    K_ASTOTAL = 20,                             // steps of the listed paths
    K_DTILES = 21,                              // tiles whose masks the last detection read
    K_WOPEN = 22,                               // open faces of the wall checks
    K_NCTR = 23
};

constexpr uint8_t FROZEN = 7;  // counter value of a vertex restored to f by the finisher

constexpr int BLOCK = 256;

// ------------------------------------------------------------------------------------------------
// Wave64 helpers
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ int wave_excl_scan(int x, int& total) {
    const int lane = __lane_id();
    int inc = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    total = __shfl(inc, 63, 64);
    return inc - x;
}

// Every lane of the wave must call this. Returns the lane's first slot in the list.
__device__ __forceinline__ ull wave_alloc(ull* ctr, int n) {
    int total;
    int pre = wave_excl_scan(n, total);
    ull base = 0;
    if (__lane_id() == 0 && total > 0) base = atomicAdd(ctr, (ull)total);
    unsigned lo = __shfl((unsigned)(base & 0xffffffffu), 0, 64);
    unsigned hi = __shfl((unsigned)(base >> 32), 0, 64);
    return (((ull)hi << 32) | lo) + (ull)pre;
}

// Every thread of the block must call this (block-uniform control flow). Returns the thread's
// first slot in the list, claimed with one atomic per block: appends of every wave to one
// counter are serialised at the memory side, so a wave-level claim over a list of millions of
// entries costs more than the work that fills it.
__device__ __forceinline__ ull block_alloc(ull* ctr, int n) {
    __shared__ int wsum[BLOCK / 64];
    __shared__ ull bbase;
    int wt;
    const int pre = wave_excl_scan(n, wt);
    const int w = (int)(threadIdx.x >> 6);
    if (__lane_id() == 0) wsum[w] = wt;
    __syncthreads();
    int off = 0, tot = 0;
    for (int i = 0; i < BLOCK / 64; i++) {
        off += i < w ? wsum[i] : 0;
        tot += wsum[i];
    }
    if (threadIdx.x == 0) bbase = tot ? atomicAdd(ctr, (ull)tot) : 0;
    __syncthreads();
    const ull r = bbase + (ull)(off + pre);
    __syncthreads();  // wsum and bbase are reused by the block's next call
    return r;
}

// Every thread of the block must call this. Adds the number of threads with x set to *ctr.
__device__ __forceinline__ void block_add(ull* ctr, bool x) {
    __shared__ int wcnt[BLOCK / 64];
    const ull b = __ballot(x ? 1 : 0);
    if (__lane_id() == 0) wcnt[threadIdx.x >> 6] = __popcll(b);
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int i = 0; i < BLOCK / 64; i++) tot += wcnt[i];
        if (tot) atomicAdd(ctr, (ull)tot);
    }
    __syncthreads();
}

// Every lane of the wave must call this. Adds the number of lanes with x set to *ctr.
__device__ __forceinline__ void wave_add(ull* ctr, bool x) {
    const ull b = __ballot(x ? 1 : 0);
    if (__lane_id() == 0 && b) atomicAdd(ctr, (ull)__popcll(b));
}

struct Lists4 {
    uint64_t* l[4];
    ull cap;
};

// Dense emitters handle EMIT_V vertices per thread: thread t of a block takes vertices
// base + k * BLOCK + t (k < EMIT_V), so each load of a wave is contiguous.
constexpr int EMIT_V = 8;
constexpr i64 EMIT_TILE = (i64)BLOCK * EMIT_V;

// Append the set bits of the masks of a block's EMIT_TILE vertices to the four typed lists. Space
// is claimed with one atomic per type per block after an LDS scan of the per-thread counts;
// blocks with nothing to append return at once. Every thread of the block must call this.
__device__ __forceinline__ void block_emit(i64 base, const uint64_t (&lo)[EMIT_V], const uint32_t (&hi)[EMIT_V],
                                           const Lists4& out, ull* ctr) {
    __shared__ uint32_t wtot[4][BLOCK / 64];
    __shared__ ull wbase[4][BLOCK / 64];
    int cnt[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < EMIT_V; k++) {
        cnt[0] += (int)(lo[k] & 1ull);
        cnt[1] += __popcll((lo[k] >> 1) & 0x3FFFull);
        cnt[2] += __popcll((lo[k] >> 15) & ((1ull << 36) - 1));
        cnt[3] += __popc(hi[k]);
    }
    if (__syncthreads_or(cnt[0] | cnt[1] | cnt[2] | cnt[3]) == 0) return;
    const int wave = threadIdx.x >> 6;
    int pre[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        int tot;
        pre[t] = wave_excl_scan(cnt[t], tot);
        if (__lane_id() == 0) wtot[t][wave] = (uint32_t)tot;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        const int t = threadIdx.x;
        ull sum = 0;
        for (int w = 0; w < BLOCK / 64; w++) sum += wtot[t][w];
        ull b = sum ? atomicAdd(ctr + t, sum) : 0;
        for (int w = 0; w < BLOCK / 64; w++) {
            wbase[t][w] = b;
            b += wtot[t][w];
        }
    }
    __syncthreads();
    ull at[4];
#pragma unroll
    for (int t = 0; t < 4; t++) at[t] = wbase[t][wave] + (ull)pre[t];
#pragma unroll
    for (int k = 0; k < EMIT_V; k++) {
        const uint64_t key = (uint64_t)(base + (i64)k * BLOCK + threadIdx.x) << 7;
        if ((lo[k] & 1ull) && at[0] < out.cap) out.l[0][at[0]] = key | LC_VERT;
        at[0] += lo[k] & 1ull;
        uint64_t m = out.l[1] ? (lo[k] >> 1) & 0x3FFFull : 0;
        while (m) {
            const int b = __builtin_ctzll(m);
            m &= m - 1;
            if (at[1] < out.cap) out.l[1][at[1]] = key | (uint64_t)(LC_EDGE + b);
            at[1]++;
        }
        m = (lo[k] >> 15) & ((1ull << 36) - 1);
        while (m) {
            const int b = __builtin_ctzll(m);
            m &= m - 1;
            if (at[2] < out.cap) out.l[2][at[2]] = key | (uint64_t)(LC_TRI + b);
            at[2]++;
        }
        uint32_t h = hi[k];
        while (h) {
            const int b = __builtin_ctz(h);
            h &= h - 1;
            if (at[3] < out.cap) out.l[3][at[3]] = key | (uint64_t)(LC_TET + b);
            at[3]++;
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Kernels
// ------------------------------------------------------------------------------------------------
// 75-bit mask over the local cells of a vertex: the f-critical status of every local cell
// (mismatch.h: local_crit), or the mismatched cells a vertex owns in g.
struct CritMask {
    uint64_t lo;
    uint32_t hi;
};
// Masks of all vertices, the two parts apart so that dense passes write full lines.
struct MaskArray {
    uint64_t* lo;
    uint32_t* hi;
    __device__ __forceinline__ CritMask get(i64 v) const { return CritMask{lo[v], hi[v]}; }
    __device__ __forceinline__ void put(i64 v, const CritMask& m) const {
        lo[v] = m.lo;
        hi[v] = m.hi;
    }
};
constexpr double MASK_BYTES = sizeof(uint64_t) + sizeof(uint32_t);

// The lower-star classification is fully unrolled straight-line code of about 5k instructions
// needing about 100 VGPRs (lower_star.h keeps its live state small). CODE_BLOCKS_PER_CU = 4 caps
// the code kernels at 128 VGPRs: four waves per SIMD to hide the loads of the star values.
constexpr int CODE_BLOCKS_PER_CU = 4;

// Star codes of every vertex. own (lo nullable) receives the critical cells each vertex owns, from the
// lower star itself (the first pass of the f-critical masks, without reading the codes back).
template <class T>
__global__ __launch_bounds__(BLOCK, CODE_BLOCKS_PER_CU) void k_code(const T* fld, Dims d, Counts c, CodeArray code,
                                                                    MaskArray own) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (v >= c.N) return;
    LowerStar ls;
    star_of(fld, d, v, ls);
    StarCode sc;
    encode_star(ls, sc);
    code_put(code, v, sc);
    if (own.lo) {
        CritMask m;
        crit_mask(ls, m.lo, m.hi);
        own.put(v, m);
    }
}

// g star code of vertex v and its mismatch mask: the cells v owns in g whose critical status in
// g differs from f's (owner_mismatch, main_3d.cu:2492-2550). Returns whether the code changed.
// nz_old / nz_new (nullable) receive whether the mask was nonzero before and after.
template <class T>
__device__ __forceinline__ bool code_g_at(const T* g, Dims d, i64 v, CodeArray code, MaskArray crit_f,
                                          MaskArray mm, bool* nz_old = nullptr, bool* nz_new = nullptr) {
    LowerStar ls;
    star_of(g, d, v, ls);
    StarCode sc;
    encode_star(ls, sc);
    const StarCode old = code_at(code, v);
    code_put(code, v, sc);
    const CritMask cf = crit_f.get(v);
    uint64_t c_lo, i_lo;  // owner_mismatch of sc, from the lower star's own masks
    uint32_t c_hi, i_hi;
    crit_mask(ls, c_lo, c_hi);
    member_mask(ls, i_lo, i_hi);
    CritMask m;
    m.lo = (c_lo ^ cf.lo) & i_lo;
    m.hi = (c_hi ^ cf.hi) & i_hi;
    if (nz_old) {
        const CritMask o = mm.get(v);
        *nz_old = (o.lo | (uint64_t)o.hi) != 0;
    }
    if (nz_new) *nz_new = (m.lo | (uint64_t)m.hi) != 0;
    mm.put(v, m);
    return ((old.w[0] ^ sc.w[0]) | (old.w[1] ^ sc.w[1]) | (old.w[2] ^ sc.w[2]) | (old.w[3] ^ sc.w[3])) != 0;
}

// Mark vertex v and the (up to 8) cubes that have it as a corner, each at the vertex it is anchored
// at, in the bitmap of the path checks. Anchors v - k and v - k - 1 along x share a word mostly.
__device__ __forceinline__ void mark_vertex(Dims d, uint32_t v, uint32_t* marks) {
    i64 x, y, z;
    vxyz(d, (i64)v, x, y, z);
    for (int k = 0; k < 4; k++) {
        if (y < (k & 1) || z < (k >> 1)) continue;
        const i64 a = (i64)v - (k & 1) * d.W - (k >> 1) * d.W * d.H;
        uint32_t m = 1u << (a & 31);
        if (x > 0) {
            if (a & 31) m |= m >> 1;
            else atomicOr(marks + (a >> 5) - 1, 0x80000000u);
        }
        atomicOr(marks + (a >> 5), m);
    }
}

// Dense re-evaluation; tile_nz (zeroed before) receives, per EMIT_TILE vertices, the number with
// a nonzero mismatch mask (a wave's 64 vertices lie in one tile).
template <class T>
__global__ __launch_bounds__(BLOCK, CODE_BLOCKS_PER_CU) void k_code_g(const T* g, Dims d, Counts c, CodeArray code,
                                                  MaskArray crit_f, MaskArray mm, uint32_t* tile_nz) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    bool nz = false;
    if (v < c.N) code_g_at(g, d, v, code, crit_f, mm, nullptr, &nz);
    const ull b = __ballot(nz ? 1 : 0);
    if (__lane_id() == 0 && b) atomicAdd(tile_nz + (v / EMIT_TILE), (uint32_t)__popcll(b));
}

// The list length is read on the device (*n_ptr, written by the kernel that filled the list), so
// the host launches it without waiting; the grid strides over the list. Block 0 adds the length
// to *stars, the count of star codes re-evaluated in the run. With marks != null, every vertex
// whose code changed is marked for the path checks (their results read nothing but star codes).
// tile_nz follows the masks whose nonzero-ness changes.
template <class T>
__global__ __launch_bounds__(BLOCK, CODE_BLOCKS_PER_CU) void k_code_list_g(const T* g, Dims d, CodeArray code,
                                                                         MaskArray crit_f, MaskArray mm,
                                                                         const uint32_t* list, const ull* n_ptr,
                                                                         ull* stars, uint32_t* marks,
                                                                         uint32_t* tile_nz) {
    const ull n = *n_ptr;
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(stars, n);
    for (ull i = (ull)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (ull)gridDim.x * BLOCK) {
        const uint32_t v = list[i];
        bool nz_old = false, nz_new = false;
        const bool changed = code_g_at(g, d, (i64)v, code, crit_f, mm, &nz_old, &nz_new);
        if (nz_old != nz_new) atomicAdd(tile_nz + (v / EMIT_TILE), nz_new ? 1u : 0xFFFFFFFFu);
        if (changed && marks) mark_vertex(d, v, marks);
    }
}

// The dense classifications over bit planes (star_planes.h): a wave takes PLANE_TILE consecutive
// vertices, lane l and bit 31 - b the vertex base + 64 b + l, so that a row of a tile is 64
// consecutive vertices, read and written coalesced. About 21 thousand vector instructions per tile, a
// third of them comparisons; the words of the passes take all 512 registers, so one wave runs per SIMD. It
// issues half of its time and waits for its loads and stores most of the rest, with no second wave to
// cover that (counters at 512^3: 50 % issuing, 44 % waiting). 512^3 float32: 15.2 ms with a thread per
// vertex, now 4.75 (9.4 GB, 2.0 TB/s; at the issue limit it would be 2.3); 256^3: 1.99 -> 0.61 ms. With 256
// registers and two waves the spills cost more than the second wave gives (15 ms). Codes and masks are
// stored word by word (CodeArray, MaskArray): as 32-byte structs, whose words leave a tile at different
// times, the lines were written to memory several times over (23.5 GB instead of 6.4 at 512^3, 10.7 ms).
static_assert(PLANE_TILE == EMIT_TILE, "a wave's count of nonzero masks is its tile's");

// Stores of a tile: codes, and per vertex its owned critical cells (crit_f null) or the mismatch
// with f's critical cells.
struct TileOut {
    i64 v0, n;
    CodeArray codes;
    MaskArray mask;    // lo nullable
    MaskArray crit_f;  // lo null: mask receives the owned critical cells
    bool full;         // the whole tile lies in the field (wave-uniform)
    uint32_t nz;       // bit r: the vertex of bit r has a nonzero mismatch mask

    __device__ __forceinline__ i64 vertex(int r) const { return v0 + 64 * (PLANE_ROWS - 1 - r); }
    template <class Fn>
    __device__ __forceinline__ void rows(Fn fn) const {
        if (full) {
#pragma unroll
            for (int r = 0; r < 32; r++) fn(r, vertex(r));
        } else {
#pragma unroll
            for (int r = 0; r < 32; r++)
                if (vertex(r) < n) fn(r, vertex(r));
        }
    }
    __device__ __forceinline__ void code(int k, const uint32_t* lo, const uint32_t* hi) const {
        uint64_t* const w = codes.w + k * codes.n;
        rows([&](int r, i64 v) { *reinterpret_cast<uint2*>(w + v) = make_uint2(lo[r], hi[r]); });
    }
    __device__ __forceinline__ void masks_lo(uint32_t* c0, uint32_t* c1, const uint32_t* i0, const uint32_t* i1) {
        if (!mask.lo) return;
        if (crit_f.lo) {
            uint32_t x = 0;
            rows([&](int r, i64 v) {
                const uint2 cf = *reinterpret_cast<const uint2*>(crit_f.lo + v);
                c0[r] ^= cf.x & i0[r];
                c1[r] ^= cf.y & i1[r];
                x |= (uint32_t)((c0[r] | c1[r]) != 0u) << r;
            });
            nz |= x;
        }
        rows([&](int r, i64 v) { *reinterpret_cast<uint2*>(mask.lo + v) = make_uint2(c0[r], c1[r]); });
    }
    __device__ __forceinline__ void masks_hi(uint32_t* c2, const uint32_t* i2) {
        if (!mask.lo) return;
        if (crit_f.lo) {
            uint32_t x = 0;
            rows([&](int r, i64 v) {
                c2[r] ^= crit_f.hi[v] & i2[r];
                x |= (uint32_t)(c2[r] != 0u) << r;
            });
            nz |= x;
        }
        rows([&](int r, i64 v) { mask.hi[v] = c2[r]; });
    }
};

// k_code and k_code_g (crit_f.lo and tile_nz not null) over bit planes.
template <class T>
__global__ __launch_bounds__(64, 1) void k_code_planes(const T* fld, Dims d, Step64 st, i64 n, CodeArray code,
                                                       MaskArray mask, MaskArray crit_f, uint32_t* tile_nz) {
    const i64 v0 = (i64)blockIdx.x * PLANE_TILE + threadIdx.x;
    StarWords w;
    tile_words(fld, d, st, n, v0, w);
    TileOut out{v0, n, code, mask, crit_f, ((i64)blockIdx.x + 1) * PLANE_TILE <= n, 0u};
    classify_words(w, out);
    if (tile_nz) {
        int cnt = __popc(out.nz);
        for (int o = 32; o > 0; o >>= 1) cnt += __shfl_down(cnt, o, 64);
        if (threadIdx.x == 0) tile_nz[blockIdx.x] = (uint32_t)cnt;
    }
}

// f-critical status of the local cells of every vertex (once per run), in two passes: each
// vertex writes the critical cells it owns (k_code's own output, or k_critf_own from the codes),
// then gathers the ones its 14 neighbours own that contain it (k_critf_gather: 15 coalesced reads
// of 12 bytes and one store per vertex; the reverse, each owner spreading its cells with
// atomics, wrote five times the masks' size to memory and took twice as long).
__global__ __launch_bounds__(BLOCK) void k_critf_own(CodeArray cf, i64 n, MaskArray out) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (v >= n) return;
    uint64_t lo, ilo;
    uint32_t hi, ihi;
    code_masks(code_at(cf, v), lo, hi, ilo, ihi);
    out.put(v, CritMask{lo & ilo, hi & ihi});
}

// Critical cells per type (vertex, edge, triangle, tet) over all owners: one atomic per wave and type.
__global__ __launch_bounds__(BLOCK) void k_crit_count(CodeArray code, i64 n, ull* ctr) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    int cnt[4] = {0, 0, 0, 0};
    if (v < n) {
        uint64_t lo, ilo;
        uint32_t hi, ihi;
        code_masks(code_at(code, v), lo, hi, ilo, ihi);
        lo &= ilo;
        hi &= ihi;
        cnt[0] = (int)(lo & 1ull);
        cnt[1] = __popcll((lo >> 1) & 0x3FFFull);
        cnt[2] = __popcll(lo >> 15);
        cnt[3] = __popc(hi);
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        int tot;
        wave_excl_scan(cnt[t], tot);
        if (__lane_id() == 0 && tot) atomicAdd(ctr + t, (ull)tot);
    }
}

__global__ __launch_bounds__(BLOCK) void k_critf_gather(MaskArray own, Dims d, i64 n, MaskArray out) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (v >= n) return;
    uint64_t lo;
    uint32_t hi;
    crit_gather(
        d, v,
        [&](i64 u, uint64_t& a, uint32_t& b) {
            const CritMask m = own.get(u);
            a = m.lo;
            b = m.hi;
        },
        lo, hi);
    out.put(v, CritMask{lo, hi});
}

// Dense mismatch detection: every vertex lists the mismatched cells it owns in g, from the
// per-vertex mismatch masks kept with the g star codes (12 bytes per vertex).
// A tile whose count of nonzero masks is zero is skipped without reading its masks; tiles_read
// counts the tiles whose masks were read. A grid of at most DETECT_BLOCKS blocks strides over
// the tiles: block b takes tiles b, b + grid, ..., reads the counts of 64 of them at once and
// visits only the nonzero ones, so a late sweep with a few mismatches does not dispatch a block
// per tile of the grid.
constexpr unsigned DETECT_BLOCKS = 2048;

// A block gathers the records of its tiles in LDS and claims list space when a type's buffer is full and
// at the end. (A claim per tile and type was the cost of the pass in sweeps with a few records in every
// tile: the memory side serves the claims of all blocks on the four counters one after the other.
// 512^3 fBm, 101 detections: 10.0 -> 6.9 ms.) A tile with more than DETECT_STAGE mismatched vertices, or more
// records of a type than a buffer holds, appends them at once with claims of its own (block_emit).
constexpr int DETECT_BUF = 512;
constexpr uint32_t DETECT_STAGE = 96;

__global__ __launch_bounds__(BLOCK) void k_detect(MaskArray mm, i64 n, const uint32_t* tile_nz, Lists4 out,
                                                  ull* ctr, ull* tiles_read) {
    __shared__ uint64_t nz_mask;
    __shared__ uint64_t buf[4][DETECT_BUF];
    __shared__ uint32_t wtot[4][BLOCK / 64];
    __shared__ ull claim[4];
    const int wave = threadIdx.x >> 6;
    uint32_t fill[4] = {0, 0, 0, 0};  // block-uniform
    ull tiles = 0;
    // Writes out the buffers (block-uniform control flow).
    auto flush = [&]() {
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 4; t++)
            if (threadIdx.x == 64 * t && fill[t]) claim[t] = atomicAdd(ctr + t, (ull)fill[t]);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 4; t++) {
            for (uint32_t i = threadIdx.x; i < fill[t]; i += BLOCK)
                if (claim[t] + i < out.cap) out.l[t][claim[t] + i] = buf[t][i];
            fill[t] = 0;
        }
        __syncthreads();
    };
    const i64 ntiles = (n + EMIT_TILE - 1) / EMIT_TILE, stride = (i64)gridDim.x;
    for (i64 first = blockIdx.x; first < ntiles; first += 64 * stride) {
        if (threadIdx.x < 64) {
            const i64 tile = first + (i64)threadIdx.x * stride;
            const uint64_t m = __ballot(tile < ntiles && tile_nz[tile] != 0);
            if (threadIdx.x == 0) nz_mask = m;
        }
        __syncthreads();
        uint64_t todo = nz_mask;
        __syncthreads();  // nz_mask is rewritten by the next group
        tiles += (ull)__popcll(todo);
        while (todo) {
            const i64 base = (first + (i64)__builtin_ctzll(todo) * stride) * EMIT_TILE;
            todo &= todo - 1;
            uint64_t lo[EMIT_V];
            uint32_t hi[EMIT_V];
            int cnt[4] = {0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < EMIT_V; k++) {
                const i64 v = base + (i64)k * BLOCK + threadIdx.x;
                lo[k] = 0;
                hi[k] = 0;
                if (v < n) {
                    const CritMask m = mm.get(v);
                    lo[k] = m.lo;
                    hi[k] = m.hi;
                }
                cnt[0] += (int)(lo[k] & 1ull);
                cnt[1] += __popcll((lo[k] >> 1) & 0x3FFFull);
                cnt[2] += __popcll((lo[k] >> 15) & ((1ull << 36) - 1));
                cnt[3] += __popc(hi[k]);
            }
            if (tile_nz[base / EMIT_TILE] > DETECT_STAGE) {
                block_emit(base, lo, hi, out, ctr);
                continue;
            }
            uint32_t at[4], tot[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                int wt;
                at[t] = (uint32_t)wave_excl_scan(cnt[t], wt);
                if (__lane_id() == 0) wtot[t][wave] = (uint32_t)wt;
            }
            __syncthreads();
            bool over = false, fits = true;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                tot[t] = 0;
                for (int w = 0; w < BLOCK / 64; w++) {
                    at[t] += w < wave ? wtot[t][w] : 0u;
                    tot[t] += wtot[t][w];
                }
                over = over || fill[t] + tot[t] > DETECT_BUF;
                fits = fits && tot[t] <= DETECT_BUF;
            }
            __syncthreads();  // wtot is reused by the next tile
            if (!fits) {
                block_emit(base, lo, hi, out, ctr);
                continue;
            }
            if (over) flush();
#pragma unroll
            for (int t = 0; t < 4; t++) {
                at[t] += fill[t];
                fill[t] += tot[t];
            }
            if (cnt[0] | cnt[1] | cnt[2] | cnt[3]) {
#pragma unroll
                for (int k = 0; k < EMIT_V; k++) {
                    const uint64_t key = (uint64_t)(base + (i64)k * BLOCK + threadIdx.x) << 7;
                    if (lo[k] & 1ull) buf[0][at[0]++] = key | LC_VERT;
                    for (uint64_t m = (lo[k] >> 1) & 0x3FFFull; m; m &= m - 1)
                        buf[1][at[1]++] = key | (uint64_t)(LC_EDGE + __builtin_ctzll(m));
                    for (uint64_t m = (lo[k] >> 15) & ((1ull << 36) - 1); m; m &= m - 1)
                        buf[2][at[2]++] = key | (uint64_t)(LC_TRI + __builtin_ctzll(m));
                    for (uint32_t h = hi[k]; h; h &= h - 1) buf[3][at[3]++] = key | (uint64_t)(LC_TET + __builtin_ctz(h));
                }
            }
        }
    }
    if (fill[0] | fill[1] | fill[2] | fill[3]) flush();
    if (threadIdx.x == 0 && tiles) atomicAdd(tiles_read, tiles);
}

// Critical cells owned by each vertex, from the masks of owned critical cells (own, as k_code leaves
// them) or, when own.lo is null, from the star codes; type_mask selects which types count, and a
// type whose list is null is counted but not listed.
__global__ __launch_bounds__(BLOCK) void k_fcrit(MaskArray own, CodeArray cf, Counts c, Lists4 out,
                                                 ull* ctr, int type_mask) {
    const i64 base = (i64)blockIdx.x * EMIT_TILE;
    uint64_t keep = 0;
    if (type_mask & 1) keep |= 1ull;
    if (type_mask & 2) keep |= 0x3FFFull << 1;
    if (type_mask & 4) keep |= ((1ull << 36) - 1) << 15;
    uint64_t lo[EMIT_V];
    uint32_t hi[EMIT_V];
#pragma unroll
    for (int k = 0; k < EMIT_V; k++) {
        const i64 v = base + (i64)k * BLOCK + threadIdx.x;
        lo[k] = 0;
        hi[k] = 0;
        if (v < c.N) {
            if (own.lo) {
                const CritMask m = own.get(v);
                lo[k] = m.lo;
                hi[k] = m.hi;
            } else {
                uint64_t ilo;
                uint32_t ihi;
                code_masks(code_at(cf, v), lo[k], hi[k], ilo, ihi);
            }
            lo[k] &= keep;
            if (!(type_mask & 8)) hi[k] = 0;
        }
    }
    block_emit(base, lo, hi, out, ctr);
}

// The edit set of an epoch: the vertices whose stamp holds it. With a list, each vertex is also
// appended to it once (an exchange of its stamp and a claim of a slot, both of which wait for the
// memory side); without, the stamps are plain stores and k_apply_marked reads all of them.
struct TargetSink {
    uint32_t* stamp;
    uint32_t epoch;
    uint32_t* list;  // null: mark only
    ull* ctr;
    ull cap;
    __device__ void operator()(i64 v) const {
        if (!list) {
            stamp[v] = epoch;
            return;
        }
        uint32_t old = atomicExch(stamp + v, epoch);
        if (old != epoch) {
            ull i = atomicAdd(ctr, 1ull);
            if (i < cap) list[i] = (uint32_t)v;
        }
    }
};

// The targets a lane's rule emits, held in registers so that the rule's chain of reads never
// waits on the edit set: the stamp exchanges of all of them are issued together at the end, and
// the wave claims list slots for the new ones with one atomic. No repair rule emits more than
// four; a fifth target would go through the direct sink at once.
struct HoldSink {
    TargetSink direct;
    uint32_t t0, t1, t2, t3;
    int n;
    __device__ __forceinline__ void operator()(i64 v) {
        if (n < 4) {
            t3 = t2;
            t2 = t1;
            t1 = t0;
            t0 = (uint32_t)v;
            n++;
        } else {
            direct(v);
        }
    }
    // Every lane of the wave must call this. Adds the held targets not yet in this epoch's set.
    __device__ __forceinline__ void flush() const {
        const uint32_t e = direct.epoch;
        if (!direct.list) {
            if (n > 0) direct.stamp[t0] = e;
            if (n > 1) direct.stamp[t1] = e;
            if (n > 2) direct.stamp[t2] = e;
            if (n > 3) direct.stamp[t3] = e;
            return;
        }
        uint32_t o0 = e, o1 = e, o2 = e, o3 = e;
        if (n > 0) o0 = atomicExch(direct.stamp + t0, e);
        if (n > 1) o1 = atomicExch(direct.stamp + t1, e);
        if (n > 2) o2 = atomicExch(direct.stamp + t2, e);
        if (n > 3) o3 = atomicExch(direct.stamp + t3, e);
        const bool n0 = o0 != e, n1 = o1 != e, n2 = o2 != e, n3 = o3 != e;
        ull at = wave_alloc(direct.ctr, (int)n0 + (int)n1 + (int)n2 + (int)n3);
        const ull cap = direct.cap;
        if (n0) {
            if (at < cap) direct.list[at] = t0;
            at++;
        }
        if (n1) {
            if (at < cap) direct.list[at] = t1;
            at++;
        }
        if (n2) {
            if (at < cap) direct.list[at] = t2;
            at++;
        }
        if (n3 && at < cap) direct.list[at] = t3;
    }
};

// The repair rules of all four cell types in one launch; a block holds records of one type. (A kernel per
// type, the saddles and maxima on a second stream, cost a short sweep three launches and four event
// packets more and gained nothing on long lists: 256^3 mixtures 68.9 ms per correction, together 61.8;
// 512^3 fBm 105.0 either way.) The rule runs in vertex frames
// (rules.h); a record whose numbers collide takes the rule over global ids, a wave-rare branch.
// A record is two to five dependent reads (values, then a star code, then the partner's values and
// code), and a list of a few records takes their latency: 12 us (2-saddles; 80 over global ids). Long lists
// are bound by the lines they touch: 512^3 fBm, 90 lists, 78 GB in 19 ms, 4.1 TB/s. The records are taken in
// the order of their lists: neighbouring records share the lines
// they read, which is worth more than waves of one branch. (Over global ids, where a wave paid for
// every branch body with thousands of instructions, the records were grouped by branch first; with
// these rules the grouping costs 512^3 fBm 19 ms of 195 and 256^3 mixtures 13 of 122.)
template <class T>
struct FixArgs {
    const T* f;
    CodeArray cf;
    const T* g;
    CodeArray cg;
    Dims d;
    Counts c;
    const uint8_t* counter;
    double eps, range;
    int edit_type;
};
// Tables of the rules in LDS. Every thread of the block must call load().
struct RuleLds {
    RuleTables tb;
    int32_t off[15];
    __device__ __forceinline__ void load(const Dims& d) {
        if (threadIdx.x < sizeof(RuleTables) / 4)
            reinterpret_cast<uint32_t*>(&tb)[threadIdx.x] = reinterpret_cast<const uint32_t*>(&RT)[threadIdx.x];
        if (threadIdx.x < 15) off[threadIdx.x] = threadIdx.x == 14 ? 0 : (int32_t)slot_step(d, threadIdx.x);
        __syncthreads();
    }
};
template <class T, int TYPE>
__device__ __forceinline__ void fix_record(const FixArgs<T>& a, const RuleLds& lds, uint64_t r, HoldSink& hold) {
    const uint32_t v = (uint32_t)(r >> 7);
    const int lc = (int)(r & 127u);
    LocalRules<T, HoldSink, CodeArray> L{a.f, a.cf, a.g, a.cg, a.counter, &lds.tb, lds.off,
                                         a.d, a.c, a.eps, a.edit_type, hold};
    if (__builtin_expect(!L.template run<TYPE>(v, lc), 0)) {
        Repair<T, HoldSink, CodeArray> R(a.f, a.cf, a.g, a.cg, a.d, a.c, a.counter, a.eps, a.range, a.edit_type, hold);
        const i64 id = local_cell_id(a.d, a.c, (i64)v, lc);
        if (TYPE == 1) R.fix_saddle(id);
        else if (TYPE == 2) R.fix_2saddle(id);
        else if (TYPE == 3) R.fix_maximum(id);
        hold = R.sink;
    }
}
// The blocks from first[k] on take the list of type 2, 0, 1, 3 (k = 0 to 3; an empty list has no block).
struct FixLists {
    const uint64_t* recs[4];
    ull n[4];
    unsigned first[5];
};
template <class T>
__global__ __launch_bounds__(BLOCK) void k_fix_cp(FixLists q, FixArgs<T> a, TargetSink sink) {
    __shared__ RuleLds lds;
    lds.load(a.d);
    const unsigned b = blockIdx.x;
    const int k = b < q.first[1] ? 0 : b < q.first[2] ? 1 : b < q.first[3] ? 2 : 3;
    const ull i = (ull)(b - q.first[k]) * BLOCK + threadIdx.x;
    HoldSink hold{sink, 0u, 0u, 0u, 0u, 0};
    if (i < q.n[k]) {
        const uint64_t r = q.recs[k][i];
        if (k == 0) fix_record<T, 2>(a, lds, r, hold);
        else if (k == 1) fix_record<T, 0>(a, lds, r, hold);
        else if (k == 2) fix_record<T, 1>(a, lds, r, hold);
        else fix_record<T, 3>(a, lds, r, hold);
    }
    hold.flush();
}

// Zero the counters whose bit is set in mask: one launch where a memset per run of counters
// would take several.
__global__ __launch_bounds__(64) void k_zero_ctrs(ull* ctr, uint32_t mask) {
    const int k = (int)threadIdx.x;
    if (k < K_NCTR && ((mask >> k) & 1u)) ctr[k] = 0;
}
static_assert(K_NCTR <= 32, "k_zero_ctrs takes a 32-bit mask");
constexpr uint32_t ctr_bit(int k) { return 1u << k; }
constexpr uint32_t DETECT_CTRS = ctr_bit(K_MIN) | ctr_bit(K_MIN + 1) | ctr_bit(K_MIN + 2) | ctr_bit(K_MIN + 3) |
                                 ctr_bit(K_DTILES);

// The counters into the host's pinned copy: a launch costs the host a third of the copy command that
// would do it.
__global__ __launch_bounds__(64) void k_read_ctrs(const ull* ctr, ull* host) {
    const int k = (int)threadIdx.x;
    if (k < K_NCTR) host[k] = ctr[k];
}

// The edit of vertex v (applyDeltaBuffer1 main_3d.cu:1122-1164; frozen vertices are never edited).
// ch: its value changed (the order, hence every lower star, only sees value comparisons); mv: its
// value or its counter did.
template <class T>
__device__ __forceinline__ void edit_vertex(i64 v, const T* f, T* g, uint8_t* counter, double eps, double range,
                                            int preserve_type, int edit_type, bool& ch, bool& mv) {
    const int k0 = counter[v];
    ch = mv = false;
    if (k0 == FROZEN) return;
    const T fv = f[v];
    const T g0 = g[v];
    T gv = g0;
    int k = k0;
    const double dl = edit_type == 1 ? halving_delta(eps, k) : EditArith<T>::delta0(fv, gv, eps);
    if (preserve_type == 0) {
        if (fabs_d(dl) > 1e-15 * range && k < 5 && EditArith<T>::step(fv, gv, dl, eps)) {
            k += 1;
        } else {
            k = 6;
            gv = EditArith<T>::snap(fv, eps);
        }
    } else {
        k = 6;
        gv = EditArith<T>::snap(fv, eps);
    }
    g[v] = gv;
    counter[v] = (uint8_t)k;
    ch = !(gv == g0);
    mv = ch || k != k0;
}

// moved counts the edits that changed a value or a counter. The edit set's size is read on the
// device (*n_ptr, at most cap); the grid strides over the set in block-uniform steps, so every lane
// takes part in the wave-wide appends.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_apply(const uint32_t* list, const ull* n_ptr, ull cap, const T* f, T* g,
                                                 uint8_t* counter, double eps, double range, int preserve_type,
                                                 int edit_type, uint32_t* changed, ull* chg_ctr, ull* moved) {
    const ull n = *n_ptr < cap ? *n_ptr : cap;
    for (ull base = (ull)blockIdx.x * BLOCK; base < n; base += (ull)gridDim.x * BLOCK) {
        const ull i = base + threadIdx.x;
        bool ch = false, mv = false;
        i64 v = 0;
        if (i < n) {
            v = list[i];
            edit_vertex(v, f, g, counter, eps, range, preserve_type, edit_type, ch, mv);
        }
        ull at = block_alloc(chg_ctr, ch ? 1 : 0);
        if (ch) changed[at] = (uint32_t)v;
        block_add(moved, mv);
    }
}

// The same for a marked edit set: one pass over the stamps, so the edits read and write the fields
// in order and the changed list comes out in about vertex order. Each block strides over chunks of
// BLOCK * APPLY_V vertices and gathers the changed ones in LDS, so that it claims list space once per
// APPLY_BUF of them and adds to the counters once: the memory side serves the claims of all blocks
// one after the other (a claim and two sums per chunk: 0.9 ms of a 512^3 pass, whatever it edits).
constexpr int APPLY_V = 8;
constexpr int APPLY_BUF = 4096;
static_assert(APPLY_BUF >= BLOCK * APPLY_V, "a chunk fits the buffer");
template <class T>
__global__ __launch_bounds__(BLOCK) void k_apply_marked(const uint32_t* stamp, uint32_t epoch, i64 n, const T* f, T* g,
                                                        uint8_t* counter, double eps, double range, int preserve_type,
                                                        int edit_type, uint32_t* changed, ull* chg_ctr, ull* moved,
                                                        ull* targets) {
    __shared__ uint32_t buf[APPLY_BUF];
    __shared__ int wsum[BLOCK / 64];
    __shared__ ull claim, sums[2];
    if (threadIdx.x < 2) sums[threadIdx.x] = 0;
    const int wave = threadIdx.x >> 6;
    int fill = 0;  // block-uniform
    auto flush = [&]() {
        __syncthreads();
        if (threadIdx.x == 0) claim = atomicAdd(chg_ctr, (ull)fill);
        __syncthreads();
        for (int i = threadIdx.x; i < fill; i += BLOCK) changed[claim + (ull)i] = buf[i];
        __syncthreads();
        fill = 0;
    };
    ull moves = 0, edits = 0;
    for (i64 first = (i64)blockIdx.x * (BLOCK * APPLY_V); first < n; first += (i64)gridDim.x * (BLOCK * APPLY_V)) {
        const i64 base = first + threadIdx.x;
        uint32_t in = 0;
#pragma unroll
        for (int k = 0; k < APPLY_V; k++) {
            const i64 v = base + (i64)k * BLOCK;
            in |= (uint32_t)(v < n && stamp[v] == epoch) << k;
        }
        if (!__syncthreads_or(in != 0u)) continue;
        edits += (ull)__popc(in);
        uint32_t changes = 0;
#pragma unroll
        for (int k = 0; k < APPLY_V; k++) {
            if (!((in >> k) & 1u)) continue;
            bool ch, mv;
            edit_vertex(base + (i64)k * BLOCK, f, g, counter, eps, range, preserve_type, edit_type, ch, mv);
            changes |= (uint32_t)ch << k;
            moves += (ull)mv;
        }
        int wt;
        int at = wave_excl_scan(__popc(changes), wt);
        if (__lane_id() == 0) wsum[wave] = wt;
        __syncthreads();
        int total = 0;
        for (int w = 0; w < BLOCK / 64; w++) {
            at += w < wave ? wsum[w] : 0;
            total += wsum[w];
        }
        if (fill + total > APPLY_BUF) flush();
        at += fill;
        for (uint32_t m = changes; m; m &= m - 1) buf[at++] = (uint32_t)(base + (i64)__builtin_ctz(m) * BLOCK);
        fill += total;
        // the next chunk's barrier comes before wsum is written again
    }
    if (moves) atomicAdd(&sums[0], moves);
    if (edits) atomicAdd(&sums[1], edits);
    if (fill) flush();
    __syncthreads();
    if (threadIdx.x == 0) {
        if (sums[0]) atomicAdd(moved, sums[0]);
        if (sums[1]) atomicAdd(targets, sums[1]);
    }
}

// Finisher zone, part 1: the vertices of the first n[k] records of the four mismatch lists, each
// listed once (claimed through its stamp with a fresh epoch).
__global__ __launch_bounds__(BLOCK) void k_zone_cells(Lists4 recs, ull n0, ull n1, ull n2, ull n3, Dims d,
                                                      uint32_t* stamp, uint32_t epoch, uint32_t* list, ull* ctr) {
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    i64 vs[4] = {-1, -1, -1, -1};
    if (i < n0 + n1 + n2 + n3) {
        const int k = i < n0 ? 0 : (i < n0 + n1 ? 1 : (i < n0 + n1 + n2 ? 2 : 3));
        const ull j = i - (k > 0 ? n0 : 0) - (k > 1 ? n1 : 0) - (k > 2 ? n2 : 0);
        const uint64_t r = recs.l[k][j];
        const i64 v = (i64)(r >> 7);
        const int lc = (int)(r & 127u);
        i64 x, y, z;
        vxyz(d, v, x, y, z);
        auto nb = [&](int sl) { return vidx(d, x + DIR[sl][0], y + DIR[sl][1], z + DIR[sl][2]); };
        vs[0] = v;
        if (lc >= LC_EDGE && lc < LC_TRI) {
            vs[1] = nb(lc - LC_EDGE);
        } else if (lc >= LC_TRI && lc < LC_TET) {
            vs[1] = nb(ST.tri_i[lc - LC_TRI]);
            vs[2] = nb(ST.tri_j[lc - LC_TRI]);
        } else if (lc >= LC_TET) {
            vs[1] = nb(ST.tet_s[lc - LC_TET][0]);
            vs[2] = nb(ST.tet_s[lc - LC_TET][1]);
            vs[3] = nb(ST.tet_s[lc - LC_TET][2]);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const bool in = vs[q] >= 0 && atomicExch(stamp + vs[q], epoch) != epoch;
        ull at = wave_alloc(ctr, in ? 1 : 0);
        if (in) list[at] = (uint32_t)vs[q];
    }
}

// Finisher zone, part 2: the vertices targeted by an edit set of epoch in [from, to).
__global__ __launch_bounds__(BLOCK) void k_zone(const uint32_t* stamp, uint32_t from, uint32_t to, i64 n,
                                                uint32_t* list, ull* ctr) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    bool in = false;
    if (v < n) {
        const uint32_t s = stamp[v];
        in = s >= from && s < to;
    }
    ull at = wave_alloc(ctr, in ? 1 : 0);
    if (in) list[at] = (uint32_t)v;
}

// The box B: every vertex within Chebyshev distance r of a zone vertex is listed once (claimed
// through its stamp), snapped unless already frozen (g = snap(f): the terminal edit of
// applyDeltaBuffer1, main_3d.cu:1140-1141; the reference keeps a snap of the 14 neighbours
// commented out at main_3d.cu:1144-1151) and frozen. One work item per (zone vertex, offset in
// the (2r+1)^3 box), grid-stride with a wave-uniform trip count.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_snap_boxes(const uint32_t* zone, ull nz, int r, Dims d, const T* f, T* g,
                                                      uint8_t* counter, double eps, uint32_t* stamp, uint32_t epoch,
                                                      uint32_t* box, ull* box_ctr) {
    const ull side = 2 * (ull)r + 1, cube = side * side * side, total = nz * cube;
    for (ull base = (ull)blockIdx.x * BLOCK; base < total; base += (ull)gridDim.x * BLOCK) {
        const ull j = base + threadIdx.x;
        bool in = false;
        i64 u = 0;
        if (j < total) {
            const i64 v = zone[j / cube];
            const ull o = j % cube;
            i64 x, y, z;
            vxyz(d, v, x, y, z);
            const i64 ux = x + (i64)(o % side) - r, uy = y + (i64)((o / side) % side) - r,
                      uz = z + (i64)(o / (side * side)) - r;
            if (inb(d, ux, uy, uz)) {
                u = vidx(d, ux, uy, uz);
                if (atomicExch(stamp + u, epoch) != epoch) {
                    in = true;
                    if (counter[u] != FROZEN) g[u] = EditArith<T>::snap(f[u], eps);
                    counter[u] = FROZEN;
                }
            }
        }
        ull at = wave_alloc(box_ctr, in ? 1 : 0);
        if (in) box[at] = (uint32_t)u;
    }
}

// Tie repair, marking step of one Jacobi round: a box vertex u is marked when a neighbour w has
// g(w) == g(u), f(w) < f(u) and w > u (the index tie-break orders the pair against f).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_tie_mark(const uint32_t* box, ull n, Dims d, const T* f, const T* g,
                                                    uint32_t* stamp, uint32_t epoch, ull* marked) {
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    bool mk = false;
    if (i < n) {
        const i64 u = box[i];
        const T fu = f[u], gu = g[u];
        i64 x, y, z;
        vxyz(d, u, x, y, z);
        for (int k = 0; k < 14; k++) {
            const i64 xx = x + DIR[k][0], yy = y + DIR[k][1], zz = z + DIR[k][2];
            if (!inb(d, xx, yy, zz)) continue;
            const i64 w = vidx(d, xx, yy, zz);
            if (g[w] == gu && f[w] < fu && w > u) {
                mk = true;
                break;
            }
        }
        if (mk) stamp[u] = epoch;
    }
    wave_add(marked, mk);
}

// Tie repair, raising step: marked vertices move to the next representable value.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_tie_raise(const uint32_t* box, ull n, T* g, const uint32_t* stamp,
                                                     uint32_t epoch) {
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    if (i < n) {
        const i64 u = box[i];
        if (stamp[u] == epoch) g[u] = next_up(g[u]);
    }
}

// Restore g = f and freeze every vertex (counter 7: never edited again).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_freeze_all(const T* f, T* g, uint8_t* counter, i64 n) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (v < n) {
        g[v] = f[v];
        counter[v] = FROZEN;
    }
}

// Closed stars of the changed vertices: their lower stars must be re-evaluated. One thread per
// (changed vertex, star slot); each vertex enters the dirty list once per epoch.
// The changed count is read on the device (*n_ptr); the grid strides in block-uniform steps.
__global__ __launch_bounds__(BLOCK) void k_dirty(const uint32_t* changed, const ull* n_ptr, Dims d, uint32_t* stamp,
                                                 uint32_t epoch, uint32_t* dirty, ull* dirty_ctr) {
    const ull n = *n_ptr;
    for (ull base = (ull)blockIdx.x * BLOCK; base < 15 * n; base += (ull)gridDim.x * BLOCK) {
        const ull j = base + threadIdx.x;
        bool fresh = false;
        i64 w = 0;
        if (j < 15 * n) {
            const i64 v = changed[j / 15];
            const int slot = (int)(j % 15);
            i64 x, y, z;
            vxyz(d, v, x, y, z);
            bool ok = true;
            w = v;
            if (slot < 14) {
                i64 nx = x + DIR[slot][0], ny = y + DIR[slot][1], nz = z + DIR[slot][2];
                ok = inb(d, nx, ny, nz);
                w = ok ? vidx(d, nx, ny, nz) : 0;
            }
            if (ok) fresh = atomicExch(stamp + w, epoch) != epoch;
        }
        ull at = block_alloc(dirty_ctr, fresh ? 1 : 0);
        if (fresh) dirty[at] = (uint32_t)w;
    }
}

// Dense form of k_dirty for long change lists, where one returning atomic per (changed vertex,
// star slot) costs more than a pass over all stamps: every pair stores the epoch into its star
// vertex's stamp with a plain store (all writers store the same value), then k_dirty_collect
// lists the vertices whose stamp holds the epoch, in vertex order. Same set as k_dirty.
__global__ __launch_bounds__(BLOCK) void k_dirty_mark(const uint32_t* changed, const ull* n_ptr, Dims d,
                                                      uint32_t* stamp, uint32_t epoch) {
    const ull n = *n_ptr;
    for (ull j = (ull)blockIdx.x * BLOCK + threadIdx.x; j < 15 * n; j += (ull)gridDim.x * BLOCK) {
        const i64 v = changed[j / 15];
        const int slot = (int)(j % 15);
        if (slot == 14) {
            stamp[v] = epoch;
            continue;
        }
        i64 x, y, z;
        vxyz(d, v, x, y, z);
        const i64 nx = x + DIR[slot][0], ny = y + DIR[slot][1], nz = z + DIR[slot][2];
        if (inb(d, nx, ny, nz)) stamp[vidx(d, nx, ny, nz)] = epoch;
    }
}

// DIRTY_QUADS groups of four vertices per thread, one 16-byte load of their stamps each; the
// loads of a wave are contiguous. Space in the list is claimed with one atomic per block (a wave
// per block would make the claims on the one counter the cost of the pass).
constexpr int DIRTY_QUADS = 16;
__global__ __launch_bounds__(BLOCK) void k_dirty_collect(const uint32_t* stamp, i64 n, uint32_t epoch,
                                                         uint32_t* dirty, ull* dirty_ctr) {
    __shared__ int wsum[BLOCK / 64];
    __shared__ ull bbase;
    const i64 base = (i64)blockIdx.x * BLOCK * 4 * DIRTY_QUADS;
    uint64_t m = 0;  // bit 4k + j: vertex base + 4 (k BLOCK + threadIdx.x) + j
    for (int k = 0; k < DIRTY_QUADS; k++) {
        const i64 v0 = base + 4 * ((i64)k * BLOCK + threadIdx.x);
        uint64_t q = 0;
        if (v0 + 3 < n) {
            const uint4 u = *reinterpret_cast<const uint4*>(stamp + v0);
            q = (uint64_t)(u.x == epoch) | (uint64_t)(u.y == epoch) << 1 | (uint64_t)(u.z == epoch) << 2 |
                (uint64_t)(u.w == epoch) << 3;
        } else {
            for (int j = 0; j < 4; j++)
                if (v0 + j < n && stamp[v0 + j] == epoch) q |= (uint64_t)1 << j;
        }
        m |= q << (4 * k);
    }
    int wtotal;
    const int pre = wave_excl_scan(__popcll(m), wtotal);
    const int w = (int)(threadIdx.x >> 6);
    if (__lane_id() == 0) wsum[w] = wtotal;
    __syncthreads();
    int off = 0, tot = 0;
    for (int i = 0; i < BLOCK / 64; i++) {
        off += i < w ? wsum[i] : 0;
        tot += wsum[i];
    }
    if (threadIdx.x == 0) bbase = tot ? atomicAdd(dirty_ctr, (ull)tot) : 0;
    __syncthreads();
    ull at = bbase + (ull)(off + pre);
    while (m) {
        const int b = __ffsll((unsigned long long)m) - 1;
        m &= m - 1;
        dirty[at++] = (uint32_t)(base + 4 * ((i64)(b >> 2) * BLOCK + threadIdx.x) + (b & 3));
    }
}

// Filtration main_3d.cu:2405-2490: every vertex of an f-critical cell is pinned to f - eps.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_pin(const uint64_t* recs, ull n, const T* f, T* g, Dims d, Counts c,
                                               double eps) {
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const uint64_t r = recs[i];
    const i64 v = (i64)(r >> 7);
    const int lc = (int)(r & 127u);
    i64 x, y, z;
    vxyz(d, v, x, y, z);
    i64 w[4] = {v, -1, -1, -1};
    auto nb = [&](int k) { return vidx(d, x + DIR[k][0], y + DIR[k][1], z + DIR[k][2]); };
    if (lc >= LC_EDGE && lc < LC_TRI) {
        w[1] = nb(lc - LC_EDGE);
    } else if (lc >= LC_TRI && lc < LC_TET) {
        w[1] = nb(ST.tri_i[lc - LC_TRI]);
        w[2] = nb(ST.tri_j[lc - LC_TRI]);
    } else if (lc >= LC_TET) {
        w[1] = nb(ST.tet_s[lc - LC_TET][0]);
        w[2] = nb(ST.tet_s[lc - LC_TET][1]);
        w[3] = nb(ST.tet_s[lc - LC_TET][2]);
    }
    for (int k = 0; k < 4; k++)
        if (w[k] >= 0) g[w[k]] = EditArith<T>::snap(f[w[k]], eps);
}

struct PathList {
    int64_t* id;   // cell id (edge for descending, tet for ascending)
    int64_t* rec;  // recorded vertex / divergent tet
    ull* ctr;
    ull cap;
    // Every thread of the block must call this; threads with has = false add nothing.
    __device__ void push_block(bool has, i64 a, i64 b) const {
        ull at = block_alloc(ctr, has ? 1 : 0);
        if (has && at < cap) {
            id[at] = a;
            rec[at] = b;
        }
    }
};

// The separatrix checks read the pairings of f and g from pair words (pairs.h). Where branches are
// walked (connectivity mode), one thread per (start cell, branch) writes its result at a fixed
// position and a combine step per start cell applies the reference's "first branch that fails"
// rule and appends to the list in convergent code.

// Pair words (pairs.h) of every vertex of a field. Bound by memory: the values, the codes' words 0 and 1
// and the pair word, 24 bytes a vertex (512^3: 0.94 ms, 5.3 TB/s by the counters).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_pairs(const T* fld, CodeArray code, Dims d, i64 n, uint32_t* out) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (v >= n) return;
    i64 x, y, z;
    vxyz(d, v, x, y, z);
    out[v] = pair_word(fld, code, d, v, x, y, z);
}

// Where the pairings of f and g differ (pairs.h pair_mismatch), one byte per vertex, for every
// vertex. pg (nullable) receives g's pair words.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_mism_full(const T* g, CodeArray code, const uint32_t* pf, Dims d,
                                                     i64 n, uint8_t* mis, uint32_t* pg) {
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (v >= n) return;
    i64 x, y, z;
    vxyz(d, v, x, y, z);
    const uint32_t w = pair_word(g, code, d, v, x, y, z);
    mis[v] = (uint8_t)pair_mismatch(pf[v], w);
    if (pg) pg[v] = w;
}

// The same for the marked vertices alone (mark_vertex: the cubes around every vertex whose g code
// changed since the last check; a pair word reads nothing but star codes and, to find a tet's
// owner, the order of the values, which cannot change without the codes). A block takes the marks of
// 32 * BLOCK vertices, clears them, lists the marked vertices in LDS and spreads them over its
// threads, so that a few marks cost a pass over the bitmap (N / 8 bytes).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_mism_marked(const T* g, CodeArray code, const uint32_t* pf, Dims d,
                                                       i64 n, uint32_t* marks, uint8_t* mis) {
    __shared__ uint16_t list[32 * BLOCK];
    __shared__ int wsum[BLOCK / 64];
    const i64 w = (i64)blockIdx.x * BLOCK + threadIdx.x;
    uint32_t m = w < (n + 31) / 32 ? marks[w] : 0u;
    if (!__syncthreads_or(m != 0u)) return;
    if (m) marks[w] = 0u;
    int wt;
    int at = wave_excl_scan(__popc(m), wt);
    const int wv = (int)(threadIdx.x >> 6);
    if (__lane_id() == 0) wsum[wv] = wt;
    __syncthreads();
    int total = 0;
    for (int i = 0; i < BLOCK / 64; i++) {
        at += i < wv ? wsum[i] : 0;
        total += wsum[i];
    }
    for (; m; m &= m - 1) list[at++] = (uint16_t)(threadIdx.x * 32 + __builtin_ctz(m));
    __syncthreads();
    const i64 base = (i64)blockIdx.x * BLOCK * 32;
    for (int i = threadIdx.x; i < total; i += BLOCK) {
        const i64 v = base + list[i];
        i64 x, y, z;
        vxyz(d, v, x, y, z);
        mis[v] = (uint8_t)pair_mismatch(pf[v], pair_word(g, code, d, v, x, y, z));
    }
}

// The walks' table of the tet across each face, in LDS: a divergent read of it costs no memory
// access. Every thread of the block must call this.
__device__ __forceinline__ void load_across(uint8_t* across) {
    if (threadIdx.x < 24) across[threadIdx.x] = PT.across[threadIdx.x];
    __syncthreads();
}
__device__ __forceinline__ void load_slot_steps(const Dims& d, i64* step) {
    if (threadIdx.x < 14) step[threadIdx.x] = slot_step(d, threadIdx.x);
    __syncthreads();
}

// get_false_ds_vpath (main_3d.cu:4837-4959). The reference compares the f and g edges of both
// end vertices of every f-critical edge (v1, v2), v1 > v2, and records v1 if they differ there, else
// v2 if they do there. Taken from the vertices: each vertex that differs records its f-critical
// edges (bits of its f-critical mask) except those whose larger end differs too and records them.
// A thread tests 16 vertices with one load, so an edge costs nothing unless an end differs (the
// pass reads N bytes; 512^3 fBm, 11 checks: 5.8 ms with a thread and 36 bytes per edge -> 1.4 ms).
constexpr int DS_V = 16;
__global__ __launch_bounds__(BLOCK) void k_ds_list(const uint8_t* mis, const uint64_t* critf, Dims d, Counts c, i64 n,
                                                   PathList out) {
    __shared__ i64 step[16];
    load_slot_steps(d, step);
    const i64 v0 = ((i64)blockIdx.x * BLOCK + threadIdx.x) * DS_V;
    uint32_t hit = 0;
    if (v0 < n) {
        const uint4 q = *reinterpret_cast<const uint4*>(mis + v0);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int k = 0; k < DS_V; k++) hit |= ((w[k >> 2] >> (8 * (k & 3) + 6)) & 1u) << k;
        if (n - v0 < DS_V) hit &= (1u << (n - v0)) - 1u;
    }
    // f-critical edges of vertex v that v records
    auto edges = [&](i64 v) {
        uint32_t e = (uint32_t)(critf[v] >> LC_EDGE) & 0x3FFFu;
        for (uint32_t up = e & 0x1555u; up; up &= up - 1) {  // even slots lead to larger indices
            const int s = __builtin_ctz(up);
            if (mis[v + step[s]] & MIS_SLOT) e &= ~(1u << s);
        }
        return e;
    };
    int cnt = 0;
    for (uint32_t h = hit; h; h &= h - 1) cnt += __popc(edges(v0 + __builtin_ctz(h)));
    if (!__syncthreads_or(cnt)) return;
    ull at = block_alloc(out.ctr, cnt);
    for (uint32_t h = hit; h; h &= h - 1) {
        const i64 v = v0 + __builtin_ctz(h);
        i64 x, y, z;
        vxyz(d, v, x, y, z);
        for (uint32_t e = edges(v); e; e &= e - 1) {
            if (at < out.cap) {
                out.id[at] = edge_id_dir(d, c, x, y, z, __builtin_ctz(e));
                out.rec[at] = v;
            }
            at++;
        }
    }
}

// Ascending checks (is_false main_3d.cu:4437-4497 from both cofacets of every f-critical face) in
// geometry mode. f does not change, so the tets of f's ascending paths are listed once per run: the
// steps of face i, first cofacet's path then the second's, at [off[i], off[i + 1]), one word per
// step. A check then asks for every step, independently of all others, whether f and g pair its tet
// alike (k_as_bad: a coalesced 4-byte read and a byte of mis per step, one bit out), and the first
// differing step of a face is its first set bit (k_as_list). No check walks a path, and a check
// costs the same whatever changed: 512^3 fBm, 320 M steps, 11 checks: 41 ms when each branch was
// walked by a thread over star codes -> 15 ms with the refresh of mis; a 33 x 32 x 34 mixture, whose
// longest path has some hundred steps, 230 -> 33 us per check.
// A step word is 12 v + 2 type + 1 for the first step of a path (12 N < 2^32).
__device__ __forceinline__ uint32_t step_word(const TetAt& a, bool first) {
    return (uint32_t)a.v * 12u + 2u * (uint32_t)a.type + (first ? 1u : 0u);
}

// The paths of all faces, counted (cnt[i] = steps of face i, *total their sum) or, with FILL,
// listed. Path lengths are heavy-tailed, so a lane takes a new face whenever its walks end, and each
// loop round every busy lane advances by one step: one 4-byte read (the pair word) and one LDS read.
// A wave claims AS_WS_CHUNK faces at a time from the shared counter (*next) and hands them to its
// idle lanes. Bound by the latency of the pair-word reads, which lie near one another (faces are
// listed in about vertex order). Walking twice is cheaper than keeping the counted steps.
// (512^3 fBm: the count 54 -> 5 ms, the fill 19 -> 7 ms against walks over star codes.)
constexpr unsigned AS_WS_BLOCKS = 2048;  // eight blocks per CU
// Beside the repair sweeps (on a second stream) the walk takes half the wave slots: its waves
// run until every face is walked, so with all slots the sweeps' kernels would wait for it.
constexpr unsigned AS_WS_BLOCKS_SIDE = 1024;
constexpr ull AS_WS_CHUNK = 1024;
template <bool FILL>
__global__ __launch_bounds__(BLOCK) void k_as_walk(const uint64_t* fcf, ull nf, const uint32_t* pw, Dims d, i64 cap,
                                                   uint32_t* cnt, const uint32_t* off, uint32_t* steps, ull* next,
                                                   ull* total, ull* walk_ctr) {
    __shared__ uint8_t across[24];
    __shared__ uint8_t start[72];
    if (threadIdx.x >= 64 && threadIdx.x < 64 + 72) start[threadIdx.x - 64] = PT.start[(threadIdx.x - 64) >> 1][threadIdx.x & 1];
    load_across(across);
    const int lane = __lane_id();
    bool busy = false, first = false;
    ull j = 0;
    TetAt a{-1, 0, 0, 0, 0}, b{-1, 0, 0, 0, 0};  // the tet being visited; the second path's start
    uint32_t at = 0;                              // FILL: next position
    i64 n = 0;
    ull sum = 0;
    ull cb = 0, ce = 0;  // the wave's unclaimed faces [cb, ce) (wave-uniform)
    bool dry = false;    // the shared counter has passed nf (wave-uniform)
    for (;;) {
        const ull idle = __ballot(!busy);
        if (idle && !(dry && cb >= ce)) {
            const ull nid = (ull)__popcll(idle);
            const ull rank = (ull)__popcll(idle & ((1ull << lane) - 1ull));
            const ull avail = ce - cb;
            ull jj = nf;  // this lane's new face, if idle (nf: none)
            if (nid <= avail) {
                jj = cb + rank;
                cb += nid;
            } else {
                ull nc = 0;
                if (!dry) {
                    const int leader = __ffsll((unsigned long long)idle) - 1;
                    if (lane == leader) nc = atomicAdd(next, AS_WS_CHUNK);
                    const unsigned lo = __shfl((unsigned)(nc & 0xffffffffu), leader, 64);
                    const unsigned hi = __shfl((unsigned)(nc >> 32), leader, 64);
                    nc = ((ull)hi << 32) | lo;
                    dry = nc >= nf;
                }
                if (rank < avail) jj = cb + rank;
                else if (!dry) jj = nc + (rank - avail);
                if (!dry) {
                    ce = nc + AS_WS_CHUNK < nf ? nc + AS_WS_CHUNK : nf;
                    cb = nc + (nid - avail) < ce ? nc + (nid - avail) : ce;
                } else {
                    cb = ce;
                }
            }
            if (!busy && jj < nf) {
                j = jj;
                const uint64_t r = fcf[j];
                const i64 v = (i64)(r >> 7);
                const int lt = (int)(r & 127u) - LC_TRI;
                i64 x, y, z;
                vxyz(d, v, x, y, z);
                a = start_tet(d, v, (int)x, (int)y, (int)z, start[2 * lt]);
                b = start_tet(d, v, (int)x, (int)y, (int)z, start[2 * lt + 1]);
                if (a.v < 0) {
                    a = b;
                    b.v = -1;
                }
                n = 0;
                first = true;
                if (FILL) at = off[j];
                busy = a.v >= 0;
                if (!FILL && !busy) cnt[j] = 0;
            }
        }
        if (__ballot(busy) == 0 && dry && cb >= ce) break;
        if (busy) {
            const uint32_t out = pw_out(pw[a.v], a.type);
            bool end = out == PW_NONE;
            if (!end) {
                if (FILL) steps[at++] = step_word(a, first);
                first = false;
                n++;
                cross_face(d, a, across[4 * a.type + (int)out]);
                end = a.v < 0;
                if (!end && n > 2 * cap) {  // no V-path is that long
                    atomicAdd(walk_ctr, 1ull);
                    end = true;
                    b.v = -1;
                }
            }
            if (end) {
                a = b;
                b.v = -1;
                first = true;
                busy = a.v >= 0;
                if (!FILL && !busy) {
                    cnt[j] = (uint32_t)n;
                    sum += (ull)n;
                }
            }
        }
    }
    if (!FILL) {
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_down((unsigned long long)sum, o, 64);
        if (lane == 0 && sum) atomicAdd(total, sum);
    }
}

// Bit s of bad: f and g pair the tet of step s differently. Each wave covers AS_BAD_WORDS x 64
// consecutive steps, lane l the steps 64 k + l, with that many independent reads in flight per lane;
// a 64-step word is one ballot.
constexpr int AS_BAD_WORDS = 8;
__global__ __launch_bounds__(BLOCK) void k_as_bad(ull total, const uint32_t* steps, const uint8_t* mis, uint64_t* bad) {
    const ull w = (ull)blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    const int lane = (int)(threadIdx.x & 63u);
    const ull base = w * (64 * AS_BAD_WORDS);
    uint32_t q[AS_BAD_WORDS], m[AS_BAD_WORDS];
#pragma unroll
    for (int k = 0; k < AS_BAD_WORDS; k++) {
        const ull s = base + 64 * k + lane;
        q[k] = s < total ? steps[s] : 0u;
    }
#pragma unroll
    for (int k = 0; k < AS_BAD_WORDS; k++) m[k] = mis[q[k] / 12u];
#pragma unroll
    for (int k = 0; k < AS_BAD_WORDS; k++) {
        const ull s = base + 64 * k + lane;
        const uint64_t r = __ballot(s < total && ((m[k] >> ((q[k] % 12u) >> 1)) & 1u) != 0u);
        if (lane == 0 && base + 64 * k < total) bad[(base >> 6) + k] = r;
    }
}

// First set bit of bits in [s, b), or b.
__device__ __forceinline__ uint32_t next_set(const uint64_t* bits, uint32_t s, uint32_t b) {
    uint32_t r = b;
    for (uint32_t w = s >> 6; s < b && w <= (b - 1) >> 6 && r == b; w++) {
        const uint32_t lo = w << 6;
        uint64_t m = bits[w];
        if (lo < s) m &= ~0ull << (s - lo);
        if (b - lo < 64) m &= (1ull << (b - lo)) - 1ull;
        if (m) r = lo + (uint32_t)__builtin_ctzll(m);
    }
    return r;
}

// The reference takes a face's first cofacet whose path differs, and the first differing tet on
// that path: the first set bit among the face's steps. AS_FACES faces per thread and one list
// claim per block.
// A block whose faces' steps hold no set bit reads their words of bad and leaves (a late check with
// a few differing tets; 512^3 fBm, 11 checks: 3.8 -> 1.9 ms). ids = 0 leaves out the start tets, which only
// callers of the lists ask for: finding one walks back over its path's steps.
constexpr int AS_FACES = 8;
__global__ __launch_bounds__(BLOCK) void k_as_list(ull nf, const uint32_t* off, const uint64_t* bad,
                                                   const uint32_t* steps, Dims d, int ids, PathList out) {
    const ull f0 = (ull)blockIdx.x * AS_FACES * BLOCK, f1 = f0 + AS_FACES * BLOCK < nf ? f0 + AS_FACES * BLOCK : nf;
    const uint32_t s0 = off[f0], s1 = off[f1];
    bool some = false;
    if (s0 < s1)
        for (uint32_t w = (s0 >> 6) + threadIdx.x; w <= (s1 - 1) >> 6; w += BLOCK) some = some || bad[w] != 0;
    if (!__syncthreads_or(some)) return;
    uint32_t hit[AS_FACES];
    int cnt = 0;
#pragma unroll
    for (int k = 0; k < AS_FACES; k++) {
        const ull i = ((ull)blockIdx.x * AS_FACES + k) * BLOCK + threadIdx.x;
        hit[k] = ~0u;
        if (i < nf) {
            const uint32_t a = off[i], b = off[i + 1];
            const uint32_t p = next_set(bad, a, b);
            if (p < b) {
                hit[k] = p;
                cnt++;
            }
        }
    }
    if (!__syncthreads_or(cnt)) return;
    ull at = block_alloc(out.ctr, cnt);
#pragma unroll
    for (int k = 0; k < AS_FACES; k++) {
        if (hit[k] == ~0u) continue;
        if (at < out.cap) {
            uint32_t p = hit[k];
            const uint32_t q = steps[p];
            if (ids) {
                uint32_t s = q;
                while (!(s & 1u)) s = steps[--p];  // back to the path's first tet
                out.id[at] = tet_id_of_vertex(d, s / 12u, (int)((s % 12u) >> 1));
            }
            out.rec[at] = tet_id_of_vertex(d, q / 12u, (int)((q % 12u) >> 1));
        }
        at++;
    }
}

// Ascending branch walks, thread = (face, cofacet k): connectivity mode, and geometry mode on
// grids whose paths are not listed. maxlab (nullable) holds f's maximum per start: a branch whose
// maximum in g equals it does not fail (get_false_as_vpath_connectivity main_3d.cu:4761-4835). With
// lab_from_f the start faces are g's critical faces and f's label is found here (the maximum f
// reaches from the tet when f leaves the face critical, -1 otherwise: labels exist only for f's
// critical faces, main_3d.cu:4689-4759). res[2*j] = start tet if the branch fails else -1,
// res[2*j+1] = the divergent tet. A chain of dependent 4-byte reads (129 x 96 x 111 mixture in
// float64: 3.1 ms per check over star codes and ids, now 0.06).
__global__ __launch_bounds__(BLOCK) void k_as_branch(const uint64_t* fcf, ull n, const int64_t* maxlab, int lab_from_f,
                                                     const uint64_t* critf, const uint32_t* pf, const uint32_t* pg,
                                                     Dims d, i64 cap, int64_t* res, ull* walk_ctr) {
    __shared__ uint8_t across[24];
    load_across(across);
    const ull j = (ull)blockIdx.x * BLOCK + threadIdx.x;
    if (j >= 2 * n) return;
    const uint64_t r = fcf[j >> 1];
    const i64 v = (i64)(r >> 7);
    const int lc = (int)(r & 127u);
    i64 x, y, z;
    vxyz(d, v, x, y, z);
    const TetAt a = start_tet(d, v, (int)x, (int)y, (int)z, PT.start[lc - LC_TRI][j & 1]);
    bool ovf = false, found = false;
    TetAt div = a;
    bool check = a.v >= 0;
    if (check && maxlab) check = paired_max(d, pg, across, a, cap, ovf) != maxlab[j];
    if (check && lab_from_f) {
        const bool fcrit = ((critf[v] >> lc) & 1ull) != 0;
        const i64 lab = fcrit ? paired_max(d, pf, across, a, cap, ovf) : -1;
        check = paired_max(d, pg, across, a, cap, ovf) != lab;
    }
    if (check) found = path_mismatch(d, pf, pg, across, a, cap, div, ovf);
    res[2 * j] = found ? tet_id_at(d, a) : -1;
    res[2 * j + 1] = found ? tet_id_at(d, div) : -1;
    if (ovf) atomicAdd(walk_ctr, 1ull);
}

__global__ __launch_bounds__(BLOCK) void k_as_combine(const int64_t* res, ull n, PathList out) {
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    bool has = false;
    i64 a = -1, b = -1;
    if (i < n) {
        const int64_t* p = res + 4 * i;
        has = p[0] >= 0 || p[2] >= 0;
        a = p[0] >= 0 ? p[0] : p[2];
        b = p[0] >= 0 ? p[1] : p[3];
    }
    out.push_block(has, a, b);
}

// Endpoint k of the f-critical edge of a record: the larger index first.
__device__ __forceinline__ i64 edge_end(const i64* step, uint64_t r, int k) {
    const i64 v = (i64)(r >> 7), w = v + step[(int)(r & 127u) - LC_EDGE];
    return k == 0 ? (v > w ? v : w) : (v > w ? w : v);
}

// Endpoint labels of f (get_orginal_saddle_min_pairs / _max_pairs, main_3d.cu:4613-4759), one
// thread per (f-critical edge, endpoint) and per (f-critical face, cofacet); ascending labels
// are indexed by face (resolution of the shadowed index at main_3d.cu:4750).
__global__ __launch_bounds__(BLOCK) void k_labels(const uint64_t* fce, ull ne, const uint64_t* fcf, ull nf,
                                                  const uint32_t* pf, Dims d, i64 cap, int64_t* minlab,
                                                  int64_t* maxlab, ull* walk_ctr) {
    __shared__ uint8_t across[24];
    __shared__ i64 step[16];
    load_across(across);
    load_slot_steps(d, step);
    const ull j = (ull)blockIdx.x * BLOCK + threadIdx.x;
    bool ovf = false;
    if (j < 2 * ne) {
        minlab[j] = paired_min(pf, step, edge_end(step, fce[j >> 1], (int)(j & 1)), cap, ovf);
    } else if (j < 2 * ne + 2 * nf) {
        const ull jj = j - 2 * ne;
        const uint64_t r = fcf[jj >> 1];
        const i64 v = (i64)(r >> 7);
        i64 x, y, z;
        vxyz(d, v, x, y, z);
        const TetAt a = start_tet(d, v, (int)x, (int)y, (int)z, PT.start[(int)(r & 127u) - LC_TRI][jj & 1]);
        maxlab[jj] = paired_max(d, pf, across, a, cap, ovf);
    }
    if (ovf) atomicAdd(walk_ctr, 1ull);
}

// get_false_ds_vpath_connectivity main_3d.cu:4961-5062: thread = (f-critical edge, endpoint)
// walks g's descending path; res[4*i + 2*k] = reached g minimum, res[4*i + 2*k + 1] = first
// vertex on the walk whose f and g pairings differ.
__global__ __launch_bounds__(BLOCK) void k_ds_branch(const uint64_t* fce, ull n, const uint32_t* pf,
                                                     const uint32_t* pg, Dims d, i64 cap, int64_t* res,
                                                     ull* walk_ctr) {
    __shared__ i64 step[16];
    load_slot_steps(d, step);
    const ull j = (ull)blockIdx.x * BLOCK + threadIdx.x;
    if (j >= 2 * n) return;
    i64 trouble = -1;
    bool ovf = false;
    res[2 * j] = g_min_of(pf, pg, step, edge_end(step, fce[j >> 1], (int)(j & 1)), trouble, cap, ovf);
    res[2 * j + 1] = trouble;
    if (ovf) atomicAdd(walk_ctr, 1ull);
}

// The reference carries trouble_maker from the first endpoint's walk into the second.
__global__ __launch_bounds__(BLOCK) void k_ds_combine(const uint64_t* fce, ull n, const int64_t* res,
                                                      const int64_t* minlab, Dims d, Counts c, PathList out) {
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    bool has = false;
    i64 e = -1, rec = -1;
    if (i < n) {
        const uint64_t r = fce[i];
        e = local_cell_id(d, c, (i64)(r >> 7), (int)(r & 127u));
        const int64_t* p = res + 4 * i;
        bool bad1 = p[0] != minlab[2 * i];
        bool bad2 = p[2] != minlab[2 * i + 1];
        has = bad1 || bad2;
        rec = bad1 ? p[1] : (p[1] != -1 ? p[1] : p[3]);
    }
    out.push_block(has, e, rec);
}

// 2-saddle walls, get_false_ds_wall main_3d.cu:5064-5133, made deterministic: from each f-critical
// face, a depth-first walk over f's face -> edge -> paired-face steps with a stack and a visited set
// of its own (the reference shares one stack between threads, defects D2-D5), to the first edge met
// whose f partner exists and differs from its g partner. The walks are not made: walls.h finds the
// faces from which a mismatched edge is reached, backwards and once for all walls, and follows one
// chain per open f-critical face. (A thread per face with its own visited set searched every wall, most
// of them to their end; the longest of a few thousand faces set the time: 96 x 95 x 97 fBm, 7 ms per
// launch and 28 ms per check; now 0.5 ms per check, 0.33 of it the serial levels of k_wall_levels.)
//
// Bit 16 v + kind of open: the face of that kind anchored at v is open.
__device__ __forceinline__ bool wall_open(const uint32_t* open, uint32_t id) {
    const uint64_t b = (uint64_t)(id / 12u) * 16u + id % 12u;
    return ((open[b >> 5] >> (b & 31u)) & 1u) != 0;
}
// Newly opened faces gather in LDS and enter the queue with one claim per block (a claim per wave and
// face made k_wall_seeds 765 us instead of 97 on average, 96 x 95 x 97); past WALL_BUF of them each claims a slot of its own.
constexpr uint32_t WALL_BUF = 2048;
struct WallQueue {
    uint32_t n;
    ull base;
    uint32_t id[WALL_BUF];
    // every thread of the block: before the first add
    __device__ __forceinline__ void clear() {
        if (threadIdx.x == 0) n = 0;
        __syncthreads();
    }
    __device__ __forceinline__ void add(uint32_t* open, uint32_t face, uint32_t* queue, ull cap, ull* ctr) {
        const uint64_t b = (uint64_t)(face / 12u) * 16u + face % 12u;
        const uint32_t bit = 1u << (b & 31u);
        if (atomicOr(open + (b >> 5), bit) & bit) return;
        const uint32_t k = atomicAdd(&n, 1u);
        if (k < WALL_BUF) {
            id[k] = face;
        } else {
            const ull at = atomicAdd(ctr, 1ull);
            if (at < cap) queue[at] = face;
        }
    }
    // every thread of the block: after the last add. Returns the end of the queue; past cap the faces are
    // counted but not kept.
    __device__ __forceinline__ ull flush(uint32_t* queue, ull cap, ull* ctr) {
        __syncthreads();
        const uint32_t m = n < WALL_BUF ? n : WALL_BUF;
        if (threadIdx.x == 0) base = atomicAdd(ctr, (ull)m);
        __syncthreads();
        const ull b = base;
        for (uint32_t k = threadIdx.x; k < m; k += blockDim.x)
            if (b + k < cap) queue[b + k] = id[k];
        return b + m;
    }
};

// Tables of the wall kernels in LDS. Every thread of the block must call load().
static_assert(sizeof(RuleTables) / 4 <= BLOCK && sizeof(WallTables) <= BLOCK, "one table word per thread");
struct WallLds {
    RuleTables tb;
    WallTables wt;
    int32_t off[15];
    __device__ __forceinline__ void load(const Dims& d) {
        if (threadIdx.x < sizeof(RuleTables) / 4)
            reinterpret_cast<uint32_t*>(&tb)[threadIdx.x] = reinterpret_cast<const uint32_t*>(&RT)[threadIdx.x];
        if (threadIdx.x < sizeof(WallTables))
            reinterpret_cast<uint8_t*>(&wt)[threadIdx.x] = reinterpret_cast<const uint8_t*>(&WT)[threadIdx.x];
        if (threadIdx.x < 15) off[threadIdx.x] = threadIdx.x == 14 ? 0 : (int32_t)slot_step(d, threadIdx.x);
        __syncthreads();
    }
};
template <class T>
struct WallArgs {
    const T* f;
    const T* g;
    CodeArray cf, cg;
    Dims d;
    Counts c;
    uint32_t* open;
    uint32_t* queue;
    ull cap;
    ull* ctr;  // faces in the queue
};
#define DMTZ_WALL_GRAPH(a, lds)                                                                                    \
    NullSink none;                                                                                                 \
    const LocalRules<T, NullSink, CodeArray> rules{(a).f, (a).cf, (a).g, (a).cg, nullptr, &(lds).tb, (lds).off,    \
                                                   (a).d, (a).c,  0.0,   0,      none};                            \
    const WallGraph<T, CodeArray> graph{rules, &(lds).wt};                                                         \
    using At = typename WallGraph<T, CodeArray>::At

// The faces of every mismatched edge, each edge taken at its owner in f.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_wall_seeds(WallArgs<T> a) {
    __shared__ WallLds lds;
    __shared__ WallQueue next;
    next.clear();
    lds.load(a.d);
    DMTZ_WALL_GRAPH(a, lds);
    const i64 v = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (v < a.c.N)
        graph.mismatched_edges((uint32_t)v, [&](At e) {
            graph.faces_of(e, [&](At t) { next.add(a.open, graph.face_id(t), a.queue, a.cap, a.ctr); });
        });
    next.flush(a.queue, a.cap, a.ctr);
}

// One level: the faces that lead on to the queue's faces [from, to).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_wall_level(WallArgs<T> a, ull from, ull to) {
    __shared__ WallLds lds;
    __shared__ WallQueue next;
    next.clear();
    lds.load(a.d);
    DMTZ_WALL_GRAPH(a, lds);
    const ull i = from + (ull)blockIdx.x * BLOCK + threadIdx.x;
    if (i < to)
        graph.leading_to(graph.face_at(a.queue[i]),
                         [&](At t) { next.add(a.open, graph.face_id(t), a.queue, a.cap, a.ctr); });
    next.flush(a.queue, a.cap, a.ctr);
}

// All levels from there on in one block, which only has to wait for itself between them: levels are
// many (as long as the longest chain) and small. Every face enters the queue at most once, so the
// levels end; a queue that is full ends them too.
constexpr int WALL_BLOCK = 1024;
template <class T>
__global__ __launch_bounds__(WALL_BLOCK) void k_wall_levels(WallArgs<T> a, ull from, ull to) {
    __shared__ WallLds lds;
    __shared__ WallQueue next;
    lds.load(a.d);
    DMTZ_WALL_GRAPH(a, lds);
    while (from < to && to <= a.cap) {
        next.clear();
        for (ull i = from + threadIdx.x; i < to; i += WALL_BLOCK)
            graph.leading_to(graph.face_at(a.queue[i]),
                             [&](At t) { next.add(a.open, graph.face_id(t), a.queue, a.cap, a.ctr); });
        from = to;
        to = next.flush(a.queue, a.cap, a.ctr);
        __threadfence();
        __syncthreads();  // the block reads what it has queued
    }
}

// The chain of every open f-critical face to its first mismatched edge; a face whose chain runs in a
// circle is listed in ovf for the search.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_wall_chain(WallArgs<T> a, const uint64_t* starts, ull n, PathList out,
                                                      uint32_t* ovf, ull* ovf_ctr) {
    __shared__ WallLds lds;
    lds.load(a.d);
    DMTZ_WALL_GRAPH(a, lds);
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    bool has = false;
    i64 face = -1, edge = -1;
    if (i < n) {
        const uint64_t r = starts[i];
        const At t{(uint32_t)(r >> 7), (int)(r & 127u) - LC_TRI};
        At e{0, 0};
        if (wall_open(a.open, graph.face_id(t))) {
            i64 steps;
            if (graph.follow(t, e, [&](uint32_t id) { return wall_open(a.open, id); }, steps) == 1) {
                has = true;
                face = local_cell_id(a.d, a.c, (i64)(r >> 7), (int)(r & 127u));
                edge = rules.edge_number(e);
            } else {
                ovf[atomicAdd(ovf_ctr, 1ull)] = (uint32_t)i;
            }
        }
    }
    out.push_block(has, face, edge);
}

// The search itself, for the faces whose chain runs in a circle, and for grids whose faces do not fit the
// queue's numbers. A face is marked when popped; its edges are taken in the order (v1,v2), (v1,v3),
// (v2,v3) and pushed in that order, so the last is popped first.
//
// Thread t of the launch walks start first + t (or sel[first + t]) with its own part of scratch
// (2 * slots + 2 entries: the visited set and the stack of Repair::wall_walk). A walk that
// outgrows its set is listed in ovf, to be walked again with more slots.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_ds_wall(const uint64_t* starts, const uint32_t* sel, ull first, ull n,
                                                   const T* f, CodeArray cf, const T* g, CodeArray cg,
                                                   Dims d, Counts c, uint32_t* scratch, uint32_t slots, PathList out,
                                                   uint32_t* ovf, ull* ovf_ctr) {
    const ull t = (ull)blockIdx.x * BLOCK + threadIdx.x;
    if (first + t >= n) return;
    const ull s = sel ? (ull)sel[first + t] : first + t;
    const uint64_t r = starts[s];
    const i64 face = local_cell_id(d, c, (i64)(r >> 7), (int)(r & 127u));
    Repair<T, NullSink, CodeArray> R(f, cf, g, cg, d, c, nullptr, 0, 0, 0, NullSink{});
    uint32_t* set = scratch + (size_t)t * (2 * (size_t)slots + 2);
    i64 found = -1;
    const bool overflow = R.wall_walk(face, set, set + slots, slots, found);
    if (overflow) {
        ovf[atomicAdd(ovf_ctr, 1ull)] = (uint32_t)s;
    } else if (found >= 0) {
        const ull at = atomicAdd(out.ctr, 1ull);
        if (at < out.cap) {
            out.id[at] = face;
            out.rec[at] = found;
        }
    }
}

// fix_as_vpath / fix_ds_vpath / fix_ds_wall main_3d.cu:5135-5413
template <class T>
__global__ __launch_bounds__(BLOCK) void k_fix_paths(const int64_t* as_rec, ull n_as, const int64_t* ds_rec, ull n_ds,
                                                     const int64_t* wall_rec, ull n_wall, const T* f,
                                                     CodeArray cf, const T* g, CodeArray cg, Dims d,
                                                     Counts c, const uint8_t* counter, double eps, double range,
                                                     int edit_type, TargetSink sink) {
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    Repair<T, HoldSink, CodeArray> R(f, cf, g, cg, d, c, counter, eps, range, edit_type, HoldSink{sink, 0u, 0u, 0u, 0u, 0});
    if (i < n_as) R.fix_as_vpath(as_rec[i]);
    else if (i < n_as + n_ds) R.fix_ds_vpath(ds_rec[i - n_as]);
    else if (i < n_as + n_ds + n_wall) R.fix_ds_wall(wall_rec[i - n_as - n_ds]);
    R.sink.flush();
}

// Dense pairing arrays for tests (dmtz_gradient_*): one thread per cell of each dimension.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_pairing(const T* fld, CodeArray code, Dims d, Counts c, int dim, ull n,
                                                   int64_t* out) {
    const ull i = (ull)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    FieldGrad<T, CodeArray> X(fld, code, d, c);
    switch (dim) {
        case 0: out[i] = X.pv((i64)i); break;
        case 1: out[i] = X.pe((i64)i); break;
        case 2: out[i] = X.pf((i64)i); break;
        default: out[i] = X.pt((i64)i); break;
    }
}

inline unsigned nblocks(ull n) { return (unsigned)((n + BLOCK - 1) / BLOCK); }

// Grid of a kernel that reads its element count on the device and strides over it: sized for
// the host's estimate of the count, at least one block and at most STRIDE_BLOCKS (eight blocks
// per CU of a 256-CU device).
constexpr ull STRIDE_BLOCKS = 2048;
inline unsigned stride_blocks(ull estimate) {
    const ull b = nblocks(estimate);
    return (unsigned)(b < 1 ? 1 : (b > STRIDE_BLOCKS ? STRIDE_BLOCKS : b));
}

// The dirty stars are collected by one pass over all N stamps (k_dirty_mark + k_dirty_collect)
// once the (changed vertex, star slot) pairs reach N / DIRTY_DENSE, and by one returning atomic
// per pair (k_dirty) below that.
constexpr ull DIRTY_DENSE = 256;

}  // namespace

// ================================================================================================
// Context
// ================================================================================================
struct dmtz_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    // device buffers
    void* d_f = nullptr;
    void* d_g = nullptr;
    size_t field_bytes = 0;
    uint8_t* d_counter = nullptr;
    uint32_t* d_stamp = nullptr;    // edit-set dedup stamps
    uint32_t* d_dstamp = nullptr;   // dirty-star dedup stamps
    uint32_t* d_targets = nullptr;  // edit set
    uint32_t* d_changed = nullptr;  // edited vertices whose value changed
    uint32_t* d_dirty = nullptr;    // vertices whose g star code must be re-evaluated
    uint64_t* d_code_f = nullptr;   // star codes of f and g, word by word (CodeArray)
    uint64_t* d_code_g = nullptr;
    MaskArray d_critf = {nullptr, nullptr};  // f-critical status of every vertex's local cells
    MaskArray d_mm = {nullptr, nullptr};     // mismatched cells each vertex owns in g
    uint32_t* d_tile_nz = nullptr;  // per EMIT_TILE vertices: how many have a nonzero d_mm
    uint64_t* d_rec = nullptr;    // 4 mismatch record lists of rec_cap entries
    uint64_t* d_fc = nullptr;     // 4 f-critical lists of fc_cap entries
    int64_t* d_path = nullptr;    // ds id/rec, as id/rec, wall id/rec (fc_cap each)
    bool side_stream = true;  // off in batch lanes: no second stream for the path precompute
    uint32_t* d_pairf = nullptr;     // pair words of f and, where branches are walked, of g
    uint32_t* d_pairg = nullptr;
    uint8_t* d_mis = nullptr;        // per vertex: where the pairings of f and g differ
    uint32_t* d_marks = nullptr;     // vertices whose d_mis is to be refreshed at the next path check
    uint64_t* d_as_bad = nullptr;    // per listed step: f and g pair its tet differently
    size_t pairf_cap = 0, pairg_cap = 0, mis_cap = 0, marks_cap = 0, as_bad_cap = 0;
    hipStream_t as_stream = nullptr;  // the ascending-path precompute, overlapping the first sweeps
    hipEvent_t as_ev_fork = nullptr, as_ev_count = nullptr, as_ev_done = nullptr;
    ull* h_as_total = nullptr;        // pinned: total steps of the listed paths
    uint32_t* d_wall_scr = nullptr;  // wall walks: per-thread visited sets and stacks
    size_t wall_scr_cap = 0;
    uint32_t* d_wall_ovf = nullptr;  // wall walks to repeat with more slots (two lists)
    size_t wall_ovf_cap = 0;
    uint32_t* d_wall_open = nullptr;   // open faces (16 bits per vertex) and their queue
    uint32_t* d_wall_queue = nullptr;
    size_t wall_open_cap = 0, wall_queue_cap = 0;
    int64_t* d_labels = nullptr;  // min labels (2 per f-critical edge), max labels (2 per face)
    int64_t* d_walk = nullptr;    // per-branch walk results (4 per start cell)
    ull* d_ctr = nullptr;
    ull* h_ctr = nullptr;
    i64 cap_n = 0;   // vertices the buffers are sized for
    ull rec_cap = 0;
    ull fc_cap = 0;
    uint32_t epoch = 0;
    // Sizes at which the driver changes its route; the reasons stand where each is used. (The tests lower
    // them, so that small grids take every route: testing.h.)
    struct {
        i64 plane_min = (i64)1 << 19;   // vertices from which the dense classification runs over bit planes
        i64 code_small = (i64)1 << 16;  // vertices up to which every star is re-evaluated
        ull target_dense = 256;         // records from which an edit set is marked: N over this
        ull path_steps = (ull)1 << 32;  // steps from which ascending paths are walked, not listed
        ull wall_level = 16384;         // faces from which a wall level gets a launch of its own
        ull wall_queue = 0;             // open faces a wall queue holds at first, 0: one per vertex
    } lim;
    std::vector<int64_t> traj;
    double phase[6] = {0, 0, 0, 0, 0, 0};
    // live timing of the dense detection kernel on the context stream (HIP events)
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double det_launches = 0, det_ms = 0, det_bytes = 0, det_voxels = 0;
    std::vector<dmtz_ctx*> workers;  // batch lanes: contexts of their own (stream, buffers)
    double dirty_total = 0;  // star codes re-evaluated after edits in the last correction
    int64_t stalls = 0, finished = 0, radius = 0;  // finisher outcome of the last correction
    // precomputed ascending separatrix paths of f (geometry mode)
    uint32_t* d_as_cnt = nullptr;  // steps per f-critical face, then scanned into d_as_off
    uint32_t* d_as_off = nullptr;
    uint32_t* d_as_steps = nullptr;
    void* d_scan_tmp = nullptr;
    size_t as_cnt_cap = 0, as_off_cap = 0, as_steps_cap = 0, scan_tmp_cap = 0, labels_cap = 0, walk_cap = 0;
};

namespace {

void free_bufs(dmtz_ctx* ctx) {
    (void)hipFree(ctx->d_f);
    (void)hipFree(ctx->d_g);
    (void)hipFree(ctx->d_counter);
    (void)hipFree(ctx->d_stamp);
    (void)hipFree(ctx->d_dstamp);
    (void)hipFree(ctx->d_targets);
    (void)hipFree(ctx->d_changed);
    (void)hipFree(ctx->d_dirty);
    (void)hipFree(ctx->d_code_f);
    (void)hipFree(ctx->d_code_g);
    for (MaskArray* m : {&ctx->d_critf, &ctx->d_mm}) {
        (void)hipFree(m->lo);
        (void)hipFree(m->hi);
        *m = MaskArray{nullptr, nullptr};
    }
    (void)hipFree(ctx->d_tile_nz);
    ctx->d_tile_nz = nullptr;
    ctx->d_f = ctx->d_g = nullptr;
    ctx->d_counter = nullptr;
    ctx->d_stamp = ctx->d_dstamp = ctx->d_targets = ctx->d_changed = ctx->d_dirty = nullptr;
    ctx->d_code_f = ctx->d_code_g = nullptr;
    ctx->field_bytes = 0;
    ctx->cap_n = 0;
}

void free_rec(dmtz_ctx* ctx) {
    (void)hipFree(ctx->d_rec);
    ctx->d_rec = nullptr;
    ctx->rec_cap = 0;
}

void free_paths(dmtz_ctx* ctx) {
    (void)hipFree(ctx->d_as_cnt);
    (void)hipFree(ctx->d_as_off);
    (void)hipFree(ctx->d_as_steps);
    (void)hipFree(ctx->d_scan_tmp);
    (void)hipFree(ctx->d_pairf);
    (void)hipFree(ctx->d_pairg);
    (void)hipFree(ctx->d_mis);
    (void)hipFree(ctx->d_marks);
    (void)hipFree(ctx->d_as_bad);
    (void)hipFree(ctx->d_labels);
    (void)hipFree(ctx->d_walk);
    ctx->d_as_cnt = ctx->d_as_off = ctx->d_as_steps = ctx->d_pairf = ctx->d_pairg = ctx->d_marks = nullptr;
    ctx->d_scan_tmp = nullptr;
    ctx->d_mis = nullptr;
    ctx->d_as_bad = nullptr;
    ctx->d_labels = ctx->d_walk = nullptr;
    ctx->as_cnt_cap = ctx->as_off_cap = ctx->as_steps_cap = ctx->scan_tmp_cap = 0;
    ctx->pairf_cap = ctx->pairg_cap = ctx->mis_cap = ctx->marks_cap = ctx->as_bad_cap = 0;
    ctx->labels_cap = ctx->walk_cap = 0;
    (void)hipFree(ctx->d_wall_scr);
    (void)hipFree(ctx->d_wall_ovf);
    (void)hipFree(ctx->d_wall_open);
    (void)hipFree(ctx->d_wall_queue);
    ctx->d_wall_scr = ctx->d_wall_ovf = ctx->d_wall_open = ctx->d_wall_queue = nullptr;
    ctx->wall_scr_cap = ctx->wall_ovf_cap = ctx->wall_open_cap = ctx->wall_queue_cap = 0;
}

void free_fc(dmtz_ctx* ctx) {
    (void)hipFree(ctx->d_fc);
    (void)hipFree(ctx->d_path);
    ctx->d_fc = nullptr;
    ctx->d_path = nullptr;
    ctx->fc_cap = 0;
}

#define CK(x)                                                                         \
    do {                                                                              \
        hipError_t e_ = (x);                                                          \
        if (e_ != hipSuccess) {                                                       \
            ctx->err = std::string(#x) + " failed: " + hipGetErrorString(e_);         \
            return DMTZ_E_HIP;                                                        \
        }                                                                             \
    } while (0)

int ensure(dmtz_ctx* ctx, i64 N, size_t elem, bool want_fields) {
    if (N > ctx->cap_n) {
        free_bufs(ctx);
        const size_t n = (size_t)N;
        CK(hipMalloc(&ctx->d_counter, n));
        CK(hipMalloc(&ctx->d_stamp, sizeof(uint32_t) * n));
        CK(hipMalloc(&ctx->d_dstamp, sizeof(uint32_t) * n));
        CK(hipMemsetAsync(ctx->d_stamp, 0, sizeof(uint32_t) * n, ctx->stream));
        CK(hipMemsetAsync(ctx->d_dstamp, 0, sizeof(uint32_t) * n, ctx->stream));
        CK(hipMalloc(&ctx->d_targets, sizeof(uint32_t) * n));
        CK(hipMalloc(&ctx->d_changed, sizeof(uint32_t) * n));
        CK(hipMalloc(&ctx->d_dirty, sizeof(uint32_t) * n));
        CK(hipMalloc(&ctx->d_code_f, sizeof(StarCode) * n));
        CK(hipMalloc(&ctx->d_code_g, sizeof(StarCode) * n));
        for (MaskArray* m : {&ctx->d_critf, &ctx->d_mm}) {
            CK(hipMalloc(&m->lo, sizeof(uint64_t) * n));
            CK(hipMalloc(&m->hi, sizeof(uint32_t) * n));
        }
        CK(hipMalloc(&ctx->d_tile_nz, sizeof(uint32_t) * (n / EMIT_TILE + 2)));
        ctx->cap_n = N;
        ctx->epoch = 0;
    }
    if (want_fields && ctx->field_bytes < (size_t)N * elem) {
        (void)hipFree(ctx->d_f);
        (void)hipFree(ctx->d_g);
        ctx->d_f = ctx->d_g = nullptr;
        CK(hipMalloc(&ctx->d_f, (size_t)N * elem));
        CK(hipMalloc(&ctx->d_g, (size_t)N * elem));
        ctx->field_bytes = (size_t)N * elem;
    }
    return 0;
}

// Record lists grow on demand: detection is recomputed from f and g, so an overflowing launch is
// simply repeated after the resize.
int grow_rec(dmtz_ctx* ctx, ull need) {
    if (need <= ctx->rec_cap) return 0;
    free_rec(ctx);
    ull cap = need + need / 4 + 4096;
    CK(hipMalloc(&ctx->d_rec, sizeof(uint64_t) * 4 * cap));
    ctx->rec_cap = cap;
    return 0;
}

int grow_fc(dmtz_ctx* ctx, ull need) {
    if (need <= ctx->fc_cap) return 0;
    free_fc(ctx);
    ull cap = need + need / 4 + 4096;
    CK(hipMalloc(&ctx->d_fc, sizeof(uint64_t) * 4 * cap));
    CK(hipMalloc(&ctx->d_path, sizeof(int64_t) * 6 * cap));
    ctx->fc_cap = cap;
    return 0;
}

// Grow a device buffer of P to at least need elements (by x1.25 + 4096, or to need exactly).
template <class P>
int grow_buf(dmtz_ctx* ctx, P*& p, size_t& cap, size_t need, bool exact = false) {
    if (need <= cap) return 0;
    (void)hipFree(p);
    p = nullptr;
    cap = 0;
    const size_t n = exact ? need : need + need / 4 + 4096;
    CK(hipMalloc(&p, sizeof(P) * n));
    cap = n;
    return 0;
}

int check_dims(dmtz_ctx* ctx, i64 nx, i64 ny, i64 nz) {
    if (!ctx) return DMTZ_E_ARG;
    if (nx < 3 || ny < 2 || nz < 2) {
        ctx->err = "grid must have nx >= 3, ny >= 2, nz >= 2";
        return DMTZ_E_ARG;
    }
    if (nx * ny * nz >= ((i64)1 << 31)) {
        ctx->err = "grid has 2^31 or more vertices";
        return DMTZ_E_ARG;
    }
    return 0;
}

Lists4 rec_lists(dmtz_ctx* ctx) {
    Lists4 L;
    for (int k = 0; k < 4; k++) L.l[k] = ctx->d_rec + (size_t)k * ctx->rec_cap;
    L.cap = ctx->rec_cap;
    return L;
}
Lists4 fcrit_lists(dmtz_ctx* ctx) {
    Lists4 L;
    for (int k = 0; k < 4; k++) L.l[k] = ctx->d_fc + (size_t)k * ctx->fc_cap;
    L.cap = ctx->fc_cap;
    return L;
}

ull max4(const ull* x) {
    ull m = x[0];
    for (int k = 1; k < 4; k++) m = x[k] > m ? x[k] : m;
    return m;
}

int sync_ctr(dmtz_ctx* ctx) {
    k_read_ctrs<<<1, 64, 0, ctx->stream>>>(ctx->d_ctr, ctx->h_ctr);
    CK(hipGetLastError());
    CK(hipStreamSynchronize(ctx->stream));
    return 0;
}

int overflow_check(dmtz_ctx* ctx) {
    for (int k = 0; k < 4; k++)
        if (ctx->h_ctr[K_MIN + k] > ctx->rec_cap || ctx->h_ctr[K_FC0 + k] > ctx->fc_cap) {
            ctx->err = "mismatch list capacity exceeded";
            return DMTZ_E_CAPACITY;
        }
    if (ctx->h_ctr[K_DS] > ctx->fc_cap || ctx->h_ctr[K_AS] > ctx->fc_cap || ctx->h_ctr[K_DSW] > ctx->fc_cap) {
        ctx->err = "separatrix list capacity exceeded";
        return DMTZ_E_CAPACITY;
    }
    if (ctx->h_ctr[K_TGT] > (ull)ctx->cap_n) {
        ctx->err = "edit set capacity exceeded";
        return DMTZ_E_CAPACITY;
    }
    return 0;
}

using Clock = std::chrono::steady_clock;
double secs(Clock::time_point a, Clock::time_point b) { return std::chrono::duration<double>(b - a).count(); }

template <class T>
struct Driver {
    dmtz_ctx* ctx;
    const T* f;
    T* g;
    Dims d;
    Counts c;
    double eps, range;
    dmtz_flags fl;

    CodeArray cf() const { return CodeArray{ctx->d_code_f, c.N}; }
    CodeArray cg() const { return CodeArray{ctx->d_code_g, c.N}; }

    // Detection of the four critical-cell mismatch kinds into the record lists.
    int detect() {
        if (ctx->rec_cap == 0) {
            int rc0 = grow_rec(ctx, (ull)(c.N / 4));
            if (rc0) return rc0;
        }
        for (;;) {
            int rc = detect_once();
            if (rc) return rc;
            ull m = max4(ctx->h_ctr + K_MIN);
            if (m <= ctx->rec_cap) break;
            rc = grow_rec(ctx, m);
            if (rc) return rc;
        }
        return overflow_check(ctx);
    }

    bool det_clear = false;  // the detection counters were zeroed with the epoch's (begin_edits(true))

    int detect_once() {
        if (!det_clear) {
            k_zero_ctrs<<<1, 64, 0, ctx->stream>>>(ctx->d_ctr, DETECT_CTRS);
            CK(hipGetLastError());
        }
        det_clear = false;
        const ull ntiles = (ull)((c.N + EMIT_TILE - 1) / EMIT_TILE);
        // the events take the kernel's own time stamps: recorded around it they are two packets more
        hipExtLaunchKernelGGL(k_detect, dim3((unsigned)(ntiles < DETECT_BLOCKS ? ntiles : DETECT_BLOCKS)), dim3(BLOCK),
                              0, ctx->stream, ctx->ev0, ctx->ev1, 0, ctx->d_mm, c.N, ctx->d_tile_nz, rec_lists(ctx),
                              ctx->d_ctr + K_MIN, ctx->d_ctr + K_DTILES);
        CK(hipGetLastError());
        int rc = sync_ctr(ctx);
        if (rc) return rc;
        float ms = 0;
        CK(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        // bytes the kernel must move: the tile counts, the masks of the tiles with a mismatch,
        // and one 8-byte record written per mismatch emitted
        ull m = ctx->h_ctr[0] + ctx->h_ctr[1] + ctx->h_ctr[2] + ctx->h_ctr[3];
        ctx->det_launches += 1;
        ctx->det_ms += ms;
        ctx->det_bytes += 4.0 * (double)ntiles + (double)ctx->h_ctr[K_DTILES] * (double)EMIT_TILE * MASK_BYTES +
                          8.0 * (double)m;
        ctx->det_voxels += (double)c.N;
        return 0;
    }

    TargetSink sink(bool mark = false) {
        TargetSink s;
        s.stamp = ctx->d_stamp;
        s.epoch = ctx->epoch;
        s.list = mark ? nullptr : ctx->d_targets;
        s.ctr = ctx->d_ctr + K_TGT;
        s.cap = (ull)ctx->cap_n;
        return s;
    }

    uint32_t zone_from = 0;  // first epoch of the unchanged sweeps since the last change (0: none)

    int begin_edits(bool for_apply = false) {
        ctx->epoch++;
        if (ctx->epoch == 0) {  // stamp wrap (after 2^32 edit sets): clear and restart; the finisher
                                // zone then keeps only the edit sets from here on
            CK(hipMemsetAsync(ctx->d_stamp, 0, sizeof(uint32_t) * (size_t)c.N, ctx->stream));
            CK(hipMemsetAsync(ctx->d_dstamp, 0, sizeof(uint32_t) * (size_t)c.N, ctx->stream));
            ctx->epoch = 1;
            if (zone_from) zone_from = 1;
        }
        // the edit set; with for_apply also the counters of its apply (changed and dirty lists,
        // moved edits) and of the detection after it, whose last values the host has read before this
        // epoch begins (the finisher keeps its changed list across its epochs, so it zeroes those itself)
        k_zero_ctrs<<<1, 64, 0, ctx->stream>>>(
            ctx->d_ctr, ctr_bit(K_TGT) |
                            (for_apply ? ctr_bit(K_CHG) | ctr_bit(K_DIRTY) | ctr_bit(K_MOVED) | DETECT_CTRS : 0u));
        if (for_apply) det_clear = true;
        CK(hipGetLastError());
        return 0;
    }

    // Repair phase of one critical-point sweep (main_3d.cu:6801-6833) + apply (:6837). The kinds are
    // repaired by one launch (the edits form a set: their order does not matter).

    // From N / lim.target_dense records on the edit set is marked and applied by a pass over all stamps
    // instead of listed. Listing costs a returning atomic per target (about 0.4 ns of the whole chip's
    // time each: 512^3 fBm's first list of 65 M 2-saddles 27.5 -> 13.2 ms with marks), the pass reads
    // 4 N bytes (0.3 ms at 512^3 when it edits little).
    bool mark_targets(ull nrec) const { return nrec * ctx->lim.target_dense >= (ull)c.N; }

    int fix_cp(const ull counts[4]) {
        int rc = begin_edits(true);
        if (rc) return rc;
        ull nrec = 0;
        for (int ty = 0; ty < 4; ty++)
            if (rule_active(counts, ty)) nrec += counts[ty];
        rc = repair_records(counts, mark_targets(nrec));
        if (rc) return rc;
        return apply(nrec, mark_targets(nrec));
    }

    bool rule_active(const ull counts[4], int ty) const {
        return counts[ty] != 0 && !((ty == 1 || ty == 2) && fl.preserve_saddles != 1);
    }

    // The repair rules over the current mismatch lists (counts[ty] records of type ty) into the
    // edit set of the current epoch, listed or marked.
    int repair_records(const ull counts[4], bool mark) {
        const Lists4 L = rec_lists(ctx);
        const FixArgs<T> args{f, cf(), g, cg(), d, c, ctx->d_counter, eps, range, fl.edit_type};
        const int order[4] = {2, 0, 1, 3};
        FixLists q{};
        for (int k = 0; k < 4; k++) {
            const int ty = order[k];
            const ull n = rule_active(counts, ty) ? counts[ty] : 0;
            if ((ull)q.first[k] + nblocks(n) >= FIX_BLOCKS) {  // more threads than a launch takes: the lists so far
                int rc = launch_fix(q, q.first[k], args, mark);
                if (rc) return rc;
                q = FixLists{};
            }
            q.recs[k] = L.l[ty];
            q.n[k] = n;
            q.first[k + 1] = q.first[k] + nblocks(n);
        }
        return launch_fix(q, q.first[4], args, mark);
    }
    static constexpr ull FIX_BLOCKS = ((ull)1 << 32) / BLOCK;
    int launch_fix(const FixLists& q, unsigned blocks, const FixArgs<T>& args, bool mark) {
        if (blocks == 0) return 0;
        FixLists all = q;
        for (int k = 1; k < 5; k++)
            if (all.first[k] < all.first[k - 1]) all.first[k] = all.first[k - 1];
        k_fix_cp<T><<<blocks, BLOCK, 0, ctx->stream>>>(all, args, sink(mark));
        CK(hipGetLastError());
        return 0;
    }

    // applyDeltaBuffer1 (main_3d.cu:1122-1164) over the edit set, then re-evaluation of the g star
    // codes of the closed stars of the vertices whose value changed (the g gradient of
    // main_3d.cu:6864-6874 restricted to where it can change). Nothing here waits for the
    // device: the edit set's size stays on the device, nrec (the records repaired) sizes the
    // launches, and the count of edits that changed a value or a counter (K_MOVED) is read with
    // the next detection's counters. Each vertex enters the edit set at most once per epoch, so
    // the set never exceeds the N entries of its buffer.
    int apply(ull nrec, bool marked) {  // its counters start at zero with the epoch (begin_edits(true))
        if (!nrec) return 0;            // no record, no edit
        const ull est = nrec < (ull)c.N ? nrec : (ull)c.N;
        if (marked) {
            k_apply_marked<T><<<stride_blocks(((ull)c.N + APPLY_V - 1) / APPLY_V), BLOCK, 0, ctx->stream>>>(
                ctx->d_stamp, ctx->epoch, c.N, f, g, ctx->d_counter, eps, range, fl.preserve_type, fl.edit_type,
                ctx->d_changed, ctx->d_ctr + K_CHG, ctx->d_ctr + K_MOVED, ctx->d_ctr + K_TGT);
            CK(hipGetLastError());
            return refresh(est);
        }
        k_apply<T><<<stride_blocks(est), BLOCK, 0, ctx->stream>>>(
            ctx->d_targets, ctx->d_ctr + K_TGT, (ull)ctx->cap_n, f, g, ctx->d_counter, eps, range, fl.preserve_type,
            fl.edit_type, ctx->d_changed, ctx->d_ctr + K_CHG, ctx->d_ctr + K_MOVED);
        CK(hipGetLastError());
        return refresh(est);
    }

    // Re-evaluate the g star codes of the closed stars of the vertices in the changed list (the g
    // gradient of main_3d.cu:6864-6874 restricted to where it can change). est, the host's
    // estimate of the list's length, sizes the launches; when it is large the exact length is
    // read back to choose between re-evaluating every star and the closed stars of the list
    // (both give the same codes).
    int refresh(ull est) {
        if (!est) return 0;
        // Dense from N / 64 changed vertices on where the pass runs over bit planes (512^3: 4.6 ms,
        // where lists of a quarter of the stars took 5 to 8), from N / 16 with a thread per vertex.
        const ull dense = c.N >= ctx->lim.plane_min ? 64 : 16;
        // Up to lim.code_small vertices (a wave per SIMD) the pass over all of them takes no longer than
        // the shortest list (32^3: 17 us both), and neither the list nor its length is needed: whole
        // corrections of 2 to 65 thousand vertices, both types, are 2 to 10 % faster than over lists (40^3
        // mixture 7.70 against 8.58 ms); at 110 thousand 2 % faster, at 176 thousand 7 % slower.
        if (c.N <= ctx->lim.code_small) {
            est = (ull)c.N;
        } else if (dense * est >= (ull)c.N) {  // many stars may change: decide on the exact count
            int rc = sync_ctr(ctx);
            if (rc) return rc;
            est = ctx->h_ctr[K_CHG];
            if (!est) return 0;
        }
        if (dense * est >= (ull)c.N) {  // most stars change: re-evaluate all of them
            int rc = g_codes();
            if (rc) return rc;
            as_full = true;
            ctx->dirty_total += (double)c.N;
            return 0;
        }
        if (DIRTY_DENSE * 15 * est >= (ull)c.N) {  // long list: plain stores, then one pass over the stamps
            k_dirty_mark<<<stride_blocks(15 * est), BLOCK, 0, ctx->stream>>>(ctx->d_changed, ctx->d_ctr + K_CHG, d,
                                                                            ctx->d_dstamp, ctx->epoch);
            CK(hipGetLastError());
            const ull per_block = (ull)BLOCK * 4 * DIRTY_QUADS;
            k_dirty_collect<<<(unsigned)(((ull)c.N + per_block - 1) / per_block), BLOCK, 0, ctx->stream>>>(
                ctx->d_dstamp, c.N, ctx->epoch, ctx->d_dirty, ctx->d_ctr + K_DIRTY);
        } else {
            k_dirty<<<stride_blocks(15 * est), BLOCK, 0, ctx->stream>>>(ctx->d_changed, ctx->d_ctr + K_CHG, d,
                                                                       ctx->d_dstamp, ctx->epoch, ctx->d_dirty,
                                                                       ctx->d_ctr + K_DIRTY);
        }
        CK(hipGetLastError());
        k_code_list_g<T><<<stride_blocks(15 * est), BLOCK, 0, ctx->stream>>>(
            g, d, cg(), ctx->d_critf, ctx->d_mm, ctx->d_dirty, ctx->d_ctr + K_DIRTY, ctx->d_ctr + K_STARS,
            as_ready ? ctx->d_marks : nullptr, ctx->d_tile_nz);
        CK(hipGetLastError());
        return 0;
    }

    // Finisher step (no counterpart in the reference). The zone is the vertices of the first
    // cnt[k] mismatch records and the vertices targeted since zone_from. With r = ctx->radius
    // below the longest grid side and a non-empty zone: snap every vertex within Chebyshev
    // distance r of the zone that is not frozen yet, freeze them all, and repair the ties the
    // float snap creates by one-ulp raises. Otherwise restore g = f on every vertex and freeze it.
    int finish_step(const i64* cnt) {
        const int r = (int)ctx->radius;
        int rc = begin_edits();  // fresh epoch for the cell vertices; resets the list counter
        if (rc) return rc;
        const uint32_t from = zone_from, to = ctx->epoch;
        CK(hipMemsetAsync(ctx->d_ctr + K_CHG, 0, sizeof(ull) * 3, ctx->stream));  // changed, dirty, finished
        const ull ncell = (ull)(cnt[0] + cnt[1] + cnt[2] + cnt[3]);
        if (ncell) {
            k_zone_cells<<<nblocks(ncell), BLOCK, 0, ctx->stream>>>(rec_lists(ctx), (ull)cnt[0], (ull)cnt[1],
                                                                     (ull)cnt[2], (ull)cnt[3], d, ctx->d_stamp, to,
                                                                     ctx->d_targets, ctx->d_ctr + K_TGT);
            CK(hipGetLastError());
        }
        k_zone<<<nblocks(c.N), BLOCK, 0, ctx->stream>>>(ctx->d_stamp, from, to, c.N, ctx->d_targets,
                                                         ctx->d_ctr + K_TGT);
        CK(hipGetLastError());
        rc = sync_ctr(ctx);
        if (rc) return rc;
        const ull nz = ctx->h_ctr[K_TGT];
        const i64 span = d.W > d.H ? (d.W > d.D ? d.W : d.D) : (d.H > d.D ? d.H : d.D);
        if (nz == 0 || r >= span) {
            k_freeze_all<T><<<nblocks(c.N), BLOCK, 0, ctx->stream>>>(f, g, ctx->d_counter, c.N);
            CK(hipGetLastError());
            rc = g_codes();
            if (rc) return rc;
            as_full = true;
            ctx->finished += c.N;
        } else {
            rc = begin_edits();  // fresh epoch: each vertex is claimed once
            if (rc) return rc;
            const ull side = 2 * (ull)r + 1, total = nz * side * side * side;
            const ull blocks = nblocks(total) < 65536 ? nblocks(total) : 65536;
            k_snap_boxes<T><<<blocks, BLOCK, 0, ctx->stream>>>(ctx->d_targets, nz, r, d, f, g, ctx->d_counter, eps,
                                                                ctx->d_stamp, ctx->epoch, ctx->d_changed,
                                                                ctx->d_ctr + K_CHG);
            CK(hipGetLastError());
            rc = sync_ctr(ctx);
            if (rc) return rc;
            const ull nb = ctx->h_ctr[K_CHG];
            // Jacobi rounds of the tie repair; every round raises a vertex above a lower-f
            // neighbour, so at most nb rounds can be needed
            for (ull round = 0;; round++) {
                if (round > nb) {
                    ctx->err = "finisher tie repair did not settle";
                    return DMTZ_E_WALK;
                }
                rc = begin_edits();
                if (rc) return rc;
                CK(hipMemsetAsync(ctx->d_ctr + K_FINISH, 0, sizeof(ull), ctx->stream));
                k_tie_mark<T><<<nblocks(nb), BLOCK, 0, ctx->stream>>>(ctx->d_changed, nb, d, f, g, ctx->d_stamp,
                                                                       ctx->epoch, ctx->d_ctr + K_FINISH);
                CK(hipGetLastError());
                rc = sync_ctr(ctx);
                if (rc) return rc;
                if (ctx->h_ctr[K_FINISH] == 0) break;
                k_tie_raise<T><<<nblocks(nb), BLOCK, 0, ctx->stream>>>(ctx->d_changed, nb, g, ctx->d_stamp,
                                                                        ctx->epoch);
                CK(hipGetLastError());
            }
            rc = refresh(nb);
            if (rc) return rc;
            ctx->finished += (int64_t)nb;
        }
        zone_from = 0;
        return 0;
    }

    // Star codes of f and the f-critical status of every vertex's local cells (the gradient of
    // f, main_3d.cu:6539-6564, done once per run).
    int f_codes() {
        // the owned critical cells go to the mismatch masks first, which the g codes overwrite next
        int rc = codes(f, cf(), ctx->d_mm);
        if (rc) return rc;
        k_critf_gather<<<nblocks(c.N), BLOCK, 0, ctx->stream>>>(ctx->d_mm, d, c.N, ctx->d_critf);
        CK(hipGetLastError());
        return 0;
    }

    // g star codes and mismatch masks of every vertex (the g gradient, main_3d.cu:6624-6638);
    // needs the f-critical masks.
    int g_codes() {
        if (c.N >= ctx->lim.plane_min) {
            k_code_planes<T><<<plane_blocks(), 64, 0, ctx->stream>>>(g, d, Step64(d), c.N, cg(), ctx->d_mm, ctx->d_critf,
                                                                     ctx->d_tile_nz);
            CK(hipGetLastError());
            return 0;
        }
        CK(hipMemsetAsync(ctx->d_tile_nz, 0, sizeof(uint32_t) * (size_t)((c.N + EMIT_TILE - 1) / EMIT_TILE),
                          ctx->stream));
        k_code_g<T><<<nblocks(c.N), BLOCK, 0, ctx->stream>>>(g, d, c, cg(), ctx->d_critf, ctx->d_mm,
                                                             ctx->d_tile_nz);
        CK(hipGetLastError());
        return 0;
    }

    // Grids of lim.plane_min vertices or more classify over bit planes: below, a wave per 2048 vertices
    // leaves most of the chip idle and its 50 to 60 us of work are the time of the pass, in both types,
    // against 0.125 us per thousand vertices with a thread per vertex (393 k vertices: 51 and 54 us, the same
    // over planes; 524 k: 65 and 71 against 50 and 60; 1.4 M: 165 against 57 and 68).
    unsigned plane_blocks() const { return (unsigned)((c.N + PLANE_TILE - 1) / PLANE_TILE); }

    // Star codes of every vertex of a field.
    int codes(const T* fld, CodeArray out, MaskArray own) {
        if (c.N >= ctx->lim.plane_min) {
            k_code_planes<T><<<plane_blocks(), 64, 0, ctx->stream>>>(fld, d, Step64(d), c.N, out, own, MaskArray{nullptr, nullptr}, nullptr);
            CK(hipGetLastError());
            return 0;
        }
        k_code<T><<<nblocks(c.N), BLOCK, 0, ctx->stream>>>(fld, d, c, out, own);
        CK(hipGetLastError());
        return 0;
    }

    PathList path_list(int which) {
        PathList p;
        ull cap = ctx->fc_cap;
        p.id = ctx->d_path + (size_t)(2 * which) * cap;
        p.rec = ctx->d_path + (size_t)(2 * which + 1) * cap;
        p.ctr = ctx->d_ctr + (which == 0 ? K_DS : (which == 1 ? K_AS : K_DSW));
        p.cap = cap;
        return p;
    }

    ull nfce = 0, nfcf = 0;
    // Connectivity-mode ascending checks from g's critical faces instead of f's (dmtz_paths on
    // fields whose critical cells differ; in the correction loop the two sets are equal).
    const uint64_t* as_gfaces = nullptr;
    ull n_gfaces = 0;

    // Critical cells of the types in type_mask into the f-critical lists (grown on demand), from the
    // star codes given or, with codes null, from f's owned critical cells, which lie in d_mm between
    // f_codes() and g_codes(). Types outside list_mask are counted but not listed.
    int fcrit(const CodeArray* codes, int type_mask, int list_mask = 15) {
        if (ctx->fc_cap == 0) {
            int rc0 = grow_fc(ctx, (ull)(c.N / 16));
            if (rc0) return rc0;
        }
        for (;;) {
            Lists4 FL = fcrit_lists(ctx);
            for (int k = 0; k < 4; k++)
                if (!((list_mask >> k) & 1)) FL.l[k] = nullptr;
            CK(hipMemsetAsync(ctx->d_ctr + K_FC0, 0, sizeof(ull) * 4, ctx->stream));
            k_fcrit<<<(unsigned)((c.N + EMIT_TILE - 1) / EMIT_TILE), BLOCK, 0, ctx->stream>>>(
                codes ? MaskArray{nullptr, nullptr} : ctx->d_mm, codes ? *codes : cf(), c, FL, ctx->d_ctr + K_FC0, type_mask);
            CK(hipGetLastError());
            int rc = sync_ctr(ctx);
            if (rc) return rc;
            ull m = max4(ctx->h_ctr + K_FC0);
            if (m <= ctx->fc_cap) break;
            rc = grow_fc(ctx, m);
            if (rc) return rc;
        }
        return 0;
    }

    // The start cells of the separatrix checks: f-critical faces, and edges (listed in connectivity
    // mode only: the geometry checks find them from the vertices). codes as for fcrit().
    int prepare_paths(const CodeArray* codes) {
        const bool conn = fl.preserve_geometry != 1;
        int rc = fcrit(codes, 2 | 4, conn ? 15 : 4);
        if (rc) return rc;
        Lists4 FL = fcrit_lists(ctx);
        nfce = ctx->h_ctr[K_FC0 + 1];
        nfcf = ctx->h_ctr[K_FC0 + 2];
        if (conn) {
            rc = pairs_of(f, cf(), ctx->d_pairf, ctx->pairf_cap, ctx->stream);
            if (rc) return rc;
        }
        if (conn && nfce + nfcf) {
            rc = grow_buf(ctx, ctx->d_labels, ctx->labels_cap, 2 * (nfce + nfcf));
            if (rc) return rc;
            k_labels<<<nblocks(2 * (nfce + nfcf)), BLOCK, 0, ctx->stream>>>(
                FL.l[1], nfce, FL.l[2], nfcf, ctx->d_pairf, d, c.N, ctx->d_labels, ctx->d_labels + 2 * nfce,
                ctx->d_ctr + K_WALK);
            CK(hipGetLastError());
        }
        return 0;
    }

    int pairs_of(const T* fld, CodeArray codes, uint32_t*& out, size_t& cap, hipStream_t st) {
        int rc = grow_buf(ctx, out, cap, (size_t)c.N);
        if (rc) return rc;
        k_pairs<T><<<nblocks(c.N), BLOCK, 0, st>>>(fld, codes, d, c.N, out);
        CK(hipGetLastError());
        return 0;
    }

    // Separatrix detection (main_3d.cu:6955-6970): fills the ds / as lists.
    int detect_paths() {
        CK(hipMemsetAsync(ctx->d_ctr + K_DS, 0, sizeof(ull) * 2, ctx->stream));
        int rc = fl.preserve_geometry == 1 ? check_geometry() : check_connectivity();
        if (rc) return rc;
        if (fl.preserve_connectors == 1) {
            rc = walls();
            if (rc) return rc;
        }
        rc = sync_ctr(ctx);
        if (rc) return rc;
        return overflow_check(ctx);
    }

    // Walks both branches of the n start faces and combines their results into the as list.
    int as_branches(const uint64_t* faces, ull n, const int64_t* lab, int lab_from_f) {
        if (!n) return 0;
        int rc = grow_buf(ctx, ctx->d_walk, ctx->walk_cap, 4 * n);
        if (rc) return rc;
        k_as_branch<<<nblocks(2 * n), BLOCK, 0, ctx->stream>>>(faces, n, lab, lab_from_f, ctx->d_critf.lo, ctx->d_pairf,
                                                               ctx->d_pairg, d, c.N, ctx->d_walk, ctx->d_ctr + K_WALK);
        CK(hipGetLastError());
        k_as_combine<<<nblocks(n), BLOCK, 0, ctx->stream>>>(ctx->d_walk, n, path_list(1));
        CK(hipGetLastError());
        return 0;
    }

    int check_connectivity() {
        int rc = pairs_of(g, cg(), ctx->d_pairg, ctx->pairg_cap, ctx->stream);
        if (rc) return rc;
        Lists4 FL = fcrit_lists(ctx);
        rc = as_gfaces ? as_branches(as_gfaces, n_gfaces, nullptr, 1)
                       : as_branches(FL.l[2], nfcf, ctx->d_labels + 2 * nfce, 0);
        if (rc || !nfce) return rc;
        rc = grow_buf(ctx, ctx->d_walk, ctx->walk_cap, 4 * nfce);
        if (rc) return rc;
        k_ds_branch<<<nblocks(2 * nfce), BLOCK, 0, ctx->stream>>>(FL.l[1], nfce, ctx->d_pairf, ctx->d_pairg, d, c.N,
                                                                  ctx->d_walk, ctx->d_ctr + K_WALK);
        CK(hipGetLastError());
        k_ds_combine<<<nblocks(nfce), BLOCK, 0, ctx->stream>>>(FL.l[1], nfce, ctx->d_walk, ctx->d_labels, d, c,
                                                               path_list(0));
        CK(hipGetLastError());
        return 0;
    }

    int check_geometry() {
        int rc = as_stage ? as_join() : (as_ready ? 0 : as_prepare());
        if (rc) return rc;
        const size_t words = (size_t)(c.N + 31) / 32;
        if (as_full || !as_listed) {
            if (!as_listed) {
                rc = grow_buf(ctx, ctx->d_pairg, ctx->pairg_cap, (size_t)c.N);
                if (rc) return rc;
            }
            CK(hipMemsetAsync(ctx->d_marks, 0, sizeof(uint32_t) * words, ctx->stream));
            k_mism_full<T><<<nblocks(c.N), BLOCK, 0, ctx->stream>>>(g, cg(), ctx->d_pairf, d, c.N, ctx->d_mis,
                                                                     as_listed ? nullptr : ctx->d_pairg);
        } else {
            k_mism_marked<T><<<nblocks(words), BLOCK, 0, ctx->stream>>>(g, cg(), ctx->d_pairf, d, c.N,
                                                                         ctx->d_marks, ctx->d_mis);
        }
        CK(hipGetLastError());
        as_full = false;
        if (nfcf && as_listed) {
            if (as_total) {
                k_as_bad<<<nblocks((as_total + AS_BAD_WORDS - 1) / AS_BAD_WORDS), BLOCK, 0, ctx->stream>>>(
                    as_total, ctx->d_as_steps, ctx->d_mis, ctx->d_as_bad);
                CK(hipGetLastError());
            }
            k_as_list<<<nblocks((nfcf + AS_FACES - 1) / AS_FACES), BLOCK, 0, ctx->stream>>>(
                nfcf, ctx->d_as_off, ctx->d_as_bad, ctx->d_as_steps, d, list_ids ? 1 : 0, path_list(1));
            CK(hipGetLastError());
        } else {
            rc = as_branches(fcrit_lists(ctx).l[2], nfcf, nullptr, 0);
            if (rc) return rc;
        }
        if (nfce) {
            k_ds_list<<<nblocks((c.N + DS_V - 1) / DS_V), BLOCK, 0, ctx->stream>>>(ctx->d_mis, ctx->d_critf.lo, d, c, c.N,
                                                                                   path_list(0));
            CK(hipGetLastError());
        }
        return 0;
    }

    size_t wall_words() const { return ((size_t)c.N + 1) / 2; }
    bool wall_search = false;  // no memory for the open faces: the run searches its walls

    // Room for the open faces' bits and a queue of so many. Most checks open a small part of the 12 faces
    // per vertex, so the queue begins with one per vertex (both together 6 bytes a vertex, 0.8 GB at 512^3; a
    // queue of all faces 6.4 GB) and grows when a check opens more.
    bool wall_room(ull faces) {
        if (wall_search || 12 * c.N >= ((i64)1 << 32)) return false;
        if (!grow_buf(ctx, ctx->d_wall_open, ctx->wall_open_cap, wall_words(), true) &&
            !grow_buf(ctx, ctx->d_wall_queue, ctx->wall_queue_cap, (size_t)faces, true))
            return true;
        (void)hipGetLastError();
        ctx->err.clear();  // not an error of the call: the search needs neither
        wall_search = true;
        return false;
    }
    // The walls by chains; left receives the number of faces to search, listed in the second half of
    // d_wall_ovf. done = false: there was no room, and all faces are to be searched.
    int wall_chains(bool& done, ull& left) {
        const size_t words = wall_words();
        done = wall_room(ctx->lim.wall_queue ? ctx->lim.wall_queue : (ull)c.N);
        while (done) {
            const ull cap = (ull)ctx->wall_queue_cap;
            const WallArgs<T> a{f, g, cf(), cg(), d, c, ctx->d_wall_open, ctx->d_wall_queue, cap, ctx->d_ctr + K_WOPEN};
            CK(hipMemsetAsync(ctx->d_wall_open, 0, sizeof(uint32_t) * words, ctx->stream));
            k_zero_ctrs<<<1, 64, 0, ctx->stream>>>(ctx->d_ctr, ctr_bit(K_WOPEN) | ctr_bit(K_WOVF) | ctr_bit(K_DSW));
            CK(hipGetLastError());
            k_wall_seeds<T><<<nblocks(c.N), BLOCK, 0, ctx->stream>>>(a);
            CK(hipGetLastError());
            ull from = 0, to = 0;
            for (;;) {
                int rc = sync_ctr(ctx);
                if (rc) return rc;
                to = ctx->h_ctr[K_WOPEN];
                if (to > cap || to - from < ctx->lim.wall_level || to == from) break;
                k_wall_level<T><<<nblocks(to - from), BLOCK, 0, ctx->stream>>>(a, from, to);
                CK(hipGetLastError());
                from = to;
            }
            left = 0;
            if (to == 0) return 0;
            if (to <= cap) {
                k_wall_levels<T><<<1, WALL_BLOCK, 0, ctx->stream>>>(a, from, to);
                CK(hipGetLastError());
                k_wall_chain<T><<<nblocks(nfcf), BLOCK, 0, ctx->stream>>>(
                    a, fcrit_lists(ctx).l[2], nfcf, path_list(2), ctx->d_wall_ovf + nfcf, ctx->d_ctr + K_WOVF);
                CK(hipGetLastError());
                int rc = sync_ctr(ctx);
                if (rc) return rc;
                to = ctx->h_ctr[K_WOPEN];
                left = ctx->h_ctr[K_WOVF];
                if (to <= cap) return 0;
            }
            // more faces than the queue holds: again, with room for at least those counted so far
            const ull want = to > 4 * cap ? to : 4 * cap;
            done = wall_room(want < (ull)c.F ? want : (ull)c.F);
        }
        return 0;
    }

    // 2-saddle walls (preserve_connectors, main_3d.cu:5064-5133) from every f-critical face into the
    // wall list: the open faces (levels backwards from the mismatched edges), then a chain per open
    // f-critical face. The faces left over (all of them, where the device has no memory for the queue)
    // are searched in tiers of visited-set size: with 256 slots, the walks that outgrow them with 8192,
    // then with 2^18; a search of more than 2^17 faces is a capacity error. Launches are chunked to keep
    // the per-thread sets near 1 GiB.
    int walls() {
        CK(hipMemsetAsync(ctx->d_ctr + K_DSW, 0, sizeof(ull), ctx->stream));
        if (!nfcf) return 0;
        if (c.F >= (i64)0xFFFFFFFFll) {
            ctx->err = "2-saddle walls need fewer than 2^32 - 1 faces";
            return DMTZ_E_UNSUPPORTED;
        }
        static const uint32_t tiers[3] = {256u, 8192u, 1u << 18};
        const size_t budget = (size_t)1 << 28;  // uint32 entries of per-thread sets in flight
        int rc = grow_buf(ctx, ctx->d_wall_ovf, ctx->wall_ovf_cap, 2 * (size_t)nfcf);
        if (rc) return rc;
        Lists4 FL = fcrit_lists(ctx);
        const uint32_t* sel = nullptr;
        ull n = nfcf;
        bool done = false;
        ull left = 0;
        rc = wall_chains(done, left);
        if (rc) return rc;
        if (done) {
            sel = ctx->d_wall_ovf + nfcf;
            n = left;
        } else {  // a check that ran out of room may have listed some
            CK(hipMemsetAsync(ctx->d_ctr + K_DSW, 0, sizeof(ull), ctx->stream));
        }
        for (int tier = 0; tier < 3 && n > 0; tier++) {
            const uint32_t slots = tiers[tier];
            const size_t per = 2 * (size_t)slots + 2;
            const ull chunk = (ull)(budget / per) < n ? (ull)(budget / per) : n;
            rc = grow_buf(ctx, ctx->d_wall_scr, ctx->wall_scr_cap, chunk * per);
            if (rc) return rc;
            uint32_t* ovf = ctx->d_wall_ovf + (tier % 2 == 0 ? 0 : nfcf);
            CK(hipMemsetAsync(ctx->d_ctr + K_WOVF, 0, sizeof(ull), ctx->stream));
            for (ull first = 0; first < n; first += chunk) {
                const ull last = first + chunk < n ? first + chunk : n;
                k_ds_wall<T><<<nblocks(last - first), BLOCK, 0, ctx->stream>>>(
                    FL.l[2], sel, first, last, f, cf(), g, cg(), d, c, ctx->d_wall_scr, slots,
                    path_list(2), ovf, ctx->d_ctr + K_WOVF);
                CK(hipGetLastError());
            }
            rc = sync_ctr(ctx);
            if (rc) return rc;
            n = ctx->h_ctr[K_WOVF];
            sel = ovf;
        }
        if (n > 0) {
            ctx->err = "a 2-saddle wall exceeds 2^17 faces";
            return DMTZ_E_CAPACITY;
        }
        return 0;
    }

    // Geometry checks: the pair words of f and the listed ascending paths (one word per step), made
    // once per run. Paths are listed when step words and face ids fit 32 bits and there are fewer than
    // 2^32 steps; otherwise every check walks them.
    bool as_ready = false, as_full = true, as_listed = false;
    bool list_ids = false;  // the caller reads the start cells of the ascending list
    ull as_total = 0;  // steps of the listed paths

    bool as_listable() const { return fl.preserve_geometry == 1 && c.F < ((i64)1 << 32) && 12 * c.N < ((i64)1 << 32); }

    int as_prepare() {
        int rc = as_count(ctx->stream);
        if (rc) return rc;
        CK(hipStreamSynchronize(ctx->stream));
        rc = as_fill(ctx->stream);
        if (rc) return rc;
        return as_begin();
    }

    int as_begin() {  // the paths are in place: the checks start with a full one
        as_ready = true;
        as_full = true;
        const char* lg = std::getenv("DMTZ_LOG");
        if (lg && lg[0] == '1')
            std::fprintf(stderr, "dmtz ascending paths: %llu faces, %llu steps, %s\n", (unsigned long long)nfcf,
                         (unsigned long long)as_total, as_listed ? "listed" : "walked");
        return 0;
    }

    // The precompute depends on f alone, so single-field runs start it on a stream of its own
    // right after the first detection and let it overlap the critical-point sweeps; the first
    // separatrix check waits for it (as_join). Started after the first repair phase instead, it
    // slows the dense re-classification that follows (that kernel needs the wave slots the walk
    // holds) more than it spares the rules. as_stage: 0 none in flight, 1 counting walk enqueued,
    // 2 fill enqueued.
    int as_stage = 0;

    int as_start_async() {
        if (!ctx->side_stream || !as_listable() || as_ready || !nfcf) return 0;
        if (!ctx->as_stream) {
            CK(hipStreamCreateWithFlags(&ctx->as_stream, hipStreamNonBlocking));
            CK(hipEventCreateWithFlags(&ctx->as_ev_fork, hipEventDisableTiming));
            CK(hipEventCreateWithFlags(&ctx->as_ev_count, hipEventDisableTiming));
            CK(hipEventCreateWithFlags(&ctx->as_ev_done, hipEventDisableTiming));
        }
        CK(hipEventRecord(ctx->as_ev_fork, ctx->stream));
        CK(hipStreamWaitEvent(ctx->as_stream, ctx->as_ev_fork, 0));
        int rc = as_count(ctx->as_stream);
        if (rc) return rc;
        CK(hipEventRecord(ctx->as_ev_count, ctx->as_stream));
        as_stage = 1;
        return 0;
    }

    // Enqueue the fill once the counting walk is done (wait = false: only if it already is).
    int as_advance(bool wait) {
        if (as_stage != 1) return 0;
        if (!wait) {
            const hipError_t q = hipEventQuery(ctx->as_ev_count);
            if (q == hipErrorNotReady) return 0;
            CK(q);
        } else {
            CK(hipEventSynchronize(ctx->as_ev_count));
        }
        int rc = as_fill(ctx->as_stream);
        if (rc) return rc;
        CK(hipEventRecord(ctx->as_ev_done, ctx->as_stream));
        as_stage = 2;
        return 0;
    }

    // The context's stream waits for the precompute; the checks can then use it.
    int as_join() {
        int rc = as_advance(true);
        if (rc) return rc;
        CK(hipStreamWaitEvent(ctx->stream, ctx->as_ev_done, 0));
        as_stage = 0;
        return as_begin();
    }

    // First half, on stream st: f's pair words, the counting walk and the scan of its counts; the
    // number of steps lands in *h_as_total when st gets there.
    int as_count(hipStream_t st) {
        const size_t words = (size_t)(c.N + 31) / 32;
        int rc = pairs_of(f, cf(), ctx->d_pairf, ctx->pairf_cap, st);
        if (rc) return rc;
        rc = grow_buf(ctx, ctx->d_mis, ctx->mis_cap, (size_t)c.N + DS_V);
        if (rc) return rc;
        rc = grow_buf(ctx, ctx->d_marks, ctx->marks_cap, words);
        if (rc) return rc;
        *ctx->h_as_total = 0;
        as_listed = as_listable();
        if (!as_listed || !nfcf) return 0;
        rc = grow_buf(ctx, ctx->d_as_cnt, ctx->as_cnt_cap, nfcf + 1);
        if (rc) return rc;
        rc = grow_buf(ctx, ctx->d_as_off, ctx->as_off_cap, nfcf + 1);
        if (rc) return rc;
        size_t tmp = 0;
        CK(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, ctx->d_as_cnt, ctx->d_as_off, (int)(nfcf + 1), st));
        uint8_t* tp = (uint8_t*)ctx->d_scan_tmp;
        rc = grow_buf(ctx, tp, ctx->scan_tmp_cap, tmp);
        ctx->d_scan_tmp = tp;
        if (rc) return rc;
        CK(hipMemsetAsync(ctx->d_as_cnt + nfcf, 0, sizeof(uint32_t), st));
        CK(hipMemsetAsync(ctx->d_ctr + K_ASNEXT, 0, sizeof(ull) * 2, st));
        k_as_walk<false><<<as_walk_blocks(st), BLOCK, 0, st>>>(fcrit_lists(ctx).l[2], nfcf, ctx->d_pairf, d, c.N,
                                                               ctx->d_as_cnt, nullptr, nullptr, ctx->d_ctr + K_ASNEXT,
                                                               ctx->d_ctr + K_ASTOTAL, ctx->d_ctr + K_WALK);
        CK(hipGetLastError());
        CK(hipcub::DeviceScan::ExclusiveSum(ctx->d_scan_tmp, tmp, ctx->d_as_cnt, ctx->d_as_off, (int)(nfcf + 1), st));
        CK(hipMemcpyAsync(ctx->h_as_total, ctx->d_ctr + K_ASTOTAL, sizeof(ull), hipMemcpyDeviceToHost, st));
        return 0;
    }

    // Second half, with the number of steps on the host.
    int as_fill(hipStream_t st) {
        as_total = *ctx->h_as_total;
        as_listed = as_listed && as_total < ctx->lim.path_steps;
        if (!as_listed || !nfcf || !as_total) return 0;
        int rc = grow_buf(ctx, ctx->d_as_steps, ctx->as_steps_cap, as_total);
        if (rc) return rc;
        rc = grow_buf(ctx, ctx->d_as_bad, ctx->as_bad_cap, (as_total + 63) / 64);
        if (rc) return rc;
        CK(hipMemsetAsync(ctx->d_ctr + K_ASNEXT, 0, sizeof(ull), st));
        k_as_walk<true><<<as_walk_blocks(st), BLOCK, 0, st>>>(fcrit_lists(ctx).l[2], nfcf, ctx->d_pairf, d, c.N, nullptr,
                                                              ctx->d_as_off, ctx->d_as_steps, ctx->d_ctr + K_ASNEXT,
                                                              nullptr, ctx->d_ctr + K_WALK);
        CK(hipGetLastError());
        return 0;
    }

    unsigned as_walk_blocks(hipStream_t st) const {
        const unsigned cap = st == ctx->stream ? AS_WS_BLOCKS : AS_WS_BLOCKS_SIDE, n = nblocks(nfcf);
        return n < cap ? n : cap;
    }

    int fix_paths(ull nds, ull nas, ull nw) {
        int rc = begin_edits(true);
        if (rc) return rc;
        if (fl.preserve_connectors != 1) nw = 0;
        const bool mark = mark_targets(nds + nas + nw);
        if (nds + nas + nw) {
            k_fix_paths<T><<<nblocks(nds + nas + nw), BLOCK, 0, ctx->stream>>>(
                path_list(1).rec, nas, path_list(0).rec, nds, path_list(2).rec, nw, f, cf(), g,
                cg(), d, c, ctx->d_counter, eps, range, fl.edit_type, sink(mark));
            CK(hipGetLastError());
        }
        return apply(nds + nas + nw, mark);
    }

    int filtration() {
        int rc = fcrit(nullptr, 15);
        if (rc) return rc;
        Lists4 FL = fcrit_lists(ctx);
        for (int ty = 0; ty < 4; ty++) {
            ull n = ctx->h_ctr[K_FC0 + ty];
            if (!n) continue;
            k_pin<T><<<nblocks(n), BLOCK, 0, ctx->stream>>>(FL.l[ty], n, f, g, d, c, eps);
            CK(hipGetLastError());
        }
        return 0;
    }

    // The loop of main_3d.cu:6521-7149, with an exit at a stall: a sweep is a function of
    // (g, counter, counts, sweep kind), so a sweep that changes no value or counter and whose
    // (counts, kind) repeats one seen since the last change starts a cycle the reference never
    // leaves. Without the finisher the run returns DMTZ_STALLED there; with it, finish_step() is
    // applied and the sweep's counts are re-evaluated.
    int run(dmtz_counts* out, int32_t* sweeps_out) {
        if (ctx->as_stream) CK(hipStreamSynchronize(ctx->as_stream));  // after a failed earlier run
        ctx->traj.clear();
        for (double& p : ctx->phase) p = 0;
        ctx->stalls = ctx->finished = ctx->radius = 0;
        zone_from = 0;
        auto t_start = Clock::now();
        int maxs = fl.max_sweeps > 0 ? fl.max_sweeps : 100000;
        CK(hipMemsetAsync(ctx->d_ctr, 0, sizeof(ull) * K_NCTR, ctx->stream));
        ctx->dirty_total = 0;
        auto t0 = Clock::now();
        int rc = f_codes();  // gradient of f, main_3d.cu:6539-6564
        if (rc) return rc;
        if (fl.filtration == 1) {
            rc = filtration();
            if (rc) return rc;
        }
        CK(hipMemsetAsync(ctx->d_counter, 1, (size_t)c.N, ctx->stream));  // init_counter :6782
        bool paths = fl.preserve_vpath == 1;
        if (paths) {
            rc = prepare_paths(nullptr);
            if (rc) return rc;
        }
        rc = g_codes();  // gradient of g, main_3d.cu:6624-6638
        if (rc) return rc;
        CK(hipStreamSynchronize(ctx->stream));
        auto t1 = Clock::now();
        ctx->phase[0] += secs(t0, t1);
        rc = detect();
        if (rc) return rc;
        ctx->phase[1] += secs(t1, Clock::now());
        i64 cnt[8] = {(i64)ctx->h_ctr[0], (i64)ctx->h_ctr[1], (i64)ctx->h_ctr[2], (i64)ctx->h_ctr[3], 1, 1, 1, 0};
        if (paths) {
            rc = as_start_async();
            if (rc) return rc;
        }
        i64 sweeps = 0;
        int status = 0;
        const char* lg = std::getenv("DMTZ_LOG");
        const bool log = lg && lg[0] == '1';
        auto record = [&]() {
            for (int k = 0; k < 8; k++) ctx->traj.push_back(cnt[k]);
            if (log)
                std::fprintf(stderr, "dmtz sweep %lld: %lld %lld %lld %lld | %lld %lld  (%.3f s, %lld edits, %.0f stars)\n",
                             (long long)sweeps, (long long)cnt[0], (long long)cnt[1], (long long)cnt[2],
                             (long long)cnt[3], (long long)cnt[4], (long long)cnt[5], secs(t_start, Clock::now()),
                             (long long)ctx->h_ctr[K_TGT], ctx->dirty_total + (double)ctx->h_ctr[K_STARS]);
        };
        // Re-evaluation after the apply of a critical-point sweep (main_3d.cu:6864-6921).
        auto eval_cp = [&]() -> int {
            auto tb = Clock::now();
            int r = detect();
            if (r) return r;
            ctx->phase[1] += secs(tb, Clock::now());
            cnt[0] = (i64)ctx->h_ctr[0];
            cnt[1] = fl.preserve_saddles == 1 ? (i64)ctx->h_ctr[1] : 0;
            cnt[2] = fl.preserve_saddles == 1 ? (i64)ctx->h_ctr[2] : 0;
            cnt[3] = (i64)ctx->h_ctr[3];
            return 0;
        };
        // Re-evaluation after the apply of a separatrix sweep (main_3d.cu:7069-7143).
        auto eval_path = [&]() -> int {
            auto tc = Clock::now();
            int r = detect();
            if (r) return r;
            auto td = Clock::now();
            ctx->phase[1] += secs(tc, td);
            cnt[0] = (i64)ctx->h_ctr[0];
            cnt[1] = (i64)ctx->h_ctr[1];
            cnt[2] = (i64)ctx->h_ctr[2];
            cnt[3] = (i64)ctx->h_ctr[3];
            cnt[4] = cnt[5] = cnt[6] = cnt[7] = 0;
            if (cnt[0] == 0 && cnt[1] == 0 && cnt[2] == 0 && cnt[3] == 0) {
                r = detect_paths();
                if (r) return r;
                cnt[4] = (i64)ctx->h_ctr[K_DS];
                cnt[5] = (i64)ctx->h_ctr[K_AS];
                cnt[6] = fl.preserve_connectors == 1 ? (i64)ctx->h_ctr[K_DSW] : 0;
                ctx->phase[2] += secs(td, Clock::now());
            }
            return 0;
        };
        std::vector<std::vector<i64>> seen;  // (counts, kind) since the last change
        // After the re-evaluation of a sweep of the given kind (0 critical points, 1 separatrices).
        // Sets stalled when the run stalls without the finisher.
        bool stalled = false;
        auto after_sweep = [&](int kind) -> int {
            std::vector<i64> key(cnt, cnt + 8);
            key.push_back(kind);
            if (ctx->h_ctr[K_MOVED] > 0) {  // edits of the sweep that changed a value or a counter
                seen.assign(1, key);
                zone_from = 0;
                return 0;
            }
            if (zone_from == 0) zone_from = ctx->epoch;  // this sweep's edit set opens the zone
            bool any = false;
            for (int k = 0; k < 8; k++) any = any || cnt[k] != 0;
            if (!any) return 0;
            for (const auto& sk : seen)
                if (sk == key) {
                    ctx->stalls++;
                    if (fl.finish != 1) {
                        stalled = true;
                        return 0;
                    }
                    ctx->radius = ctx->radius ? 2 * ctx->radius : 1;  // 1, 2, 4, ...
                    int r = finish_step(cnt);
                    if (r) return r;
                    r = kind == 0 ? eval_cp() : eval_path();
                    if (r) return r;
                    key.assign(cnt, cnt + 8);
                    key.push_back(kind);
                    seen.assign(1, key);
                    return 0;
                }
            seen.push_back(key);
            return 0;
        };
        while (cnt[5] > 0 || cnt[4] > 0 || cnt[6] > 0 || cnt[2] > 0 || cnt[3] > 0 || cnt[0] > 0 || cnt[1] > 0) {
            while (cnt[3] > 0 || cnt[2] > 0 || cnt[0] > 0 || cnt[1] > 0) {
                if (sweeps >= maxs) {
                    status = DMTZ_NOT_CONVERGED;
                    goto done;
                }
                sweeps++;
                auto ta = Clock::now();
                ull cc[4] = {(ull)cnt[0], (ull)cnt[1], (ull)cnt[2], (ull)cnt[3]};
                rc = fix_cp(cc);
                if (rc) return rc;
                ctx->phase[3] += secs(ta, Clock::now());
                rc = eval_cp();
                if (rc) return rc;
                rc = after_sweep(0);
                if (rc) return rc;
                record();
                if (stalled) {
                    status = DMTZ_STALLED;
                    goto done;
                }
                rc = as_advance(false);
                if (rc) return rc;
            }
            if (!paths) break;
            if (sweeps >= maxs) {
                status = DMTZ_NOT_CONVERGED;
                goto done;
            }
            sweeps++;
            {
                auto ta = Clock::now();
                rc = detect_paths();
                if (rc) return rc;
                auto tb = Clock::now();
                ctx->phase[2] += secs(ta, tb);
                ull nds = ctx->h_ctr[K_DS], nas = ctx->h_ctr[K_AS], nw = ctx->h_ctr[K_DSW];
                rc = fix_paths(nds, nas, nw);
                if (rc) return rc;
                ctx->phase[4] += secs(tb, Clock::now());
                rc = eval_path();
                if (rc) return rc;
                rc = after_sweep(1);
                if (rc) return rc;
                record();
                if (stalled) {
                    status = DMTZ_STALLED;
                    goto done;
                }
            }
        }
    done:
        if (!paths) cnt[4] = cnt[5] = cnt[6] = cnt[7] = 0;
        if (as_stage) {  // a precompute the run did not need: let it finish, it is not used
            CK(hipStreamSynchronize(ctx->as_stream));
            as_stage = 0;
        }
        CK(hipStreamSynchronize(ctx->stream));
        ctx->phase[5] = secs(t_start, Clock::now());
        if (out) {
            out->min = cnt[0];
            out->saddle1 = cnt[1];
            out->saddle2 = cnt[2];
            out->max = cnt[3];
            out->ds_vpath = cnt[4];
            out->as_vpath = cnt[5];
            out->ds_wall = cnt[6];
            out->as_wall = cnt[7];
        }
        if (sweeps_out) *sweeps_out = (int32_t)sweeps;
        CK(hipMemcpyAsync(ctx->h_ctr, ctx->d_ctr, sizeof(ull) * K_NCTR, hipMemcpyDeviceToHost, ctx->stream));
        CK(hipStreamSynchronize(ctx->stream));
        ctx->dirty_total += (double)ctx->h_ctr[K_STARS];
        if (ctx->h_ctr[K_WALK] > 0) {
            ctx->err = "a separatrix walk exceeded N steps (cyclic gradient path)";
            return DMTZ_E_WALK;
        }
        return status;
    }
};

template <class T>
int correct_dev(dmtz_ctx* ctx, const T* d_f, T* d_g, i64 nx, i64 ny, i64 nz, double eps, double range,
                const dmtz_flags* flags, dmtz_counts* out, uint8_t* d_counter_out, int32_t* sweeps_out) {
    int rc = check_dims(ctx, nx, ny, nz);
    if (rc) return rc;
    if (!flags || !d_f || !d_g) {
        ctx->err = "null argument";
        return DMTZ_E_ARG;
    }
    if (flags->mode != 0) {
        ctx->err = "unknown mode";
        return DMTZ_E_ARG;
    }
    Dims d{nx, ny, nz};
    Counts c = make_counts(d);
    rc = ensure(ctx, c.N, sizeof(T), false);
    if (rc) return rc;
    Driver<T> drv{ctx, d_f, d_g, d, c, eps, range, *flags};
    rc = drv.run(out, sweeps_out);
    if (rc < 0) return rc;
    if (d_counter_out) {
        hipError_t e = hipMemcpyAsync(d_counter_out, ctx->d_counter, (size_t)c.N, hipMemcpyDeviceToDevice, ctx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) {
            ctx->err = hipGetErrorString(e);
            return DMTZ_E_HIP;
        }
    }
    return rc;
}

template <class T>
int correct_host(dmtz_ctx* ctx, const T* f, T* g, i64 nx, i64 ny, i64 nz, double eps, double range,
                 const dmtz_flags* flags, dmtz_counts* out, uint8_t* counter_out, int32_t* sweeps_out) {
    int rc = check_dims(ctx, nx, ny, nz);
    if (rc) return rc;
    if (!f || !g) {
        ctx->err = "null argument";
        return DMTZ_E_ARG;
    }
    i64 N = nx * ny * nz;
    rc = ensure(ctx, N, sizeof(T), true);
    if (rc) return rc;
    CK(hipMemcpyAsync(ctx->d_f, f, sizeof(T) * (size_t)N, hipMemcpyHostToDevice, ctx->stream));
    CK(hipMemcpyAsync(ctx->d_g, g, sizeof(T) * (size_t)N, hipMemcpyHostToDevice, ctx->stream));
    int st = correct_dev<T>(ctx, (const T*)ctx->d_f, (T*)ctx->d_g, nx, ny, nz, eps, range, flags, out, nullptr,
                            sweeps_out);
    if (st < 0) return st;
    CK(hipMemcpyAsync(g, ctx->d_g, sizeof(T) * (size_t)N, hipMemcpyDeviceToHost, ctx->stream));
    if (counter_out)
        CK(hipMemcpyAsync(counter_out, ctx->d_counter, (size_t)N, hipMemcpyDeviceToHost, ctx->stream));
    CK(hipStreamSynchronize(ctx->stream));
    return st;
}

// The classifier alone (dmtz_classify_*): star codes of the field, then counts and masks of the
// cells left unpaired.
template <class T>
int classify_host(dmtz_ctx* ctx, const T* fld, i64 nx, i64 ny, i64 nz, int64_t* counts4, uint64_t* crit_lo,
                  uint32_t* crit_hi) {
    int rc = check_dims(ctx, nx, ny, nz);
    if (rc) return rc;
    if (!fld || !counts4) {
        ctx->err = "null argument";
        return DMTZ_E_ARG;
    }
    const i64 N = nx * ny * nz;
    rc = ensure(ctx, N, sizeof(T), true);
    if (rc) return rc;
    Dims d{nx, ny, nz};
    Counts c = make_counts(d);
    CK(hipMemcpyAsync(ctx->d_f, fld, sizeof(T) * (size_t)N, hipMemcpyHostToDevice, ctx->stream));
    k_code<T><<<nblocks(N), BLOCK, 0, ctx->stream>>>((const T*)ctx->d_f, d, c, CodeArray{ctx->d_code_f, c.N},
                                                   MaskArray{nullptr, nullptr});
    CK(hipGetLastError());
    CK(hipMemsetAsync(ctx->d_ctr, 0, sizeof(ull) * 4, ctx->stream));
    k_crit_count<<<nblocks(N), BLOCK, 0, ctx->stream>>>(CodeArray{ctx->d_code_f, N}, N, ctx->d_ctr);
    CK(hipGetLastError());
    rc = sync_ctr(ctx);
    if (rc) return rc;
    for (int k = 0; k < 4; k++) counts4[k] = (int64_t)ctx->h_ctr[k];
    if (crit_lo || crit_hi) {
        k_critf_own<<<nblocks(N), BLOCK, 0, ctx->stream>>>(CodeArray{ctx->d_code_f, N}, N, ctx->d_critf);
        CK(hipGetLastError());
        if (crit_lo)
            CK(hipMemcpyAsync(crit_lo, ctx->d_critf.lo, sizeof(uint64_t) * (size_t)N, hipMemcpyDeviceToHost, ctx->stream));
        if (crit_hi)
            CK(hipMemcpyAsync(crit_hi, ctx->d_critf.hi, sizeof(uint32_t) * (size_t)N, hipMemcpyDeviceToHost, ctx->stream));
        CK(hipStreamSynchronize(ctx->stream));
    }
    return 0;
}

// Batch correction (dmtz_correct_batch_*). Fields run concurrently in up to BATCH_LANES lanes,
// each a host thread with a worker context of its own (its own stream and buffers), so the
// sweeps of different fields overlap on the device and their per-sweep host round trips
// overlap too. Lanes take the fields largest first from a shared counter. Every field's result
// is what a single correction gives (each run is deterministic and lanes share nothing).
constexpr int BATCH_LANES = 8;

template <class T, class Field>
int correct_one(dmtz_ctx* w, const Field& fd, const dmtz_flags* flags, dmtz_counts* cnt, int32_t* sw) {
    return fd.on_device ? correct_dev<T>(w, fd.f, fd.g, fd.nx, fd.ny, fd.nz, fd.eps, fd.range, flags, cnt, nullptr, sw)
                        : correct_host<T>(w, fd.f, fd.g, fd.nx, fd.ny, fd.nz, fd.eps, fd.range, flags, cnt, nullptr,
                                          sw);
}

template <class T, class Field>
int correct_batch(dmtz_ctx* ctx, const Field* fields, int32_t n, const dmtz_flags* flags, dmtz_counts* counts_out,
                  int32_t* status_out, int32_t* sweeps_out) {
    if (!ctx || !flags || (n > 0 && !fields) || n < 0) {
        if (ctx) ctx->err = "null or invalid argument";
        return DMTZ_E_ARG;
    }
    if (n == 0) return 0;
    const int lanes = n < BATCH_LANES ? n : BATCH_LANES;
    while ((int)ctx->workers.size() < lanes) {
        dmtz_ctx* w = nullptr;
        const int rc = dmtz_ctx_create(&w, ctx->device);
        if (rc) {
            ctx->err = "batch lane context creation failed";
            return rc;
        }
        w->side_stream = false;  // one stream per lane: more would share the four hardware queues
        ctx->workers.push_back(w);
    }
    for (dmtz_ctx* w : ctx->workers) w->err.clear();
    std::vector<int32_t> order(n);
    for (int32_t i = 0; i < n; i++) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
        return fields[a].nx * fields[a].ny * fields[a].nz > fields[b].nx * fields[b].ny * fields[b].nz;
    });
    std::vector<int> rcs(n, DMTZ_E_NOT_RUN);  // fields that never start keep this status
    std::vector<dmtz_counts> cnts(n);
    std::vector<int32_t> sws(n, 0);
    std::atomic<int32_t> next{0};
    std::atomic<bool> failed{false};
    auto lane = [&](dmtz_ctx* w) {
        (void)hipSetDevice(w->device);
        for (;;) {
            const int32_t k = next.fetch_add(1);
            if (k >= n || failed.load()) break;
            const int32_t i = order[k];
            rcs[i] = correct_one<T>(w, fields[i], flags, &cnts[i], &sws[i]);
            if (rcs[i] < 0) failed.store(true);
        }
    };
    std::vector<std::thread> threads;
    for (int l = 1; l < lanes; l++) threads.emplace_back(lane, ctx->workers[l]);
    lane(ctx->workers[0]);
    for (auto& t : threads) t.join();
    (void)hipSetDevice(ctx->device);
    int worst = 0;
    for (int l = 0; l < lanes; l++) {  // kernel statistics of the lanes go to the caller's context
        dmtz_ctx* w = ctx->workers[l];
        ctx->det_launches += w->det_launches;
        ctx->det_ms += w->det_ms;
        ctx->det_bytes += w->det_bytes;
        ctx->det_voxels += w->det_voxels;
        w->det_launches = w->det_ms = w->det_bytes = w->det_voxels = 0;
    }
    int first_err = 0;  // first error in field order (DMTZ_E_NOT_RUN only follows an error)
    for (int32_t i = 0; i < n; i++) {
        if (status_out) status_out[i] = rcs[i];
        if (rcs[i] < 0) {
            if (rcs[i] != DMTZ_E_NOT_RUN && first_err == 0) first_err = rcs[i];
            continue;
        }
        if (counts_out) counts_out[i] = cnts[i];
        if (sweeps_out) sweeps_out[i] = sws[i];
        if (rcs[i] != 0) worst = 1;
    }
    if (first_err) {
        for (dmtz_ctx* w : ctx->workers)
            if (!w->err.empty()) ctx->err = w->err;
        return first_err;
    }
    return worst;
}

template <class T>
int gradient_host(dmtz_ctx* ctx, const T* fld, i64 nx, i64 ny, i64 nz, int64_t* pv, int64_t* pe, int64_t* pf,
                  int64_t* pt) {
    int rc = check_dims(ctx, nx, ny, nz);
    if (rc) return rc;
    Dims d{nx, ny, nz};
    Counts c = make_counts(d);
    rc = ensure(ctx, c.N, sizeof(T), true);
    if (rc) return rc;
    CK(hipMemcpyAsync(ctx->d_f, fld, sizeof(T) * (size_t)c.N, hipMemcpyHostToDevice, ctx->stream));
    k_code<T><<<nblocks(c.N), BLOCK, 0, ctx->stream>>>((const T*)ctx->d_f, d, c, CodeArray{ctx->d_code_f, c.N},
                                                   MaskArray{nullptr, nullptr});
    CK(hipGetLastError());
    int64_t* outs[4] = {pv, pe, pf, pt};
    i64 sizes[4] = {c.N, c.E, c.F, c.T};
    for (int k = 0; k < 4; k++) {
        int64_t* dbuf = nullptr;
        CK(hipMalloc(&dbuf, sizeof(int64_t) * (size_t)(sizes[k] > 0 ? sizes[k] : 1)));
        if (sizes[k] > 0) {
            k_pairing<T><<<nblocks(sizes[k]), BLOCK, 0, ctx->stream>>>((const T*)ctx->d_f, CodeArray{ctx->d_code_f, c.N}, d, c, k,
                                                                        (ull)sizes[k], dbuf);
            hipError_t e = hipGetLastError();
            if (e == hipSuccess)
                e = hipMemcpyAsync(outs[k], dbuf, sizeof(int64_t) * (size_t)sizes[k], hipMemcpyDeviceToHost, ctx->stream);
            if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
            (void)hipFree(dbuf);
            if (e != hipSuccess) {
                ctx->err = hipGetErrorString(e);
                return DMTZ_E_HIP;
            }
        } else {
            (void)hipFree(dbuf);
        }
    }
    return 0;
}

template <class T>
int targets_host(dmtz_ctx* ctx, const T* f, const T* g, i64 nx, i64 ny, i64 nz, double eps, double range,
                 const dmtz_flags* flags, uint8_t* targets, int64_t* counts4) {
    int rc = check_dims(ctx, nx, ny, nz);
    if (rc) return rc;
    Dims d{nx, ny, nz};
    Counts c = make_counts(d);
    rc = ensure(ctx, c.N, sizeof(T), true);
    if (rc) return rc;
    CK(hipMemcpyAsync(ctx->d_f, f, sizeof(T) * (size_t)c.N, hipMemcpyHostToDevice, ctx->stream));
    CK(hipMemcpyAsync(ctx->d_g, g, sizeof(T) * (size_t)c.N, hipMemcpyHostToDevice, ctx->stream));
    CK(hipMemsetAsync(ctx->d_counter, 1, (size_t)c.N, ctx->stream));
    CK(hipMemsetAsync(ctx->d_ctr, 0, sizeof(ull) * K_NCTR, ctx->stream));
    Driver<T> drv{ctx, (const T*)ctx->d_f, (T*)ctx->d_g, d, c, eps, range, *flags};
    rc = drv.f_codes();
    if (rc) return rc;
    rc = drv.g_codes();
    if (rc) return rc;
    rc = drv.detect();
    if (rc) return rc;
    ull cc[4] = {ctx->h_ctr[0], ctx->h_ctr[1], ctx->h_ctr[2], ctx->h_ctr[3]};
    for (int k = 0; k < 4; k++) counts4[k] = (int64_t)cc[k];
    rc = drv.begin_edits();
    if (rc) return rc;
    rc = drv.repair_records(cc, false);
    if (rc) return rc;
    rc = sync_ctr(ctx);
    if (rc) return rc;
    ull nt = ctx->h_ctr[K_TGT];
    std::vector<uint32_t> tl(nt);
    if (nt) CK(hipMemcpyAsync(tl.data(), ctx->d_targets, sizeof(uint32_t) * nt, hipMemcpyDeviceToHost, ctx->stream));
    CK(hipStreamSynchronize(ctx->stream));
    std::memset(targets, 0, (size_t)c.N);
    for (ull k = 0; k < nt; k++) targets[tl[k]] = 1;
    return 0;
}

template <class T>
int paths_host(dmtz_ctx* ctx, const T* f, const T* g, i64 nx, i64 ny, i64 nz, const dmtz_flags* flags,
               int64_t* counts2, int64_t* ds_id, int64_t* ds_rec, int64_t* as_id, int64_t* as_rec, int64_t cap,
               uint8_t* targets) {
    int rc = check_dims(ctx, nx, ny, nz);
    if (rc) return rc;
    if (!flags || !counts2) {
        ctx->err = "null argument";
        return DMTZ_E_ARG;
    }
    Dims d{nx, ny, nz};
    Counts c = make_counts(d);
    rc = ensure(ctx, c.N, sizeof(T), true);
    if (rc) return rc;
    CK(hipMemcpyAsync(ctx->d_f, f, sizeof(T) * (size_t)c.N, hipMemcpyHostToDevice, ctx->stream));
    CK(hipMemcpyAsync(ctx->d_g, g, sizeof(T) * (size_t)c.N, hipMemcpyHostToDevice, ctx->stream));
    CK(hipMemsetAsync(ctx->d_counter, 1, (size_t)c.N, ctx->stream));
    CK(hipMemsetAsync(ctx->d_ctr, 0, sizeof(ull) * K_NCTR, ctx->stream));
    dmtz_flags fl = *flags;
    fl.preserve_vpath = 1;
    fl.preserve_connectors = 0;
    Driver<T> drv{ctx, (const T*)ctx->d_f, (T*)ctx->d_g, d, c, 0.0, 0.0, fl};
    rc = drv.f_codes();
    if (rc) return rc;
    rc = drv.g_codes();
    if (rc) return rc;
    uint64_t* gfaces = nullptr;
    if (fl.preserve_geometry != 1) {
        // get_false_as_vpath_connectivity starts from g's critical faces (main_3d.cu:4766)
        const CodeArray gc = drv.cg();
        rc = drv.fcrit(&gc, 4);
        if (rc) return rc;
        drv.n_gfaces = ctx->h_ctr[K_FC0 + 2];
        CK(hipMalloc(&gfaces, sizeof(uint64_t) * (drv.n_gfaces + 1)));
        hipError_t e = hipMemcpyAsync(gfaces, fcrit_lists(ctx).l[2], sizeof(uint64_t) * drv.n_gfaces,
                                      hipMemcpyDeviceToDevice, ctx->stream);
        if (e != hipSuccess) {
            (void)hipFree(gfaces);
            ctx->err = hipGetErrorString(e);
            return DMTZ_E_HIP;
        }
        drv.as_gfaces = gfaces;
    }
    const CodeArray fcodes = drv.cf();
    drv.list_ids = true;
    rc = drv.prepare_paths(&fcodes);
    if (rc == 0) rc = drv.detect_paths();
    if (gfaces) {
        (void)hipStreamSynchronize(ctx->stream);
        (void)hipFree(gfaces);
    }
    if (rc) return rc;
    ull nds = ctx->h_ctr[K_DS], nas = ctx->h_ctr[K_AS];
    counts2[0] = (int64_t)nds;
    counts2[1] = (int64_t)nas;
    PathList pd = drv.path_list(0), pa = drv.path_list(1);
    ull kd = nds < (ull)cap ? nds : (ull)cap, ka = nas < (ull)cap ? nas : (ull)cap;
    if (kd && ds_id) CK(hipMemcpyAsync(ds_id, pd.id, sizeof(int64_t) * kd, hipMemcpyDeviceToHost, ctx->stream));
    if (kd && ds_rec) CK(hipMemcpyAsync(ds_rec, pd.rec, sizeof(int64_t) * kd, hipMemcpyDeviceToHost, ctx->stream));
    if (ka && as_id) CK(hipMemcpyAsync(as_id, pa.id, sizeof(int64_t) * ka, hipMemcpyDeviceToHost, ctx->stream));
    if (ka && as_rec) CK(hipMemcpyAsync(as_rec, pa.rec, sizeof(int64_t) * ka, hipMemcpyDeviceToHost, ctx->stream));
    CK(hipStreamSynchronize(ctx->stream));
    if (targets) {
        rc = drv.begin_edits();
        if (rc) return rc;
        if (nds + nas) {
            k_fix_paths<T><<<nblocks(nds + nas), BLOCK, 0, ctx->stream>>>(
                pa.rec, nas, pd.rec, nds, nullptr, 0, (const T*)ctx->d_f, drv.cf(), (const T*)ctx->d_g,
                drv.cg(), d, c, ctx->d_counter, 0.0, 0.0, fl.edit_type, drv.sink());
            CK(hipGetLastError());
        }
        rc = sync_ctr(ctx);
        if (rc) return rc;
        ull nt = ctx->h_ctr[K_TGT];
        std::vector<uint32_t> tl(nt);
        if (nt) CK(hipMemcpyAsync(tl.data(), ctx->d_targets, sizeof(uint32_t) * nt, hipMemcpyDeviceToHost, ctx->stream));
        CK(hipStreamSynchronize(ctx->stream));
        std::memset(targets, 0, (size_t)c.N);
        for (ull k = 0; k < nt; k++) targets[tl[k]] = 1;
    }
    CK(hipMemcpyAsync(ctx->h_ctr, ctx->d_ctr, sizeof(ull) * K_NCTR, hipMemcpyDeviceToHost, ctx->stream));
    CK(hipStreamSynchronize(ctx->stream));
    if (ctx->h_ctr[K_WALK] > 0) {
        ctx->err = "a separatrix walk exceeded N steps (cyclic gradient path)";
        return DMTZ_E_WALK;
    }
    return 0;
}

// The 2-saddle wall list on (f, g) as they stand, and optionally the edit set of fix_ds_wall over
// it (eps and range enter its threshold, main_3d.cu:5331).
template <class T>
int walls_host(dmtz_ctx* ctx, const T* f, const T* g, i64 nx, i64 ny, i64 nz, double eps, double range,
               const dmtz_flags* flags, int64_t* count, int64_t* face, int64_t* edge, int64_t cap, uint8_t* targets) {
    int rc = check_dims(ctx, nx, ny, nz);
    if (rc) return rc;
    if (!count || cap < 0) {
        ctx->err = "null argument";
        return DMTZ_E_ARG;
    }
    Dims d{nx, ny, nz};
    Counts c = make_counts(d);
    rc = ensure(ctx, c.N, sizeof(T), true);
    if (rc) return rc;
    CK(hipMemcpyAsync(ctx->d_f, f, sizeof(T) * (size_t)c.N, hipMemcpyHostToDevice, ctx->stream));
    CK(hipMemcpyAsync(ctx->d_g, g, sizeof(T) * (size_t)c.N, hipMemcpyHostToDevice, ctx->stream));
    CK(hipMemsetAsync(ctx->d_counter, 1, (size_t)c.N, ctx->stream));
    CK(hipMemsetAsync(ctx->d_ctr, 0, sizeof(ull) * K_NCTR, ctx->stream));
    dmtz_flags fl{};
    if (flags) fl = *flags;
    fl.preserve_vpath = 1;
    fl.preserve_connectors = 1;
    Driver<T> drv{ctx, (const T*)ctx->d_f, (T*)ctx->d_g, d, c, eps, range, fl};
    rc = drv.f_codes();
    if (rc) return rc;
    rc = drv.g_codes();
    if (rc) return rc;
    const CodeArray fcodes = drv.cf();
    rc = drv.prepare_paths(&fcodes);
    if (rc) return rc;
    rc = drv.walls();
    if (rc) return rc;
    rc = sync_ctr(ctx);
    if (rc) return rc;
    rc = overflow_check(ctx);
    if (rc) return rc;
    const ull nw = ctx->h_ctr[K_DSW];
    *count = (int64_t)nw;
    PathList pw = drv.path_list(2);
    const ull k = nw < (ull)cap ? nw : (ull)cap;
    if (k && face) CK(hipMemcpyAsync(face, pw.id, sizeof(int64_t) * k, hipMemcpyDeviceToHost, ctx->stream));
    if (k && edge) CK(hipMemcpyAsync(edge, pw.rec, sizeof(int64_t) * k, hipMemcpyDeviceToHost, ctx->stream));
    CK(hipStreamSynchronize(ctx->stream));
    if (targets) {
        rc = drv.begin_edits();
        if (rc) return rc;
        if (nw) {
            k_fix_paths<T><<<nblocks(nw), BLOCK, 0, ctx->stream>>>(
                nullptr, 0, nullptr, 0, pw.rec, nw, (const T*)ctx->d_f, drv.cf(), (const T*)ctx->d_g,
                drv.cg(), d, c, ctx->d_counter, eps, range, fl.edit_type, drv.sink());
            CK(hipGetLastError());
        }
        rc = sync_ctr(ctx);
        if (rc) return rc;
        const ull nt = ctx->h_ctr[K_TGT];
        std::vector<uint32_t> tl(nt);
        if (nt) CK(hipMemcpyAsync(tl.data(), ctx->d_targets, sizeof(uint32_t) * nt, hipMemcpyDeviceToHost, ctx->stream));
        CK(hipStreamSynchronize(ctx->stream));
        std::memset(targets, 0, (size_t)c.N);
        for (ull q = 0; q < nt; q++) targets[tl[q]] = 1;
    }
    return 0;
}

template <class T>
int eps_from_rel(const T* f, int64_t n, double rel, double* eps_out, double* range_out) {
    if (!f || n <= 0) return DMTZ_E_ARG;
    double lo = (double)f[0], hi = (double)f[0];
    for (int64_t i = 1; i < n; i++) {
        double x = (double)f[i];
        lo = x < lo ? x : lo;
        hi = x > hi ? x : hi;
    }
    double range = hi - lo;
    if (range_out) *range_out = range;
    if (eps_out) *eps_out = range * rel;  // bound1 = (maxValue - minValue) * range1, :6307
    return 0;
}

}  // namespace
