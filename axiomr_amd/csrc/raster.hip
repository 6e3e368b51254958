// raster.hip - the gfx950 kernels of the tiled render path.
//
// Stage map (reference: src/tiled_pipeline.cpp:143-322 drawMesh):
//   k_prep        zero the per-frame counters and bin counters
//   k_setup       one lane per face: transform, frustum classification, cull,
//                 triangle setup                         (tpl.cpp:185-240, 53-119)
//                 and an entry in every bin it touches   (tpl.cpp:368-393)
//   k_clip        faces that cross a frustum plane: the full 6-plane clipper
//                 (pipeline.cpp:176-370), then cull/setup/bins as above
//   k_raster      one workgroup per bin: coverage and early-Z into LDS keys,
//                 then per-pixel resolve: depth test against the framebuffer,
//                 shading of the winner, BGRA/depth store  (tpl.cpp:395-594,
//                 1125-1181)
//
// Numerics: every coverage and depth value is computed with the reference's
// FP32 formulas in its evaluation order (no contraction), anchored at the
// reference's 16-pixel tiles and 8-pixel steps whatever the bin size here.
// The per-pixel winner is the minimum of the 64-bit key
// (ordered depth, submission key), which equals the reference's first-wins
// strict-less depth test over triangles in submission order.
#include <cstdlib>
#include <rocprofiler-sdk-roctx/roctx.h>
#include "axr_types.hpp"
#include "shade.hpp"
#include "internal.hpp"
#include <hip/hip_ext.h>

#pragma clang fp contract(off)

namespace axr {

// ---------------------------------------------------------------------------
// helpers

template <bool BATCH>
__device__ __forceinline__ const ViewDesc& view_at(const KArgs& ka, uint32_t v) {
    if constexpr (BATCH) return ka.table[v];
    else return ka.one;
}

// Largest i in [0, n) with a[i] <= x (a ascending, a[0] <= x).
__device__ __forceinline__ uint32_t find_le(const uint32_t* a, uint32_t n, uint32_t x) {
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (a[mid] <= x) lo = mid; else hi = mid;
    }
    return lo;
}

// Largest i in [0, n) with a[i] <= x (a ascending, a[0] <= x), searched by
// the whole wave: 64 probes per round, so about log64(n) dependent loads.
// Every lane of the wave must call it with the same arguments.
__device__ __forceinline__ uint32_t wave_find_le(const uint32_t* a, uint32_t n, uint32_t x) {
    uint32_t lo = 0, hi = n;
    const uint32_t lane = __lane_id();
    while (hi - lo > 1) {
        const uint32_t step = (hi - lo + 63) / 64;
        const uint32_t p = lo + lane * step;
        const bool le = p < hi && a[p] <= x;
        const unsigned long long m = __ballot(le);      // a prefix of the lanes (a is ascending)
        const uint32_t last = 63u - (uint32_t)__clzll((long long)m);
        lo = lo + last * step;
        hi = lo + step < hi ? lo + step : hi;
    }
    return lo;
}

// View of face slot g for every lane of a wave (all 64 lanes call it):
// one 64-way search for the wave's first face, then only lanes past that
// view's last face search on their own (a wave rarely spans two views).
__device__ __forceinline__ uint32_t wave_view_of(const uint32_t* bases, uint32_t nviews, uint32_t g, uint32_t total) {
    uint32_t g0 = __shfl(g, 0);
    g0 = g0 < total ? g0 : total - 1;
    const uint32_t v0 = wave_find_le(bases, nviews, g0);
    if (g >= total) return v0;
    return g < bases[v0 + 1] ? v0 : find_le(bases, nviews, g);
}

// The group of submission rank `rank`: the last one that starts at or before
// it.  FEW: groups 1 to 3 are taken from the view (the kernel's arguments, in
// scalar registers); the search in memory is two or three dependent loads
// before a face's indices can be loaded.
template <bool FEW>
__device__ __forceinline__ DevGroup group_of(const ViewDesc& V, uint32_t rank) {
    if (V.ngroups == 1) return V.g0;
    if (FEW && V.ngroups <= 4) {
        DevGroup g = V.g0;
        if (V.g1.rank_base <= rank) g = V.g1;
        if (V.ngroups > 2 && V.g2.rank_base <= rank) g = V.g2;
        if (V.ngroups > 3 && V.g3.rank_base <= rank) g = V.g3;
        return g;
    }
    uint32_t lo = 0, hi = V.ngroups;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (gld(V.groups, mid).rank_base <= rank) lo = mid; else hi = mid;
    }
    return gld(V.groups, lo);
}

__device__ __forceinline__ vec3 load_pos(const float* p, uint32_t i) {
    return gld(reinterpret_cast<const vec3*>(p), i);
}

// One face as the setup stage sees it: submission rank s within its view,
// its group, mesh face index, vertex indices and clip-space corners
// (reference tiled_pipeline.cpp:185-212: gl_Position = mvp * position).
struct FaceGeo {
    DevGroup G;
    uint32_t face, i0, i1, i2;
    vec4 c0, c1, c2;
};

template <bool BATCH>
__device__ __forceinline__ void face_geo(const ViewDesc& V, uint32_t s, FaceGeo& f) {
    f.G = group_of<!BATCH>(V, s);
    f.face = f.G.first + (s - f.G.rank_base);
    const uint3 ix = gld(reinterpret_cast<const uint3*>(V.idx), f.face);
    f.i0 = ix.x;
    f.i1 = ix.y;
    f.i2 = ix.z;
    f.c0 = V.mvp * make4(load_pos(V.pos, f.i0), 1.0f);
    f.c1 = V.mvp * make4(load_pos(V.pos, f.i1), 1.0f);
    f.c2 = V.mvp * make4(load_pos(V.pos, f.i2), 1.0f);
}

// Every 32-bit word of v as the wave's first active lane holds it: for a
// value the whole wave holds in common, so the compiler keeps it in scalar
// registers (and addresses through it with a scalar base).
template <class X>
__device__ __forceinline__ X wave_uniform(const X& v) {
    static_assert(sizeof(X) % 4 == 0, "whole words");
    X r;
    uint32_t w[sizeof(X) / 4];
    __builtin_memcpy(w, &v, sizeof(X));
    for (int i = 0; i < (int)(sizeof(X) / 4); ++i) w[i] = __builtin_amdgcn_readfirstlane(w[i]);
    __builtin_memcpy(&r, w, sizeof(X));
    return r;
}

// The wave's LDS writes before its reads of other lanes' entries.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Wave-aggregated append: returns this lane's slot for lanes with pred set.
__device__ __forceinline__ uint32_t wave_append(uint32_t* counter, bool pred) {
    unsigned long long mask = __ballot(pred);
    uint32_t base = 0;
    int leader = __ffsll((long long)mask) - 1;
    if (pred && (int)__lane_id() == leader) base = atomicAdd(counter, (uint32_t)__popcll(mask));
    base = __shfl(base, leader < 0 ? 0 : leader);
    return base + (uint32_t)__popcll(mask & __lanemask_lt());
}

// A frame's sticky error bit.  The pinned host word is set as well (a
// system-scope store, seen by the host once the kernel has completed), so
// the host learns of an error without copying the counters back after every
// wait; errors are rare, so the store over the host link is too.
__device__ __forceinline__ void raise_error(const Arena& ar, uint32_t bit) {
    atomicOr(&ar.counters[CNT_ERROR], bit);
    if (ar.host_err) __hip_atomic_store(ar.host_err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ void set_error(const Arena& ar, uint32_t bit, uint32_t need_slot, uint32_t need) {
    raise_error(ar, bit);
    atomicMax(&ar.counters[need_slot], need);
}

// Queue face slot g of every lane with pred set for the clipper (the whole
// wave calls it).  A wave's faces go to one of CLIP_SUBS sub-queues, what does
// not fit there to the shared queue, whose size alone decides whether a frame
// fits: one counter for all waves would serialize them, ~9 ns each, 250 us
// for the 4M-triangle soup's 62,500 waves.
__device__ __forceinline__ void queue_clip(const Arena& ar, bool pred, uint32_t g) {
    const unsigned long long mask = __ballot(pred);
    if (mask == 0ull) return;
    const uint32_t sub = ((blockIdx.x * blockDim.x + threadIdx.x) >> 6) % CLIP_SUBS;
    const uint32_t n = (uint32_t)__popcll(mask), mine = (uint32_t)__popcll(mask & __lanemask_lt());
    const int leader = __ffsll((long long)mask) - 1;
    const uint32_t cap = ar.clip_sub_cap;
    uint32_t o = cap;
    if (cap) {
        if ((int)__lane_id() == leader) o = atomicAdd(&ar.clip_next[sub * POOL_STRIDE], n);
        o = __shfl(o, leader);
    }
    const uint32_t fit = o < cap ? (cap - o < n ? cap - o : n) : 0u;   // the first `fit` of them
    if (pred && mine < fit) ar.clip_faces[sub * cap + o + mine] = g;
    if (fit == n) return;
    uint32_t q = 0;
    if ((int)__lane_id() == leader) q = atomicAdd(&ar.counters[CNT_CLIP_FACES], n - fit);
    q = __shfl(q, leader) + mine - fit;
    if (!pred || mine < fit) return;
    if (q < ar.cap_clip_faces) ar.clip_faces[CLIP_SUBS * cap + q] = g;
    else set_error(ar, ERR_CLIP_FACES, CNT_NEED_CLIP_FACES, q + 1);
}

// The frame's last pass leaves the clipper's counters zero (called by the
// threads of one workgroup).
__device__ __forceinline__ void reset_clip_counters(const Arena& ar) {
    if (threadIdx.x == 0) {
        ar.counters[CNT_CLIP_FACES] = 0;
        ar.counters[CNT_CLIP_RECS] = 0;
    }
    if (ar.clip_next && threadIdx.x < CLIP_SUBS) ar.clip_next[threadIdx.x * POOL_STRIDE] = 0;
}

// reference tiled_pipeline.cpp:15-23
__device__ __forceinline__ float clampW(float w) {
    const float tiny = 1e-6f;
    if (fabsf(w) < tiny) w = (w < 0.0f) ? -tiny : tiny;
    return w;
}

// reference pipeline.cpp:274-285
__device__ __forceinline__ float plane_dist(const vec4& v, int plane) {
    switch (plane) {
    case 0: return v.x + v.w;
    case 1: return v.w - v.x;
    case 2: return v.y + v.w;
    case 3: return v.w - v.y;
    case 4: return v.z + v.w;
    default: return v.w - v.z;
    }
}

enum { CLS_INSIDE = 0, CLS_DROP = 1, CLS_CLIP = 2 };
// The clipper's result for the cases it decides without interpolating: a
// triangle inside every plane passes through unchanged, and one entirely
// outside the first plane it is not entirely inside is dropped.  Every other
// triangle goes through the full clipper.
__device__ __forceinline__ int classify(const vec4& a, const vec4& b, const vec4& c) {
    for (int p = 0; p < 6; ++p) {
        float d0 = plane_dist(a, p), d1 = plane_dist(b, p), d2 = plane_dist(c, p);
        if (d0 >= 0.f && d1 >= 0.f && d2 >= 0.f) continue;
        if (d0 < 0.f && d1 < 0.f && d2 < 0.f) return CLS_DROP;
        return CLS_CLIP;
    }
    return CLS_INSIDE;
}

// Triangle setup: screen position (y up) and ndc z of one corner
// (reference tiled_pipeline.cpp:59-65).
// INSIDE, here and in raster_setup: the host's bound (pass_skips) put the
// mesh inside every frustum plane with w in [1e-5, 1e30], so w is not clamped
// and lies in the exponent range of the refined reciprocal, and no screen
// coordinate is NaN or outside int range: the same bits with some 40 fewer
// instructions a face.
template <bool INSIDE>
__device__ __forceinline__ void to_screen(const vec4& c, int W, int H, float& sx, float& sy, float& z) {
    float invW = INSIDE ? rcp_rn_normal(c.w) : rcp_rn(clampW(c.w));
    z = c.z * invW;
    sx = (((c.x * invW) + 1.0f) * 0.5f) * (float)W;
    sy = (((c.y * invW) + 1.0f) * 0.5f) * (float)H;
}

// reference tiled_pipeline.cpp:89-119
__device__ __forceinline__ bool is_backface(const TriRec& r) {
    float dx1 = r.a.z - r.a.x, dy1 = r.a.w - r.a.y;
    float dx2 = r.b.x - r.a.x, dy2 = r.b.y - r.a.y;
    return (dx1 * dy2 - dx2 * dy1) < 0;
}

template <bool INSIDE = false>
__device__ __forceinline__ TriRec make_rec(const vec4& c0, const vec4& c1, const vec4& c2, int W, int H) {
    TriRec r;
    float z0, z1, z2;
    to_screen<INSIDE>(c0, W, H, r.a.x, r.a.y, z0);
    to_screen<INSIDE>(c1, W, H, r.a.z, r.a.w, z1);
    to_screen<INSIDE>(c2, W, H, r.b.x, r.b.y, z2);
    r.b.z = z0; r.b.w = z1;
    r.c.x = __float_as_uint(z2);
    return r;
}

// Edge functions of one triangle as the reference raster prepares them
// (tiled_pipeline.cpp:436-487), plus its pixel bounds.
struct RasterTri {
    float a0, b0, c0, a1, b1, c1, a2, b2, c2;
    float inv_area;
    float z0, z1, z2;
    int fx0, fy0, cx1, cy1;   // (int)floor(min), (int)ceil(max)
};

// The largest float below 1e-12: the reference's area test compares in double
// ((double)area < 1e-12), which for a float is area <= this.
constexpr float AREA_NONE = 9.99999996e-13f;
static_assert((double)AREA_NONE < 1.0e-12 && (double)1.00000011e-12f > 1.0e-12, "neighbours of 1e-12");

template <bool INSIDE = false>
__device__ __forceinline__ bool raster_setup(const TriRec& r, RasterTri& t) {
    const float x0 = r.a.x, y0 = r.a.y, x1 = r.a.z, y1 = r.a.w, x2 = r.b.x, y2 = r.b.y;
    if constexpr (INSIDE) {
        t.fx0 = (int)floorf(fminf(fminf(x0, x1), x2));
        t.fy0 = (int)floorf(fminf(fminf(y0, y1), y2));
        t.cx1 = (int)ceilf(fmaxf(fmaxf(x0, x1), x2));
        t.cy1 = (int)ceilf(fmaxf(fmaxf(y0, y1), y2));
    } else {
        t.fx0 = cvt_i32(floorf(smin3(x0, x1, x2)));
        t.fy0 = cvt_i32(floorf(smin3(y0, y1, y2)));
        t.cx1 = cvt_i32(ceilf(smax3(x0, x1, x2)));
        t.cy1 = cvt_i32(ceilf(smax3(y0, y1, y2)));
    }
    float c0 = x1 * y2 - x2 * y1;
    float c1 = x2 * y0 - x0 * y2;
    float c2 = x0 * y1 - x1 * y0;
    float area = (c0 + c1) + c2;
    if (area >= 0 && area <= AREA_NONE) return false;
    float a0 = y1 - y2, b0 = x2 - x1;
    float a1 = y2 - y0, b1 = x0 - x2;
    float a2 = y0 - y1, b2 = x1 - x0;
    if (area < 0) {
        a0 = -a0; b0 = -b0; c0 = -c0;
        a1 = -a1; b1 = -b1; c1 = -c1;
        a2 = -a2; b2 = -b2; c2 = -c2;
        area = -area;
    }
    t.a0 = a0; t.b0 = b0; t.c0 = c0;
    t.a1 = a1; t.b1 = b1; t.c1 = c1;
    t.a2 = a2; t.b2 = b2; t.c2 = c2;
    t.inv_area = rcp_rn(area);
    t.z0 = r.b.z; t.z1 = r.b.w; t.z2 = __uint_as_float(r.c.x);
    return true;
}

// Pixel rectangle [x0,x1) x [y0,y1) that the reference raster visits for
// this triangle over the whole screen.
struct Rect { int x0, y0, x1, y1; };
__device__ __forceinline__ Rect screen_rect(const RasterTri& t, int W, int H) {
    return Rect{imax(0, t.fx0), imax(0, t.fy0), imin(W, t.cx1), imin(H, t.cy1)};
}

// Coverage and depth of pixel (px, py), reference tiled_pipeline.cpp:502-562:
// the row value is anchored at sx = max(16*(px/16), floor(minX)); pixels 8..15
// past the anchor take one +8*a step; then + a*lane.
__device__ __forceinline__ bool cover(const RasterTri& t, int px, int py, float& al, float& be, float& ga, float& z) {
    const int sx = imax(px & ~15, t.fx0);
    const float sxc = (float)sx + 0.5f;
    const float pyc = (float)py + 0.5f;
    float r0 = (t.a0 * sxc + t.b0 * pyc) + t.c0;
    float r1 = (t.a1 * sxc + t.b1 * pyc) + t.c1;
    float r2 = (t.a2 * sxc + t.b2 * pyc) + t.c2;
    const int d = px - sx;
    if (d >= 8) {
        r0 = r0 + t.a0 * 8.0f;
        r1 = r1 + t.a1 * 8.0f;
        r2 = r2 + t.a2 * 8.0f;
    }
    const float lane = (float)(d & 7);
    const float e0 = r0 + t.a0 * lane;
    const float e1 = r1 + t.a1 * lane;
    const float e2 = r2 + t.a2 * lane;
    if (!(e0 >= 0.f && e1 >= 0.f && e2 >= 0.f)) return false;
    al = e0 * t.inv_area;
    be = e1 * t.inv_area;
    ga = e2 * t.inv_area;
    z = (t.z0 * al + t.z1 * be) + t.z2 * ga;
    return true;
}

// Keeps a branch that few waves take a branch: the compiler turns a short one
// into selects, whose operations then run for every pixel.
__device__ __forceinline__ void keep_branch() { asm volatile(""); }

// cover()'s z for a pixel d past the anchor whose edge products are
// x0 = a0 * (anchor + 0.5), ...: the walks take those once per run of pixels.
// Few lanes of a wave are ever 8 or more past their anchor, so that step is a
// branch on the wave's lanes.
__device__ __forceinline__ bool cover_from(const RasterTri& t, float x0, float x1, float x2, int d, float pyc, float& z) {
    float r0 = (x0 + t.b0 * pyc) + t.c0;
    float r1 = (x1 + t.b1 * pyc) + t.c1;
    float r2 = (x2 + t.b2 * pyc) + t.c2;
    float lane = (float)d;
    if (d >= 8) {
        keep_branch();
        r0 = r0 + t.a0 * 8.0f;
        r1 = r1 + t.a1 * 8.0f;
        r2 = r2 + t.a2 * 8.0f;
        lane = lane - 8.0f;   // whole numbers: exact
    }
    const float e0 = r0 + t.a0 * lane;
    const float e1 = r1 + t.a1 * lane;
    const float e2 = r2 + t.a2 * lane;
    if (!(e0 >= 0.f && e1 >= 0.f && e2 >= 0.f)) return false;
    z = (t.z0 * (e0 * t.inv_area) + t.z1 * (e1 * t.inv_area)) + t.z2 * (e2 * t.inv_area);
    return z < INFINITY;
}

// 64-bit depth key: order-preserving image of z (with -0 folded onto +0, the
// reference's strict-less test treats them as equal) above the submission key.
__device__ __forceinline__ unsigned long long depth_key(float z, uint32_t key) {
    uint32_t u = __float_as_uint(z);
    if ((u << 1) == 0) u = 0;
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((unsigned long long)u << 32) | key;
}
constexpr unsigned long long EMPTY_KEY = ~0ull;

// ---------------------------------------------------------------------------
// k_prep: zero per-frame counters (the sticky error word and the "need"
// high-water marks are left alone), the bin counters and the bins' chunk
// table.

// The arena cleans itself during a frame (k_raster zeroes what it consumed),
// so k_prep runs only after the arena is (re)allocated or after an overflow.
__global__ void k_prep(Arena ar, uint32_t ntiles) {
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid < CNT_ERROR || tid == CNT_BIG_ITEMS || tid == CNT_BIG_RECS) ar.counters[tid] = 0;
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = tid; i < ntiles; i += stride) ar.tile_count[i] = 0;
    for (uint32_t i = tid; i < ar.cap_chunks; i += stride) ar.bin_chunks[i] = 0;
    if (ar.pool_next)
        for (uint32_t i = tid; i < (POOL_SUBS + 1) * POOL_STRIDE; i += stride) ar.pool_next[i] = 0;
    if (ar.clip_next)
        for (uint32_t i = tid; i < CLIP_SUBS * POOL_STRIDE; i += stride) ar.clip_next[i] = 0;
    for (uint32_t i = tid; i < ar.cap_vkeys; i += stride) ar.vkeys[i] = ~0ull;
}

// ---------------------------------------------------------------------------
// binning helpers

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const int lane = (int)__lane_id();
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t t = __shfl_up(v, o);
        if (lane >= o) v += t;
    }
    return v;
}

// Bins of T x T pixels that a pixel rectangle of view V touches: nx x ny from
// bin `first` on, rows `pitch` bins apart.
template <int T>
struct BinRange {
    uint32_t first, pitch, nx, n;
    __device__ __forceinline__ BinRange(const ViewDesc& V, const Rect& rc, bool on) {
        first = pitch = nx = n = 0;
        if (on) {
            const int tx0 = rc.x0 / T, ty0 = rc.y0 / T;
            nx = (uint32_t)((rc.x1 - 1) / T - tx0 + 1);
            n = nx * (uint32_t)((rc.y1 - 1) / T - ty0 + 1);
            pitch = (uint32_t)V.tiles_x;
            first = V.tile_base + (uint32_t)ty0 * pitch + (uint32_t)tx0;
        }
    }
};
__device__ __forceinline__ uint32_t bin_of(uint32_t first, uint32_t pitch, uint32_t nx, uint32_t k) {
    return first + k / nx * pitch + k % nx;
}

// Bins (binned mode).  A bin's entries, record references, fill levels: the
// first holds 2^bin0_shift entries at a place of the bin's own, level k holds
// 2^(bin0_shift + k) wherever the pools had room (bin_chunks names the place).
// The lane that takes an entry writes it there at once, so no pass after the
// setup sorts pairs into bins (pairs of 16 bytes, a prefix sum over the bins
// and a scatter took two launches, 8 us of a small frame, and 120 us of the
// 4M-triangle soup's 730).  The host sizes the first level for four times the
// mean of faces per bin, so most bins of most frames never leave it.

// Room for one chunk of n entries: from the sub-pool that the bin's number
// picks (one counter for all bins would serialize the allocations, ~11 ns
// each) or, when that is full or the chunk a large part of it, the shared
// pool, whose size alone decides whether a frame fits.  0 if it does not,
// else the chunk's first entry + 1.
__device__ __forceinline__ uint32_t pool_take(const Arena& ar, uint32_t bin, uint32_t n) {
    const uint32_t sub = bin % POOL_SUBS;
    uint32_t* next = ar.pool_next + sub * POOL_STRIDE;
    if (n <= ar.sub_cap / 4u && __hip_atomic_load(next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < ar.sub_cap) {
        const uint32_t o = atomicAdd(next, n);
        if (o + n <= ar.sub_cap) return sub * ar.sub_cap + o + 1u;
    }
    const uint32_t o = atomicAdd(ar.pool_next + POOL_SUBS * POOL_STRIDE, n);
    if ((unsigned long long)o + n <= ar.pool_cap) return POOL_SUBS * ar.sub_cap + o + 1u;
    set_error(ar, ERR_PAIRS, CNT_NEED_PAIRS, o + n < o ? ~0u : o + n);
    return 0u;
}

// Store this lane's Q entries (act: it has one), whose slots the wave has
// taken; all 64 lanes call it.  The lane that took a level's first slot
// allocates the level and publishes it in the chunk table; the others wait for
// that word.  The wait ends: a level's first slot was taken before any later
// one of it, and the wave that took it publishes all the levels it opened
// before it waits for any other wave's (place_entries).
constexpr uint32_t BIN_WAIT_TRIES = 1u << 20;   // about a second
template <uint32_t Q>
struct BinStore {
    const Arena& ar;
    const bool (&act)[Q];
    const uint32_t (&bin)[Q], (&slot)[Q], (&ref)[Q];
    __device__ __forceinline__ uint32_t* cell(uint32_t q, const BinSlot& b) const {
        return ar.bin_chunks + (size_t)bin[q] * BIN_LEVELS + b.level;
    }
    __device__ __forceinline__ bool near(uint32_t q) {
        const bool first = (slot[q] >> ar.bin0_shift) == 0u;
        if (act[q] && first) ar.bins[((size_t)bin[q] << ar.bin0_shift) + slot[q]] = ref[q];
        return act[q] && !first;
    }
    __device__ __forceinline__ bool any(bool far) const { return __ballot(far) != 0ull; }
    __device__ __forceinline__ void open(uint32_t q) {
        const BinSlot b = bin_slot(ar.bin0_shift, slot[q]);
        if (act[q] && b.level != 0u && b.offset == 0u) {
            const uint32_t at = pool_take(ar, bin[q], 1u << (ar.bin0_shift + b.level));
            __hip_atomic_store(cell(q, b), at ? at : CHUNK_NONE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __device__ __forceinline__ void fill(uint32_t q) {
        const BinSlot b = bin_slot(ar.bin0_shift, slot[q]);
        const bool spill = act[q] && b.level != 0u;
        uint32_t at = 0u;
        for (uint32_t tries = 0; __ballot(spill && at == 0u) != 0ull; ++tries) {
            if (spill && at == 0u) at = __hip_atomic_load(cell(q, b), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (tries == BIN_WAIT_TRIES && spill && at == 0u) {   // never seen; a frame that is redrawn, not a hang
                raise_error(ar, ERR_PAIRS);
                at = CHUNK_NONE;
            }
        }
        if (spill && at != CHUNK_NONE) ar.bin_pool[(size_t)(at - 1u) + b.offset] = ref[q];
    }
};

// Entry i of bin t.
__device__ __forceinline__ uint32_t bin_get(const Arena& ar, uint32_t t, uint32_t i) {
    const BinSlot b = bin_slot(ar.bin0_shift, i);
    if (b.level == 0u) return ar.bins[((size_t)t << ar.bin0_shift) + i];
    return ar.bin_pool[(size_t)(ar.bin_chunks[(size_t)t * BIN_LEVELS + b.level] - 1u) + b.offset];
}

// Put one record per lane (on) into every bin of its rectangle, for a whole
// wave (all 64 lanes must call it).
// Where at least half the lanes repeat their neighbour's first bin (a mesh's
// consecutive faces) and none has more than a handful of bins, the wave goes
// round by round, a bin per lane, and lanes of one bin share one atomic on
// its count.  Else (a soup; large triangles) sharing finds nothing and a
// lane with more bins would keep the others waiting, so the wave's (lane,
// bin) pairs are laid end to end and the lanes take them in turn, EMIT_AHEAD
// atomics in flight each.
constexpr uint32_t EMIT_ROUNDS = 6, EMIT_AHEAD = 4;

template <int T>
__device__ __forceinline__ void emit_bins_wave(const Arena& ar, const ViewDesc& V, bool on, const Rect& rc,
                                               uint32_t ref) {
    const BinRange<T> br(V, rc, on);
    const uint32_t n = br.n, lane = __lane_id();
    const uint32_t bin0 = n ? br.first : ~0u, prev0 = __shfl_up(bin0, 1);
    const unsigned long long any = __ballot(n != 0u);
    if (any == 0ull) return;
    if (__ballot(n > EMIT_ROUNDS) == 0ull && 2 * __popcll(__ballot(n != 0u && bin0 == prev0)) >= __popcll(any)) {
        for (uint32_t k = 0;; ++k) {
            const bool act = k < n;
            const unsigned long long live = __ballot(act);
            if (live == 0ull) return;
            const uint32_t bin = act ? bin_of(br.first, br.pitch, br.nx, k) : ~0u;
            uint32_t slot = 0;
            // group the lanes by bin (register work only), then every
            // group's first lane takes the group's slots with one atomic,
            // all groups' atomics in flight together
            unsigned long long pending = live, mine = 0ull;
            int leader_of_mine = 0;
            while (pending) {
                const int leader = __ffsll((long long)pending) - 1;
                const uint32_t lb = __builtin_amdgcn_readlane(bin, leader);
                const unsigned long long m = __ballot(act && bin == lb);
                if ((m >> lane) & 1ull) {
                    mine = m;
                    leader_of_mine = leader;
                }
                pending &= ~m;
            }
            if (act && leader_of_mine == (int)lane) slot = atomicAdd(&ar.tile_count[count_word(bin)], (uint32_t)__popcll(mine));
            slot = __shfl(slot, leader_of_mine) + (uint32_t)__popcll(mine & __lanemask_lt());
            const bool acts[1] = {act};
            const uint32_t bins[1] = {bin}, slots[1] = {slot}, refs[1] = {ref};
            BinStore<1> store{ar, acts, bins, slots, refs};
            place_entries<1>(store);
        }
    }
    const uint32_t incl = wave_incl_scan(n), start = incl - n, total = __shfl(incl, 63);
    for (uint32_t j0 = 0; j0 < total; j0 += 64u * EMIT_AHEAD) {
        bool act[EMIT_AHEAD];
        uint32_t bin[EMIT_AHEAD], slot[EMIT_AHEAD], r[EMIT_AHEAD];
#pragma unroll
        for (uint32_t q = 0; q < EMIT_AHEAD; ++q) {
            const uint32_t j = j0 + 64u * q + lane;
            // the last lane whose pairs start at or before j (a lane without
            // pairs shares its start with the next lane that has some)
            int o = 0;
            for (int step = 32; step; step >>= 1)
                if (__shfl(start, o + step) <= j) o += step;
            // the owner's own: the lanes of a batch's wave may lie in two views
            const uint32_t first = __shfl(br.first, o), pitch = __shfl(br.pitch, o), nx = __shfl(br.nx, o);
            const uint32_t k = j - __shfl(start, o);
            r[q] = __shfl(ref, o);
            slot[q] = bin[q] = 0u;
            act[q] = j < total;
            if (act[q]) {
                bin[q] = bin_of(first, pitch, nx, k);
                slot[q] = atomicAdd(&ar.tile_count[count_word(bin[q])], 1u);
            }
        }
        BinStore<EMIT_AHEAD> store{ar, act, bin, slot, r};
        place_entries<EMIT_AHEAD>(store);
    }
}

// ---------------------------------------------------------------------------
// visibility mode: helpers

// Pixels of a large triangle's screen rectangle per work item: one wave,
// four pixels per lane.
constexpr uint32_t BIG_CHUNK = 256;

__device__ __forceinline__ unsigned long long* big_counter(const Arena& ar) {
    return reinterpret_cast<unsigned long long*>(ar.counters + CNT_BIG_ITEMS);
}

// Mark the bins of rectangle rc as holding visibility keys.
template <int T>
__device__ __forceinline__ void flag_bins(const Arena& ar, const ViewDesc& V, const Rect& rc) {
    const int tx1 = (rc.x1 - 1) / T, ty1 = (rc.y1 - 1) / T;
    for (int ty = rc.y0 / T; ty <= ty1; ++ty)
        for (int tx = rc.x0 / T; tx <= tx1; ++tx) ar.tile_count[V.tile_base + (uint32_t)(ty * V.tiles_x + tx)] = 1u;
}

// The same by a whole wave (the same rc in every lane).
template <int T>
__device__ __forceinline__ void flag_bins_wave(const Arena& ar, const ViewDesc& V, const Rect& rc) {
    const int tx0 = rc.x0 / T, ty0 = rc.y0 / T, nx = (rc.x1 - 1) / T - tx0 + 1, ny = (rc.y1 - 1) / T - ty0 + 1;
    for (int k = (int)__lane_id(); k < nx * ny; k += 64)
        ar.tile_count[V.tile_base + (uint32_t)((ty0 + k / nx) * V.tiles_x + tx0 + k % nx)] = 1u;
}

// One lane rasterizes a whole (small) triangle: every covered pixel of rc
// takes the minimum of its 64-bit key.
template <int T>
__device__ __forceinline__ void vis_raster_rect(const Arena& ar, const ViewDesc& V, const RasterTri& rt, const Rect& rc,
                                                uint32_t key) {
    unsigned long long* vk = ar.vkeys + V.pix_base;
    bool any = false;
    // Rectangles of at most 8 columns, as nearly all of a fine mesh's: no
    // pixel lies 8 or more past its anchor, and by columns the anchor, its
    // products and the pixel's step are taken once per column (the operations
    // of cover() on the same values, so the same bits)
    if (__ballot(rc.x1 - rc.x0 > 8 || rc.x0 != rt.fx0) == 0ull) {
        for (int px = rc.x0; px < rc.x1; ++px) {
            const int sx = imax(px & ~15, rt.fx0);
            const float sxc = (float)sx + 0.5f, step = (float)(px - sx);
            const float x0 = rt.a0 * sxc, x1 = rt.a1 * sxc, x2 = rt.a2 * sxc;
            const float s0 = rt.a0 * step, s1 = rt.a1 * step, s2 = rt.a2 * step;
            for (int py = rc.y0; py < rc.y1; ++py) {
                const float pyc = (float)py + 0.5f;
                const float e0 = ((x0 + rt.b0 * pyc) + rt.c0) + s0;
                const float e1 = ((x1 + rt.b1 * pyc) + rt.c1) + s1;
                const float e2 = ((x2 + rt.b2 * pyc) + rt.c2) + s2;
                if (e0 >= 0.f && e1 >= 0.f && e2 >= 0.f) {
                    const float z = (rt.z0 * (e0 * rt.inv_area) + rt.z1 * (e1 * rt.inv_area)) + rt.z2 * (e2 * rt.inv_area);
                    if (z < INFINITY) {
                        atomicMin(&vk[(size_t)py * (size_t)V.W + (size_t)px], depth_key(z, key));
                        any = true;
                    }
                }
            }
        }
    } else {
        for (int py = rc.y0; py < rc.y1; ++py)
            for (int px = rc.x0; px < rc.x1; ++px) {
                float al, be, ga, z;
                if (cover(rt, px, py, al, be, ga, z) && z < INFINITY) {
                    atomicMin(&vk[(size_t)py * (size_t)V.W + (size_t)px], depth_key(z, key));
                    any = true;
                }
            }
    }
    if (any) flag_bins<T>(ar, V, rc);
}

__device__ __forceinline__ uint32_t big_chunks(uint32_t area) { return (area + BIG_CHUNK - 1) / BIG_CHUNK; }

__device__ __forceinline__ void big_store(const Arena& ar, const TriRec& r, uint32_t ri, uint32_t i0, uint32_t nch) {
    if (ri >= ar.cap_big_recs || i0 + nch > ar.cap_big_items || i0 + nch < i0) {
        raise_error(ar, ERR_BIG);
        atomicMax(&ar.counters[CNT_NEED_BIG_RECS], ri + 1);
        atomicMax(&ar.counters[CNT_NEED_BIG_ITEMS], i0 + nch);
        return;
    }
    ar.big_rec[ri] = r;
    ar.big_start[ri] = i0;
}

// Queue large triangles (one per flagged lane, whole wave calls): one
// record each plus ceil(area / BIG_CHUNK) work items.  Records and items
// come from one 64-bit counter, so item starts grow with the record index.
__device__ __forceinline__ void big_append_wave(const Arena& ar, bool big, const TriRec& r, uint32_t area) {
    const unsigned long long mask = __ballot(big);
    if (mask == 0ull) return;
    const uint32_t nch = big ? big_chunks(area) : 0u;
    const uint32_t incl = wave_incl_scan(nch);
    const uint32_t total = __shfl(incl, 63);
    unsigned long long old = 0;
    if (__lane_id() == 0) old = atomicAdd(big_counter(ar), ((unsigned long long)__popcll(mask) << 32) | total);
    const uint32_t lo = __shfl((uint32_t)old, 0), hi = __shfl((uint32_t)(old >> 32), 0);
    if (!big) return;
    big_store(ar, r, hi + (uint32_t)__popcll(mask & __lanemask_lt()), lo + incl - nch, nch);
}

// ---------------------------------------------------------------------------
// k_setup: one lane per face (submission order across views).

// Face slot of this lane: 2^face_shift consecutive faces per wave, in its
// first lanes (~0: none).  A draw of few faces takes 16 faces per wave, so
// that the wave's other lanes help with what comes after the setup: bin
// entries, coverage.
__device__ __forceinline__ uint32_t face_slot(const KArgs& ka) {
    const uint32_t wave = (blockIdx.x * 256u + threadIdx.x) >> 6, lane = __lane_id();
    return (lane >> ka.face_shift) == 0u ? (wave << ka.face_shift) + lane : ~0u;
}

// A triangle record stored with the non-temporal hint: the batch's records
// far exceed the caches and are read back only by the raster.
__device__ __forceinline__ void store_rec_nt(TriRec* p, const TriRec& r) {
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    v4u* q = reinterpret_cast<v4u*>(p);
    gst_nt(q, 0, v4u{__float_as_uint(r.a.x), __float_as_uint(r.a.y), __float_as_uint(r.a.z), __float_as_uint(r.a.w)});
    gst_nt(q, 1, v4u{__float_as_uint(r.b.x), __float_as_uint(r.b.y), __float_as_uint(r.b.z), __float_as_uint(r.b.w)});
    gst_nt(q, 2, v4u{r.c.x, r.c.y, r.c.z, r.c.w});
}

// Face slot g of view V (all 64 lanes of the wave call it).
template <int T, bool BATCH, bool INSIDE>
__device__ __forceinline__ void setup_face(const KArgs& ka, const Arena& ar, uint32_t g, bool active, const ViewDesc& V) {
    bool want_clip = false, binnable = false;
    Rect rc{0, 0, 0, 0};
    if (active) {
        const uint32_t s = g - V.face_base;
        FaceGeo f;
        face_geo<BATCH>(V, s, f);
        int cls = CLS_INSIDE;
        if constexpr (!INSIDE) cls = classify(f.c0, f.c1, f.c2);
        want_clip = cls == CLS_CLIP;
        if (cls == CLS_INSIDE) {
            TriRec r = make_rec<INSIDE>(f.c0, f.c1, f.c2, V.W, V.H);
            if (!is_backface(r)) {
                RasterTri rt;
                if (raster_setup<INSIDE>(r, rt)) {
                    rc = screen_rect(rt, V.W, V.H);
                    if (rc.x0 < rc.x1 && rc.y0 < rc.y1) {
                        r.c.y = s * 8u;
                        r.c.z = f.face;
                        r.c.w = f.G.material & REC_MATERIAL_MASK;
                        store_rec_nt(ar.rec + g, r);
                        binnable = true;
                    }
                }
            }
        }
    }
    queue_clip(ar, want_clip, g);
    if (want_clip && ka.skip_clip) raise_error(ar, ERR_SKIPPED);
    emit_bins_wave<T>(ar, V, binnable, rc, g);
}

// INSIDE: the host's bound put every view's mesh inside every frustum plane
// (ka.skip_clip), so the classification is left out, as in k_vis.  A batch
// wave whose faces lie in one view leaves it out for a view the bound puts
// inside (ViewDesc::inside), a branch on a value the wave holds in common.
template <int T, bool BATCH, bool INSIDE = false>
__global__ __launch_bounds__(256) void k_setup(KArgs ka, Arena ar) {
    const uint32_t g = face_slot(ka);
    const bool active = g < ka.total_faces;
    if (ar.counters[CNT_ERROR]) return;
    if constexpr (BATCH) {
        const uint32_t vi = wave_view_of(ka.face_bases, ka.nviews, g, ka.total_faces);
        const uint32_t v0 = __builtin_amdgcn_readfirstlane(vi);
        if (__ballot(vi != v0) == 0ull) {
            // the whole wave in one view (the usual case): the view's fields
            // in scalar registers, loaded once for the wave
            const ViewDesc V = wave_uniform(ka.table[v0]);
            if (INSIDE || V.inside) setup_face<T, BATCH, true>(ka, ar, g, active, V);
            else setup_face<T, BATCH, false>(ka, ar, g, active, V);
        } else {
            setup_face<T, BATCH, INSIDE>(ka, ar, g, active, ka.table[vi]);
        }
    } else {
        setup_face<T, BATCH, INSIDE>(ka, ar, g, active, ka.one);
    }
}

// ---------------------------------------------------------------------------
// Walks of triangles' pixel rectangles by a wave (k_vis, k_raster): a lane
// walks at most CAP pixels of its own rectangle, the rest of every longer one
// is cut into pieces of CAP pixels that the wave's lanes take in turn.  What a
// walker needs of a triangle, per lane, and the first piece of each lane in
// the wave's numbering:
constexpr int VIS_CAP = 8;
struct WalkPieces {
    float4 e0[64];        // a0, b0, c0, a1
    float4 e1[64];        // b1, c1, a2, b2
    float4 e2[64];        // c2, inv_area, z0, z1
    float4 e3[64];        // z2, bits(fx0), bits(rect), bits(key)
    uint32_t start[64];
};
__device__ __forceinline__ void put_piece(WalkPieces* wp, uint32_t lane, const RasterTri& rt, uint32_t, uint32_t rect,
                                          uint32_t key) {
    wp->e0[lane] = make_float4(rt.a0, rt.b0, rt.c0, rt.a1);
    wp->e1[lane] = make_float4(rt.b1, rt.c1, rt.a2, rt.b2);
    wp->e2[lane] = make_float4(rt.c2, rt.inv_area, rt.z0, rt.z1);
    wp->e3[lane] = make_float4(rt.z2, __int_as_float(rt.fx0), __uint_as_float(rect), __uint_as_float(key));
}
__device__ __forceinline__ void get_piece(const WalkPieces* wp, const Arena&, uint32_t o, RasterTri& t, uint32_t& rect,
                                          uint32_t& key) {
    const float4 f0 = wp->e0[o], f1 = wp->e1[o], f2 = wp->e2[o], f3 = wp->e3[o];
    t.a0 = f0.x; t.b0 = f0.y; t.c0 = f0.z; t.a1 = f0.w;
    t.b1 = f1.x; t.c1 = f1.y; t.a2 = f1.z; t.b2 = f1.w;
    t.c2 = f2.x; t.inv_area = f2.y; t.z0 = f2.z; t.z1 = f2.w;
    t.z2 = f3.x; t.fx0 = __float_as_int(f3.y);
    rect = __float_as_uint(f3.z);
    key = __float_as_uint(f3.w);
}

// ---------------------------------------------------------------------------
// k_vis: visibility mode's setup.  One lane per face: the same transform,
// classification, cull and setup as k_setup; a triangle whose screen
// rectangle has at most small_footprint pixels is rasterized by its lane
// straight into the key buffer, a larger one is queued as work items,
// faces that cross a plane go to the clipper.

// SHARE: where a rectangle of the wave outlasts VIS_SHARE pixels, its lanes
// would idle while one walks it; then a lane walks VIS_CAP pixels of its own
// rectangle and the rest goes in pieces of VIS_CAP to all lanes in turn, as
// in k_raster.  At 1080p k_vis takes 38 us without and 18 with it for 32,000
// faces, 22 and 10 for 2,000; but 21.2 and 22.1 for a million faces and 23.0
// and 24.3 for 200,000, whose rectangles are a few pixels.  So the host takes
// it where the target has at least VIS_SHARE pixels per face.
constexpr uint32_t VIS_SHARE = 16;

struct VisPieces : WalkPieces {   // rect: x0 | y0 << 16
    uint32_t size[64];            // w | h << 16
    uint32_t view[64];
};

// Pixels [q0, q1) of the rectangle [x0, x0 + w) x [y0, ...) of view V in
// row-major order: every covered one takes the minimum of its key and flags
// its bin.
template <int T>
__device__ __forceinline__ void vis_span(const Arena& ar, const ViewDesc& V, const RasterTri& rt, int x0, int y0, int w,
                                         int q0, int q1, uint32_t key, float inv_w) {
    unsigned long long* vk = ar.vkeys + V.pix_base;
    // row of q0 as in walk_span (q0 <= 1024, the footprint limit)
    const int dy = q0 == 0 ? 0 : (int)(((float)q0 + 0.5f) * inv_w);
    int px = x0 + (q0 - dy * w), py = y0 + dy;
    uint32_t flagged = ~0u;
    for (int q = q0; q < q1; ++q) {
        const int sx = imax(px & ~15, rt.fx0);
        const float sxc = (float)sx + 0.5f;
        float z;
        if (cover_from(rt, rt.a0 * sxc, rt.a1 * sxc, rt.a2 * sxc, px - sx, (float)py + 0.5f, z)) {
            atomicMin(&vk[(size_t)py * (size_t)V.W + (size_t)px], depth_key(z, key));
            const uint32_t b = V.tile_base + (uint32_t)(py / T * V.tiles_x + px / T);
            if (b != flagged) ar.tile_count[b] = 1u;
            flagged = b;
        }
        if (++px == x0 + w) {
            px = x0;
            ++py;
        }
    }
}

// All 64 lanes call it; on: this lane has a triangle of view vi with
// rectangle rc.
template <int T, bool BATCH>
__device__ __forceinline__ void vis_walk_wave(VisPieces* wp, const KArgs& ka, const Arena& ar, bool on, const RasterTri& rt,
                                              const Rect& rc, uint32_t vi, uint32_t key) {
    const uint32_t lane = __lane_id();
    const int w = on ? rc.x1 - rc.x0 : 0, fp = on ? w * (rc.y1 - rc.y0) : 0;
    if (on) vis_span<T>(ar, view_at<BATCH>(ka, vi), rt, rc.x0, rc.y0, w, 0, imin(fp, VIS_CAP), key, 0.0f);
    const uint32_t pieces = fp > VIS_CAP ? (uint32_t)(fp - 1) / VIS_CAP : 0u;
    const uint32_t incl = wave_incl_scan(pieces), total = __shfl(incl, 63);
    wp->start[lane] = incl - pieces;
    if (pieces) {
        put_piece(wp, lane, rt, 0u, (uint32_t)rc.x0 | ((uint32_t)rc.y0 << 16), key);
        wp->size[lane] = (uint32_t)w | ((uint32_t)(rc.y1 - rc.y0) << 16);
        wp->view[lane] = vi;
    }
    wave_lds_fence();
    for (uint32_t j = lane; j < total; j += 64u) {
        uint32_t o = 0;   // the owner, as in walk_wave
        for (uint32_t step = 32; step; step >>= 1)
            if (wp->start[o + step] <= j) o += step;
        RasterTri t;
        uint32_t rect, pkey;
        get_piece(wp, ar, o, t, rect, pkey);
        const int tw = (int)(wp->size[o] & 0xFFFFu), th = (int)(wp->size[o] >> 16);
        const int q0 = VIS_CAP * (int)(j - wp->start[o] + 1);
        vis_span<T>(ar, view_at<BATCH>(ka, BATCH ? wp->view[o] : 0u), t, (int)(rect & 0xFFFFu), (int)(rect >> 16), tw, q0,
                    imin(q0 + VIS_CAP, tw * th), pkey, 1.0f / (float)tw);
    }
}

// INSIDE: the host's bound put the mesh's bounding sphere inside every
// frustum plane (ka.skip_clip), so every face classifies as inside and the
// classification is left out (a separate instantiation: a runtime test of the
// flag is compiled to a select, which still computes it).
template <int T, bool BATCH, bool INSIDE, bool SHARE>
__global__ __launch_bounds__(256, BATCH && SHARE ? 6 : 8) void k_vis(KArgs ka, Arena ar) {
    if (ar.counters[CNT_ERROR]) return;
    const uint32_t g = face_slot(ka);
    bool act = g < ka.total_faces;
    uint32_t vi = 0, s = 0, face = 0;
    if constexpr (BATCH) vi = wave_view_of(ka.face_bases, ka.nviews, g, ka.total_faces);
    const ViewDesc& V = view_at<BATCH>(ka, vi);
    DevGroup G;
    vec3 p0, p1, p2;
    if (act) {
        s = g - V.face_base;
        G = group_of<!BATCH>(V, s);
        face = G.first + (s - G.rank_base);
        const uint3 ix = gld(reinterpret_cast<const uint3*>(V.idx), face);
        p0 = load_pos(V.pos, ix.x);
        p1 = load_pos(V.pos, ix.y);
        p2 = load_pos(V.pos, ix.z);
    }
    if constexpr (INSIDE) {
        // faces clearly facing away from the eye are culled before the
        // transform (the pre-test of KArgs::cull_sign; a face within its
        // margin goes on to the exact screen-space test)
        if (ka.cull_sign != 0.0f && act) {
            const vec3 e = make3(ka.cull_eye[0], ka.cull_eye[1], ka.cull_eye[2]);
            const float le = fabsf(e.x) + fabsf(e.y) + fabsf(e.z);
            const vec3 a = p0 - e, b = p1 - p0, c = p2 - p0;
            const float d = ka.cull_sign * dot(a, cross(b, c));
            const float la = fabsf(a.x) + fabsf(a.y) + fabsf(a.z) + le;
            const float lb = fabsf(b.x) + fabsf(b.y) + fabsf(b.z), lc = fabsf(c.x) + fabsf(c.y) + fabsf(c.z);
            if (d < -fmaxf(ka.cull_tau, 1e-3f * la * lb * lc)) act = false;
        }
    }
    bool want_clip = false, small = false, big = false;
    TriRec r;
    RasterTri rt;
    Rect rc{0, 0, 0, 0};
    uint32_t area = 0;
    if (act) {
        const vec4 c0 = V.mvp * make4(p0, 1.0f);
        const vec4 c1 = V.mvp * make4(p1, 1.0f);
        const vec4 c2 = V.mvp * make4(p2, 1.0f);
        int cls = CLS_INSIDE;
        if constexpr (!INSIDE) cls = classify(c0, c1, c2);
        want_clip = cls == CLS_CLIP;
        if (cls == CLS_INSIDE) {
            r = make_rec<INSIDE>(c0, c1, c2, V.W, V.H);
            if (!is_backface(r) && raster_setup<INSIDE>(r, rt)) {
                rc = screen_rect(rt, V.W, V.H);
                if (rc.x0 < rc.x1 && rc.y0 < rc.y1) {
                    area = (uint32_t)((rc.x1 - rc.x0) * (rc.y1 - rc.y0));
                    big = area > (uint32_t)ka.small_footprint;
                    small = !big;
                    if (big) {
                        r.c.y = s * 8u;
                        r.c.z = vi;
                        r.c.w = G.material & REC_MATERIAL_MASK;
                    }
                }
            }
        }
    }
    if constexpr (SHARE) {
        __shared__ VisPieces pieces[4];
        if (__ballot(small && area > VIS_SHARE) == 0ull) {
            if (small) vis_raster_rect<T>(ar, V, rt, rc, s * 8u);
        } else {
            vis_walk_wave<T, BATCH>(pieces + (threadIdx.x >> 6), ka, ar, small, rt, rc, vi, s * 8u);
        }
    } else {
        if (small) vis_raster_rect<T>(ar, V, rt, rc, s * 8u);
    }
    queue_clip(ar, want_clip, g);
    if ((want_clip && ka.skip_clip) || (big && ka.skip_big)) raise_error(ar, ERR_SKIPPED);
    big_append_wave(ar, big, r, area);
}

// ---------------------------------------------------------------------------
// k_clip: the reference's clipper on the faces k_setup queued, one wave per
// face.  A clipped vertex is the 14 vertex floats followed by the clip
// position; the polygon (at most 8 triangles) lives in LDS, twice, and a
// plane that some vertex is not inside of moves it from one copy to the
// other: a lane per vertex takes the plane distances, a lane per triangle
// decides the case and names the sources of its output vertices, then all
// lanes compute the output floats (18 per vertex), every float by the
// reference's operations in its order.  A queue rarely holds more than a few
// thousand faces and each is a long chain of dependent steps, so the latency
// of one face bounds the pass: one lane per face kept both copies in scratch
// (3.4 KB a lane) and walked each float in turn.

constexpr int CLIP_FLOATS = 18;
constexpr int MAX_CLIPPED_VERTS = 24;

struct ClipPoly { float f[MAX_CLIPPED_VERTS][CLIP_FLOATS]; };
// Sources of an output vertex: a copy of vertex src & 255, or (bit 16 set)
// the point at t between it and vertex (src >> 8) & 255.
struct ClipPlan {
    uint32_t src[MAX_CLIPPED_VERTS];
    float t[MAX_CLIPPED_VERTS];
};
constexpr uint32_t CLIP_LERP = 1u << 16;
struct ClipWave {
    ClipPoly poly[2];
    ClipPlan plan;
};

__device__ __forceinline__ vec4 cv_clip(const float* v) { return make4(v[14], v[15], v[16], v[17]); }

// Float c of the vertex at t between a and b (reference pipeline.cpp:243-272).
__device__ __forceinline__ float cv_interp(const float* a, const float* b, float t, int c) {
    const float s = 1.0f - t;
    if (c >= 5 && c < 14) {   // normal, tangent, bitangent: normalized
        const int k = 5 + (c - 5) / 3 * 3;
        const vec3 m = make3(a[k] * s + b[k] * t, a[k + 1] * s + b[k + 1] * t, a[k + 2] * s + b[k + 2] * t);
        return (a[c] * s + b[c] * t) * (1.0f / sqrtf(dot(m, m)));
    }
    if (c == 3 || c == 4) {   // uv: perspective-correct
        const float w0 = a[17], w1 = b[17];
        const float u = (a[c] * w0) * s + (b[c] * w1) * t;
        const float iw = w0 * s + w1 * t;
        return u / iw;
    }
    return a[c] * s + b[c] * t;   // position, clip position
}

__device__ __forceinline__ float edge_t(float din, float dout) {
    float denom = din - dout;
    return (fabsf(denom) < 1e-7f) ? 0.5f : (din / denom);
}

// One plane (reference pipeline.cpp:196-228, 302-370): the polygon of
// `count` vertices in w->poly[cur] against `plane`.  Returns the new vertex
// count; cur names the copy that holds it.  All 64 lanes call it.
__device__ __forceinline__ int clip_plane_wave(ClipWave* w, int& cur, int count, int plane) {
    const int lane = (int)__lane_id();
    const float d = lane < count ? plane_dist(cv_clip(w->poly[cur].f[lane]), plane) : 0.0f;
    // every vertex inside: every triangle passes through unchanged
    if (__ballot(lane < count && !(d >= 0.f)) == 0ull) return count;
    const int ntri = count / 3, v = 3 * (lane < ntri ? lane : 0);
    float d0 = __shfl(d, v), d1 = __shfl(d, v + 1), d2 = __shfl(d, v + 2);
    int a = v, b = v + 1, c = v + 2, r = 0;
    if (d0 >= 0.f && d1 >= 0.f && d2 >= 0.f) {
        r = 1;   // unchanged
    } else if (!(d0 < 0.f && d1 < 0.f && d2 < 0.f)) {
        const bool in0 = d0 >= 0.f, in1 = d1 >= 0.f, in2 = d2 >= 0.f;
        if (in1 && !in0) {
            a = v + 1; b = v + 2; c = v;
            const float t = d0; d0 = d1; d1 = d2; d2 = t;
        } else if (in2 && !in1) {
            a = v + 2; b = v; c = v + 1;
            const float t = d2; d2 = d1; d1 = d0; d0 = t;
        }
        r = d1 >= 0.f ? 3 : 2;   // two triangles, or one cut off
    }
    if (lane >= ntri) r = 0;
    // output positions in triangle order; a triangle whose vertices no longer
    // fit the 24 is dropped, a later smaller one may still fit
    int n = 0, at = 0;
    bool fits = false;
    for (int i = 0; i < ntri; ++i) {
        const int ri = __builtin_amdgcn_readlane(r, i);
        const int need = ri == 0 ? 0 : (ri == 3 ? 6 : 3);
        const bool ok = n + need <= MAX_CLIPPED_VERTS;
        if (lane == i) {
            at = n;
            fits = ok;
        }
        if (ok) n += need;
    }
    if (fits && r) {
        uint32_t* src = w->plan.src + at;
        float* tt = w->plan.t + at;
        const uint32_t ac = (uint32_t)a | ((uint32_t)c << 8) | CLIP_LERP;
        src[0] = (uint32_t)a;
        if (r == 1) {
            src[1] = (uint32_t)b;
            src[2] = (uint32_t)c;
        } else if (r == 2) {
            src[1] = (uint32_t)a | ((uint32_t)b << 8) | CLIP_LERP;
            tt[1] = edge_t(d0, d1);
            src[2] = ac;
            tt[2] = edge_t(d0, d2);
        } else {
            const uint32_t bc = (uint32_t)b | ((uint32_t)c << 8) | CLIP_LERP;
            const float tb = edge_t(d1, d2);
            src[1] = (uint32_t)b;
            src[2] = bc;
            tt[2] = tb;
            src[3] = (uint32_t)a;
            src[4] = bc;
            tt[4] = tb;
            src[5] = ac;
            tt[5] = edge_t(d0, d2);
        }
    }
    wave_lds_fence();
    const ClipPoly& in = w->poly[cur];
    ClipPoly& out = w->poly[cur ^ 1];
    for (int i = lane; i < n * CLIP_FLOATS; i += 64) {
        const int ov = i / CLIP_FLOATS, c2 = i % CLIP_FLOATS;
        const uint32_t src = w->plan.src[ov];
        const float* p = in.f[src & 255u];
        out.f[ov][c2] = (src & CLIP_LERP) ? cv_interp(p, in.f[(src >> 8) & 255u], w->plan.t[ov], c2) : p[c2];
    }
    wave_lds_fence();
    cur ^= 1;
    return n;
}

// One lane's edge setup and rectangle as every lane of the wave sees it.
__device__ __forceinline__ RasterTri bcast_tri(const RasterTri& t, int lane) {
    RasterTri r;
    uint32_t w[sizeof(RasterTri) / 4];
    __builtin_memcpy(w, &t, sizeof(RasterTri));
    for (int i = 0; i < (int)(sizeof(RasterTri) / 4); ++i) w[i] = __builtin_amdgcn_readlane(w[i], lane);
    __builtin_memcpy(&r, w, sizeof(RasterTri));
    return r;
}

// Waves per workgroup and workgroups of the clipper: 4,096 waves, which the
// queues of the measured scenes (hundreds to a few ten thousand faces) keep
// busy for a handful of faces each.
constexpr int CLIP_WAVES = 4;
constexpr int CLIP_BLOCKS = 1024;

template <int T, bool BATCH, bool VIS>
__global__ __launch_bounds__(64 * CLIP_WAVES) void k_clip(KArgs ka, Arena ar) {
    __shared__ ClipWave lds[CLIP_WAVES];
    if (ar.counters[CNT_ERROR]) return;
    const int lane = (int)__lane_id();
    // the sub-queues' entries, one sub-queue per lane, then the shared ones
    const uint32_t cap = ar.clip_sub_cap;
    const uint32_t have = cap ? (uint32_t)imin((int)ar.clip_next[lane * POOL_STRIDE], (int)cap) : 0u;
    const uint32_t upto = wave_incl_scan(have), in_subs = __shfl(upto, 63);
    const uint32_t n = in_subs + (uint32_t)imin((int)ar.counters[CNT_CLIP_FACES], (int)ar.cap_clip_faces);
    ClipWave* w = lds + (threadIdx.x >> 6);
    // the same queue entry for the whole wave
    for (uint32_t q = __builtin_amdgcn_readfirstlane(blockIdx.x * CLIP_WAVES + (threadIdx.x >> 6)); q < n;
         q += gridDim.x * CLIP_WAVES) {
        uint32_t entry = CLIP_SUBS * cap + (q - in_subs);
        if (q < in_subs) {
            const int sub = __popcll(__ballot(upto <= q));
            entry = (uint32_t)sub * cap + q - (__shfl(upto, sub) - __shfl(have, sub));
        }
        entry = __builtin_amdgcn_readfirstlane(entry);
        const uint32_t g = __builtin_amdgcn_readfirstlane(ar.clip_faces[entry]);
        uint32_t vi = 0;
        if constexpr (BATCH) vi = wave_find_le(ka.face_bases, ka.nviews, g);
        const ViewDesc& V = view_at<BATCH>(ka, vi);
        const uint32_t s = g - V.face_base;
        const DevGroup G = group_of<!BATCH>(V, s);
        const uint32_t face = G.first + (s - G.rank_base);
        int cur = 0;
        wave_lds_fence();   // the previous face's reads of the polygon are done
        if (lane < 3 * 14) {
            const uint32_t vtx = gld(V.idx, 3 * (size_t)face + (size_t)(lane / 14));
            w->poly[0].f[lane / 14][lane % 14] = gld(reinterpret_cast<const float*>(V.verts), 14 * (size_t)vtx + (size_t)(lane % 14));
        }
        if (lane < 3) {
            const uint32_t vtx = gld(V.idx, 3 * (size_t)face + (size_t)lane);
            const vec4 c = V.mvp * make4(load_pos(V.pos, vtx), 1.0f);
            float* f = w->poly[0].f[lane];
            f[14] = c.x; f[15] = c.y; f[16] = c.z; f[17] = c.w;
        }
        wave_lds_fence();
        int count = 3;
        for (int plane = 0; plane < 6 && count; ++plane) count = clip_plane_wave(w, cur, count, plane);
        const uint32_t ntri = (uint32_t)(count / 3);
        if (ntri == 0) continue;
        // one or two pieces (all but the faces across several planes) of a
        // sub-queue's entry go to its own two records, the others to records
        // that one counter hands out
        uint32_t base = 2u * entry;
        if (ntri > 2u || entry >= CLIP_SUBS * cap) {
            if (lane == 0) base = 2u * CLIP_SUBS * cap + atomicAdd(&ar.counters[CNT_CLIP_RECS], ntri);
            base = __builtin_amdgcn_readfirstlane(base);
        }
        if (base + ntri > ar.cap_clip_recs) {
            if (lane == 0) set_error(ar, ERR_CLIP_RECS, CNT_NEED_CLIP_RECS, base + ntri);
            continue;
        }
        // one lane per triangle: cull, setup, record
        bool on = false;
        TriRec r;
        RasterTri rt;
        Rect rc{0, 0, 0, 0};
        if (lane < (int)ntri) {
            const float(*f)[CLIP_FLOATS] = w->poly[cur].f + 3 * lane;
            r = make_rec(cv_clip(f[0]), cv_clip(f[1]), cv_clip(f[2]), V.W, V.H);
            if (!is_backface(r) && raster_setup(r, rt)) {
                rc = screen_rect(rt, V.W, V.H);
                on = rc.x0 < rc.x1 && rc.y0 < rc.y1;
            }
            if (on) {
                r.c.y = s * 8u + (uint32_t)lane;
                r.c.z = vi;
                r.c.w = G.material & REC_MATERIAL_MASK;
                ar.clip_rec[base + lane] = r;
            }
        }
        const unsigned long long live = __ballot(on);
        float* dst = reinterpret_cast<float*>(ar.clip_verts + 3 * (size_t)base);
        for (int i = lane; i < count * 14; i += 64) {
            const int v = i / 14;
            if ((live >> (v / 3)) & 1ull) dst[i] = w->poly[cur].f[v][i % 14];
        }
        if constexpr (VIS) {
            const uint32_t area = on ? (uint32_t)((rc.x1 - rc.x0) * (rc.y1 - rc.y0)) : 0u;
            const bool big = area > (uint32_t)ka.small_footprint;
            unsigned long long* vk = ar.vkeys + V.pix_base;
            for (unsigned long long m = __ballot(on && !big); m; m &= m - 1ull) {
                const int j = __ffsll((long long)m) - 1;
                const RasterTri t = bcast_tri(rt, j);
                const Rect tc = screen_rect(t, V.W, V.H);
                const uint32_t tw = (uint32_t)(tc.x1 - tc.x0), np = tw * (uint32_t)(tc.y1 - tc.y0);
                bool any = false;
                for (uint32_t p = (uint32_t)lane; p < np; p += 64u) {
                    const int px = tc.x0 + (int)(p % tw), py = tc.y0 + (int)(p / tw);
                    float al, be, ga, z;
                    if (cover(t, px, py, al, be, ga, z) && z < INFINITY) {
                        atomicMin(&vk[(size_t)py * (size_t)V.W + (size_t)px], depth_key(z, s * 8u + (uint32_t)j));
                        any = true;
                    }
                }
                if (__ballot(any)) flag_bins_wave<T>(ar, V, tc);
            }
            big_append_wave(ar, big, r, area);
            if (lane == 0) ar.clip_base[g] = base;
        } else {
            emit_bins_wave<T>(ar, V, on, rc, REF_CLIP | (base + (uint32_t)lane));
            if (lane == 0) {
                TriRec m;
                m.a = make_float4(0, 0, 0, 0);
                m.b = make_float4(0, 0, 0, 0);
                m.c = make_uint4(0u, s * 8u, base, REC_CLIPPED | (G.material & REC_MATERIAL_MASK));
                ar.rec[g] = m;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// k_raster: one workgroup per bin.


__device__ __forceinline__ const TriRec& rec_of(const Arena& ar, uint32_t ref) {
    return (ref & REF_CLIP) ? ar.clip_rec[ref & ~REF_CLIP] : ar.rec[ref];
}

// Vertex stage of the winner's three corners, then its fragment stage
// (reference tiled_pipeline.cpp:185-212 vertex, 564-575 fragment).  Clipped
// pieces take their corners from the clip records' vertices.
// um: the material every face of the view uses, held in scalar registers
// (a single-group mesh), or null: the record's material is loaded.
template <class S>
__device__ __forceinline__ vec4 shade_at(const ViewDesc& V, const Arena& ar, uint32_t material, uint32_t prim,
                                         bool clipped, uint32_t slot, uint32_t i0, uint32_t i1, uint32_t i2,
                                         vec3 bar, const DevMaterial* um = nullptr) {
    ShadeCtx c;
    c.u = &V.u;
    DevMaterial mat;
    if (um) mat = *um;
    else mat = gld(V.materials, material & REC_MATERIAL_MASK);
    c.m = &mat;
    c.face_colors = V.face_colors;
    c.prim = prim;
    typename S::Var var[3];
    if constexpr (sizeof(typename S::Var) > 1) {
        if (clipped) {
            for (int k = 0; k < 3; ++k) var[k] = S::vs(ar.clip_verts[3 * (size_t)slot + k], V.u);
        } else if (V.vary) {
            const typename S::Var* vy = static_cast<const typename S::Var*>(V.vary);
            var[0] = gld(vy, i0);
            var[1] = gld(vy, i1);
            var[2] = gld(vy, i2);
        } else {
            var[0] = S::vs(gld(V.verts, i0), V.u);
            var[1] = S::vs(gld(V.verts, i1), V.u);
            var[2] = S::vs(gld(V.verts, i2), V.u);
        }
    }
    return S::fs(bar, var, c);
}

template <class S>
__device__ __forceinline__ vec4 shade_winner(const ViewDesc& V, const Arena& ar, const TriRec& r, uint32_t slot,
                                            bool clipped, uint32_t rank, uint3 ix, vec3 bar, const DevMaterial* um = nullptr) {
    uint32_t prim = r.c.z;
    if (clipped) {
        const DevGroup G = group_of<false>(V, rank);
        prim = G.first + (rank - G.rank_base);
    }
    return shade_at<S>(V, ar, r.c.w, prim, clipped, slot, ix.x, ix.y, ix.z, bar, um);
}

// A clear that a draw absorbs (its values; on = false: none).
struct ClearSpec {
    bool on;
    uint32_t bgra;
    float depth;
};

__device__ __forceinline__ void clear_pixel(const ViewDesc& V, size_t pix, const ClearSpec& cs) {
    gst(V.color, pix, cs.bgra);
    gst(V.depth, pix, cs.depth);
    if (V.ids) gst(V.ids, pix, 0xFFFFFFFFu);
}

// Pixel p (row-major) of the bin at (ox, oy), if it lies on the screen.
template <int T>
__device__ __forceinline__ void clear_bin_pixel(const ViewDesc& V, int ox, int oy, int p, const ClearSpec& cs) {
    const int px = ox + (p % T), py = oy + (p / T);
    if (px < V.W && py < V.H) clear_pixel(V, (size_t)py * (size_t)V.W + (size_t)px, cs);
}

// Pixels p0, p0 + step, ... of a bin without keys, when the draw absorbs a
// clear.
template <int T>
__device__ __forceinline__ void clear_bin(const ViewDesc& V, int ox, int oy, const ClearSpec& cs, int p0, int step) {
    for (int p = p0; p < T * T; p += step) clear_bin_pixel<T>(V, ox, oy, p, cs);
}

// known: the depth plane is known to hold known_depth here (a clear written
// just before the draw); else it is loaded.
template <class S>
__device__ __forceinline__ void resolve_pixel(const ViewDesc& V, const Arena& ar, unsigned long long k, int px, int py,
                                              bool known, float known_depth, const ClearSpec& cs, const DevMaterial* um) {
    const uint32_t key = (uint32_t)k;
    const uint32_t rank = key >> 3, j = key & 7u;
    // the framebuffer's depth is under way with the record, the corners'
    // indices during the edge setup
    const size_t pix = (size_t)py * (size_t)V.W + (size_t)px;
    float dfb = known_depth;
    if (!known) dfb = gld(V.depth, pix);
    TriRec r = ar.rec[V.face_base + rank];
    bool clipped = false;
    uint32_t slot = 0;
    uint3 ix = make_uint3(0u, 0u, 0u);
    if (r.c.w & REC_CLIPPED) {
        clipped = true;
        slot = r.c.z + j;
        r = ar.clip_rec[slot];
    } else if constexpr (sizeof(typename S::Var) > 1) {
        ix = gld(reinterpret_cast<const uint3*>(V.idx), r.c.z);
    }
    RasterTri rt;
    raster_setup(r, rt);
    float al, be, ga, z;
    cover(rt, px, py, al, be, ga, z);
    if (!(z < dfb)) {   // reference mergeTileResults: strict less
        if (cs.on) clear_pixel(V, pix, cs);
        return;
    }
    const vec4 col = shade_winner<S>(V, ar, r, slot, clipped, rank, ix, make3(al, be, ga), um);
    gst_nt(V.depth, pix, z);
    gst_nt(V.color, pix, pack_bgra(col));
    if (V.ids) gst_nt(V.ids, pix, key);
}

template <int T, int NT, class S>
// The bin's covered pixels are listed first (plist, count in *ncov, which
// starts at zero), so that every wave shades covered pixels only: a bin on
// a silhouette takes fewer shading rounds than one pass over its rows.
__device__ __forceinline__ void resolve_tile(const ViewDesc& V, const Arena& ar, const unsigned long long* keys,
                                             int ox, int oy, bool known, float known_depth, const ClearSpec& cs,
                                             uint16_t* plist, uint32_t* ncov) {
    static_assert((T * T) % 64 == 0 && NT % 64 == 0, "every wave makes the same number of passes");
    for (int p = threadIdx.x; p < T * T; p += NT) {
        const bool cov = keys[p] != EMPTY_KEY;
        const uint32_t slot = wave_append(ncov, cov);
        if (cov) plist[slot] = (uint16_t)p;
        else if (cs.on) clear_bin_pixel<T>(V, ox, oy, p, cs);
    }
    __syncthreads();
    const uint32_t n = *ncov;
    if (V.ngroups == 1) {
        // one material for the whole view: its fields (texture pointers
        // among them) in scalar registers, loaded once
        const DevMaterial um = wave_uniform(gld(V.materials, V.g0.material & REC_MATERIAL_MASK));
        for (uint32_t i = threadIdx.x; i < n; i += NT) {
            const int p = plist[i];
            resolve_pixel<S>(V, ar, keys[p], ox + (p % T), oy + (p / T), known, known_depth, cs, &um);
        }
    } else {
        for (uint32_t i = threadIdx.x; i < n; i += NT) {
            const int p = plist[i];
            resolve_pixel<S>(V, ar, keys[p], ox + (p % T), oy + (p / T), known, known_depth, cs, nullptr);
        }
    }
}

// Shader functor of a shader kind.
template <int SK> struct ShaderOf;
template <> struct ShaderOf<SHADER_FLAT> { using type = FlatShader; };
template <> struct ShaderOf<SHADER_PHONG> { using type = PhongShader; };
template <> struct ShaderOf<SHADER_PBR> { using type = PBRShader; };
template <> struct ShaderOf<SHADER_GOURAUD> { using type = GouraudShader; };
template <> struct ShaderOf<SHADER_PHONG_POINT> { using type = PhongPointShader; };
template <> struct ShaderOf<SHADER_FLAT_COLOR> { using type = FlatColorShader; };

template <int T, int NT, int SK>
__device__ __forceinline__ void resolve_tile_kind(const ViewDesc& V, const Arena& ar, const unsigned long long* keys,
                                                  int ox, int oy, bool kn, float kd, const ClearSpec& cs, uint16_t* pl,
                                                  uint32_t* nc) {
    if constexpr (SK >= 0) {
        resolve_tile<T, NT, typename ShaderOf<SK>::type>(V, ar, keys, ox, oy, kn, kd, cs, pl, nc);
    } else {
        switch (V.u.kind) {
        case SHADER_FLAT: resolve_tile<T, NT, FlatShader>(V, ar, keys, ox, oy, kn, kd, cs, pl, nc); break;
        case SHADER_PHONG: resolve_tile<T, NT, PhongShader>(V, ar, keys, ox, oy, kn, kd, cs, pl, nc); break;
        case SHADER_PBR: resolve_tile<T, NT, PBRShader>(V, ar, keys, ox, oy, kn, kd, cs, pl, nc); break;
        case SHADER_GOURAUD: resolve_tile<T, NT, GouraudShader>(V, ar, keys, ox, oy, kn, kd, cs, pl, nc); break;
        case SHADER_PHONG_POINT: resolve_tile<T, NT, PhongPointShader>(V, ar, keys, ox, oy, kn, kd, cs, pl, nc); break;
        default: resolve_tile<T, NT, FlatColorShader>(V, ar, keys, ox, oy, kn, kd, cs, pl, nc); break;
        }
    }
}

// ---------------------------------------------------------------------------
// Coverage of a bin's triangles.  One lane per triangle walking its pixel
// rectangle (bbox within the bin) leaves most lanes idle while the wave waits
// for its largest rectangle: on the 256-view batch the rectangles average 11.5
// pixels but a wave's largest is far bigger, and 42% of the lane slots did
// work.  So the walks are capped and shared.  The cap weighs idle lanes
// against the pieces' own cost: a search, then the edge setup from LDS or from
// the record again (below).

// Pixels [q0, q1) of the rectangle [x0, x0 + w) x [y0, ...) (bin coordinates)
// in row-major order; every covered pixel takes the minimum of its key.
// A bin of up to 16 px lies in one of the reference's 16-pixel tile columns, so
// the rectangle's pixels share one anchor, whose edge products are taken once
// (the 4M-triangle soup's k_raster 194 -> 184 us).  At 32 px the walk would
// have to be split at the columns' border, which cost the batch's kernel 3 %.
template <int T>
__device__ __forceinline__ void walk_span(const RasterTri& rt, int x0, int y0, int w, int q0, int q1, uint32_t key,
                                          unsigned long long* keys, int ox, int oy, float inv_w) {
    // row of q0 = floor(q0 / w): q0 < 2^16 and w <= 32, so (q0 + 0.5) / w is
    // at least 1/64 from an integer and its rounded product within 2^-7 of it
    const int dy = q0 == 0 ? 0 : (int)(((float)q0 + 0.5f) * inv_w);
    if constexpr (T <= 16) {
        const int lx = x0 + (q0 - dy * w), ly = y0 + dy;
        const int sx = imax(ox & ~15, rt.fx0);
        const float sxc = (float)sx + 0.5f;
        const float a0 = rt.a0 * sxc, a1 = rt.a1 * sxc, a2 = rt.a2 * sxc;
        int d = ox + lx - sx, at = ly * T + lx;
        const int d1 = ox + x0 + w - sx;
        float pyc = (float)(oy + ly) + 0.5f;   // halves below 2^23: adding 1 is exact
        for (int q = q0; q < q1; ++q) {
            float z;
            if (cover_from(rt, a0, a1, a2, d, pyc, z)) atomicMin(&keys[at], depth_key(z, key));
            ++at;
            if (++d == d1) {
                keep_branch();
                d -= w;
                at += T - w;
                pyc += 1.0f;
            }
        }
    } else {
        int px = x0 + ox + (q0 - dy * w), py = y0 + oy + dy;
        const int x1 = x0 + ox + w;
        for (int q = q0; q < q1; ++q) {
            float al, be, ga, z;
            if (cover(rt, px, py, al, be, ga, z) && z < INFINITY)
                atomicMin(&keys[(py - oy) * T + (px - ox)], depth_key(z, key));
            if (++px == x1) {
                px -= w;
                ++py;
            }
        }
    }
}

// A wave's triangles whose rectangles outlast the cap, for the
// pieces: per lane what a walker needs of its triangle, and the first piece
// of each lane in the wave's numbering.  Two layouts:
//   WalkPieces  the edge setup itself, rectangle and key (17 words a lane);
//   WalkRefs    the bin entry's record reference and the rectangle (3 words):
//               the walker loads the record again and repeats the edge setup
//               (the same operations on the same bits), for a raster kernel
//               whose occupancy its LDS would otherwise bound.
struct WalkRefs {
    uint32_t ref[64];
    uint32_t rect[64];
    uint32_t start[64];
};
// rect: x0 | y0 << 8 | w << 16 | h << 24, in bin coordinates
//
// Pixels per piece.  k_raster in us with 4, 8 and 12: a 150k soup at 16 px
// 20.6, 22.2, 25.0 and 12 PBR objects 17.3, 18.4, 20.2 with the edge setup in
// LDS; with references the 1M-triangle frame at 16 px 43.7, 41.5, - and 40
// mixed views at 32 px 218, 215, 202.
template <int T, class P> constexpr int kWalkCap = T == 32 ? 8 : 4;
template <int T> constexpr int kWalkCap<T, WalkRefs> = T == 32 ? 12 : 8;

__device__ __forceinline__ void put_piece(WalkRefs* wp, uint32_t lane, const RasterTri&, uint32_t ref, uint32_t rect,
                                          uint32_t) {
    wp->ref[lane] = ref;
    wp->rect[lane] = rect;
}
__device__ __forceinline__ void get_piece(const WalkRefs* wp, const Arena& ar, uint32_t o, RasterTri& t, uint32_t& rect,
                                          uint32_t& key) {
    const TriRec r = rec_of(ar, wp->ref[o]);
    raster_setup(r, t);
    rect = wp->rect[o];
    key = r.c.y;
}

// All 64 lanes call it with their own triangle (w = h = 0 for none); ref is
// its bin entry's record reference, (x0, y0, w, h) its rectangle in bin
// coordinates.
template <int T, class P>
__device__ __forceinline__ void walk_wave(P* wp, const Arena& ar, const RasterTri& rt, uint32_t ref, int x0, int y0,
                                          int w, int h, uint32_t key, unsigned long long* keys, int ox, int oy) {
    constexpr int CAP = kWalkCap<T, P>;
    const int fp = w * h;
    walk_span<T>(rt, x0, y0, w, 0, imin(fp, CAP), key, keys, ox, oy, 0.0f);
    const uint32_t pieces = fp > CAP ? (uint32_t)(fp - 1) / CAP : 0u;
    const uint32_t incl = wave_incl_scan(pieces);
    const uint32_t total = __shfl(incl, 63);
    if (total == 0) return;
    const uint32_t lane = __lane_id();
    wp->start[lane] = incl - pieces;
    if (pieces)
        put_piece(wp, lane, rt, ref, (uint32_t)x0 | ((uint32_t)y0 << 8) | ((uint32_t)w << 16) | ((uint32_t)h << 24),
                  key);
    wave_lds_fence();
    for (uint32_t j = lane; j < total; j += 64u) {
        // owner: the last lane whose pieces start at or before j (a lane
        // without pieces shares its start with the next lane that has some)
        uint32_t o = 0;
        for (uint32_t step = 32; step; step >>= 1)
            if (wp->start[o + step] <= j) o += step;
        RasterTri t;
        uint32_t rect, pkey;
        get_piece(wp, ar, o, t, rect, pkey);
        const int rx = (int)(rect & 255u), ry = (int)((rect >> 8) & 255u);
        const int rw = (int)((rect >> 16) & 255u), rh = (int)(rect >> 24);
        const int q0 = CAP * (int)(j - wp->start[o] + 1);
        walk_span<T>(t, rx, ry, rw, q0, imin(q0 + CAP, rw * rh), pkey, keys, ox, oy, 1.0f / (float)rw);
    }
}

// The point-light raster kernel takes the compact layout, which with its
// launch bound (raster_min_waves) lets five waves share a SIMD instead of
// four; the other kinds keep the walkers' loads in LDS.
template <int SK> struct PiecesOf { using type = WalkPieces; };
template <> struct PiecesOf<SHADER_PHONG_POINT> { using type = WalkRefs; };

template <bool BATCH>
__device__ __forceinline__ const ViewDesc& bin_view(const KArgs& ka, const ViewDesc* sview) {
    if constexpr (BATCH) return *sview;
    else return ka.one;
}

// The entry a lane takes first.  Entries go to the waves in turn, so that a
// bin with fewer entries than the workgroup has lanes keeps every wave at work.
template <int NT>
__device__ __forceinline__ uint32_t bin_lane() { return (threadIdx.x & 63u) * (NT / 64) + (threadIdx.x >> 6); }

// ref: the lane's first entry, if that lies in the bin's first level.
// sview (batches): the bin's view is copied into LDS once per bin, so that
// every per-pixel read of its uniforms and pointers is an LDS read.
template <int T, int NT, bool BATCH, int SK>
__device__ __forceinline__ void raster_bin(const KArgs& ka, const Arena& ar, uint32_t t, uint32_t n, uint32_t ref,
                                           unsigned long long* keys, uint32_t& ncov, uint16_t* plist, ViewDesc* sview,
                                           typename PiecesOf<SK>::type* pieces) {
    if constexpr (BATCH) {
        const uint32_t vi = ka.tile_views[t];
        const uint32_t* src = reinterpret_cast<const uint32_t*>(ka.table + vi);
        for (uint32_t i = threadIdx.x; i < sizeof(ViewDesc) / 4; i += NT)
            reinterpret_cast<uint32_t*>(sview)[i] = gld(src, i);
    }
    for (int p = threadIdx.x; p < T * T; p += NT) keys[p] = EMPTY_KEY;
    if (threadIdx.x == 0) ncov = 0;
    __syncthreads();
    const ViewDesc& V = bin_view<BATCH>(ka, sview);
    const uint32_t local = t - V.tile_base;
    const int ox = (int)(local % (uint32_t)V.tiles_x) * T, oy = (int)(local / (uint32_t)V.tiles_x) * T;
    const int ex = imin(ox + T, V.W), ey = imin(oy + T, V.H);
    // every wave has read n: the count is consumed, leave it zero for the next frame
    if (threadIdx.x == 0) ar.tile_count[count_word(t)] = 0;

    typename PiecesOf<SK>::type* wp = pieces + (threadIdx.x >> 6);
    uint32_t next = bin_lane<NT>();
    if ((next >> ar.bin0_shift) != 0u && next < n) ref = bin_get(ar, t, next);
    for (uint32_t b0 = 0; b0 < n; b0 += NT) {
        const uint32_t i = next, mine = ref;
        RasterTri rt;
        int x0 = 0, y0 = 0, w = 0, h = 0;
        uint32_t key = 0;
        TriRec r;
        if (i < n) r = rec_of(ar, mine);
        next += NT;
        if (next < n) ref = bin_get(ar, t, next);   // arrives during the walk
        if (i < n) {
            if (raster_setup(r, rt)) {
                x0 = imax(ox, rt.fx0);
                y0 = imax(oy, rt.fy0);
                w = imin(ex, rt.cx1) - x0;
                h = imin(ey, rt.cy1) - y0;
                if (w <= 0 || h <= 0) w = h = 0;
                key = r.c.y;
            }
        }
        walk_wave<T>(wp, ar, rt, mine, x0 - ox, y0 - oy, w, h, key, keys, ox, oy);
        wave_lds_fence();   // the pieces are read before the next entries' are written
    }
    __syncthreads();

    // every entry has been read: leave the chunk table empty as well
    if (threadIdx.x > 0 && threadIdx.x <= bin_slot(ar.bin0_shift, n - 1).level) ar.bin_chunks[(size_t)t * BIN_LEVELS + threadIdx.x] = 0;

    // a batch's clear is a pass of its own before the frame (k_clear_views)
    const ClearSpec cs{!BATCH && ka.clear != 0, ka.clear_bgra, ka.clear_depth};
    resolve_tile_kind<T, NT, SK>(V, ar, keys, ox, oy, cs.on || (BATCH && ka.depth_is_clear != 0), ka.clear_depth, cs,
                                 plist, &ncov);
}

// One workgroup per bin; an empty bin's leaves after one load, or after
// writing the clear that a plain draw absorbs (ka.clear: a pass of its own
// took 6 us of a 1080p frame, and as long again to start; the 256-view batch,
// mostly empty bins, keeps its streaming pass).  Workgroups
// are dispatched to the 8 XCDs round-robin, so block ids are permuted to give
// an XCD runs of XCD_RUN neighbouring bins, which share triangles, vertices
// and texels in its L2; short runs, because the bins of a frame are not
// equally full (one run per XCD of a small frame's bins put its whole object
// on one XCD).  SK >= 0: built for one shader kind (see k_resolve).
constexpr uint32_t NUM_XCD = 8;
constexpr uint32_t XCD_RUN = 4;

// The bin of a workgroup, and the workgroups that cover n bins.
__device__ __forceinline__ uint32_t bin_of_block(uint32_t b) {
    const uint32_t x = b % NUM_XCD, j = b / NUM_XCD;
    return (j / XCD_RUN * NUM_XCD + x) * XCD_RUN + j % XCD_RUN;
}
static uint32_t bin_blocks(uint32_t n) {
    const uint32_t round = NUM_XCD * XCD_RUN;
    return (n + round - 1) / round * round;
}
// A launch holds fewer than 2^32 threads: more bins go in several.
constexpr uint32_t LAUNCH_BINS = 1u << 23;
static_assert(LAUNCH_BINS % (NUM_XCD * XCD_RUN) == 0, "whole rounds");

// Register bounds per shader kind (waves per SIMD the registers allow; the
// LDS of a 128-thread block at 32 px bins, 19.9 KB with the full walk
// pieces, allows four).  At most 80 VGPRs for the kinds that fit without
// spilling.  The point-light kind at five waves (at most 96 VGPRs, 8
// spilled) with the compact walk pieces (12.7 KB of LDS): the 256-view
// batch's k_raster 1.224 -> 1.192 ms; the compact pieces alone cost
// 0.04 ms and slowed the flat-colour soup by 11 %, so the other kinds keep
// the full ones.  Phong and PBR take the registers they need (held to 80,
// the point-light kind had spilled 22 VGPRs and run 1.68 against 1.38 ms).
constexpr int raster_min_waves(int sk) {
    return (sk == SHADER_FLAT || sk == SHADER_GOURAUD || sk == SHADER_FLAT_COLOR) ? 6
           : sk == SHADER_PHONG_POINT                                            ? 5
                                                                                 : 1;
}

template <int T, int NT, bool BATCH, int SK>
__global__ __launch_bounds__(NT, raster_min_waves(SK)) void k_raster(KArgs ka, Arena ar) {
    __shared__ unsigned long long keys[T * T];
    __shared__ uint16_t plist[T * T];
    __shared__ uint32_t ncov;
    __shared__ ViewDesc sview[1];
    __shared__ typename PiecesOf<SK>::type pieces[NT / 64];
    // A bin that few others share the chip with is a chain of trips to memory,
    // up to 0.9 us each for what another XCD wrote: the error word, the count
    // and the lanes' first entries leave together (as the framebuffer's depth
    // does with the record in resolve_pixel, and the indices during the edge
    // setup).  512 flat faces at 256x256: 9.1 -> 8.4 us with the launch; twelve
    // PBR draws at 1241x719: 17.5 -> 16.8 each; 40 mixed views: 202 -> 193.
    const uint32_t t = ka.first_bin + bin_of_block(blockIdx.x), error = ar.counters[CNT_ERROR];
    uint32_t count = 0, ref = 0;
    if (t < ka.total_tiles) {
        count = ar.tile_count[count_word(t)];
        const uint32_t i = bin_lane<NT>();
        if ((i >> ar.bin0_shift) == 0u) ref = ar.bins[((size_t)t << ar.bin0_shift) + i];
    }
    const bool failed = error != 0u;
    const bool clear = !BATCH && ka.clear != 0;
    if (failed && !clear) return;
    if (blockIdx.x == 0 && !failed) {
        // the per-frame counters were last needed by k_clip
        reset_clip_counters(ar);
        for (uint32_t i = threadIdx.x; i <= POOL_SUBS; i += NT) ar.pool_next[i * POOL_STRIDE] = 0;
    }
    if (t >= ka.total_tiles) return;
    const uint32_t n = failed ? 0u : count;
    if (n == 0u) {
        // an empty bin, or a failed frame: only the clear, if the draw absorbs
        // one, as a separate clear pass would have
        if (clear) {
            const ViewDesc& V = ka.one;
            const int tx = (int)(t % (uint32_t)V.tiles_x), ty = (int)(t / (uint32_t)V.tiles_x);
            clear_bin<T>(V, tx * T, ty * T, ClearSpec{true, ka.clear_bgra, ka.clear_depth}, (int)threadIdx.x, NT);
        }
        return;
    }
    raster_bin<T, NT, BATCH, SK>(ka, ar, t, n, ref, keys, ncov, plist, sview, pieces);
}

// ---------------------------------------------------------------------------
// k_big: visibility mode, the work items of large triangles.  One wave per
// item: BIG_CHUNK consecutive pixels (row-major) of the triangle's screen
// rectangle, four per lane.

template <int T, bool BATCH>
__global__ __launch_bounds__(256) void k_big(KArgs ka, Arena ar) {
    if (ar.counters[CNT_ERROR]) return;
    const unsigned long long c = *big_counter(ar);
    const uint32_t nitems = imin((int)(uint32_t)c, (int)ar.cap_big_items);
    const uint32_t nrecs = imin((int)(uint32_t)(c >> 32), (int)ar.cap_big_recs);
    const uint32_t lane = __lane_id();
    const uint32_t nw = gridDim.x * 4u;
    for (uint32_t it = (blockIdx.x * 256u + threadIdx.x) >> 6; it < nitems; it += nw) {
        const uint32_t ri = wave_find_le(ar.big_start, nrecs, it);
        const TriRec r = ar.big_rec[ri];
        uint32_t vi = 0;
        if constexpr (BATCH) vi = r.c.z;
        const ViewDesc& V = view_at<BATCH>(ka, vi);
        RasterTri rt;
        raster_setup(r, rt);
        const Rect rc = screen_rect(rt, V.W, V.H);
        const uint32_t w = (uint32_t)(rc.x1 - rc.x0);
        const uint32_t np = w * (uint32_t)(rc.y1 - rc.y0);
        const uint32_t p0 = (it - ar.big_start[ri]) * BIG_CHUNK;
        const uint32_t p1 = p0 + BIG_CHUNK < np ? p0 + BIG_CHUNK : np;
        unsigned long long* vk = ar.vkeys + V.pix_base;
        const uint32_t key = r.c.y;
        for (uint32_t p = p0 + lane; p < p1; p += 64u) {
            const int px = rc.x0 + (int)(p % w), py = rc.y0 + (int)(p / w);
            float al, be, ga, z;
            if (cover(rt, px, py, al, be, ga, z) && z < INFINITY) {
                atomicMin(&vk[(size_t)py * (size_t)V.W + (size_t)px], depth_key(z, key));
                ar.tile_count[V.tile_base + (uint32_t)((py / T) * V.tiles_x + px / T)] = 1u;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// k_resolve: visibility mode's last stage.  A wave or a workgroup per bin; bins
// without keys are skipped at once.  Every pixel with a key: recompute the winner's
// setup from its face (or read its clipped piece), depth-test against the
// framebuffer (strict less, reference mergeTileResults), shade, store, and
// leave the key empty for the next frame.

// Shades the winner of key k at (px, py) if it passes the depth test
// against dfb (the framebuffer's depth, or the depth of a clear the draw
// absorbs): returns whether it did, with its depth and packed colour.
// VARY: the view may carry the batch's vertex-stage outputs (V.vary); false
// for plain draws, whose views never do.
// INSIDE: the draw's faces all lie inside the frustum (the host's bound).
template <class S, bool VARY, bool INSIDE>
__device__ __forceinline__ bool shade_vis_pixel(const ViewDesc& V, const Arena& ar, unsigned long long k, int px,
                                                int py, float dfb, float& z, uint32_t& bgra) {
    const uint32_t key = (uint32_t)k;
    const uint32_t s = key >> 3, j = key & 7u;
    const DevGroup G = group_of<!VARY>(V, s);
    const uint32_t face = G.first + (s - G.rank_base);
    const uint3 ix = gld(reinterpret_cast<const uint3*>(V.idx), face);
    const uint32_t i0 = ix.x, i1 = ix.y, i2 = ix.z;
    // the shaders' vertex stage reads the whole vertex; its first three
    // floats are the position (the packed copy setup read holds the same bits)
    constexpr bool kVerts = sizeof(typename S::Var) > 1;
    Vertex56 v0, v1, v2;
    vec3 p0, p1, p2;
    if (kVerts && !(VARY && V.vary)) {
        v0 = gld(V.verts, i0);
        v1 = gld(V.verts, i1);
        v2 = gld(V.verts, i2);
        p0 = make3(v0.px, v0.py, v0.pz);
        p1 = make3(v1.px, v1.py, v1.pz);
        p2 = make3(v2.px, v2.py, v2.pz);
    } else {
        p0 = load_pos(V.pos, i0);
        p1 = load_pos(V.pos, i1);
        p2 = load_pos(V.pos, i2);
    }
    const vec4 c0 = V.mvp * make4(p0, 1.0f), c1 = V.mvp * make4(p1, 1.0f), c2 = V.mvp * make4(p2, 1.0f);
    TriRec r;
    bool clipped = false;
    uint32_t slot = 0;
    if (!INSIDE && classify(c0, c1, c2) == CLS_CLIP) {
        clipped = true;
        slot = ar.clip_base[V.face_base + s] + j;   // written by k_clip
        r = ar.clip_rec[slot];
    } else {
        r = make_rec<INSIDE>(c0, c1, c2, V.W, V.H);
    }
    RasterTri rt;
    raster_setup<INSIDE>(r, rt);
    float al, be, ga;
    cover(rt, px, py, al, be, ga, z);
    if (!(z < dfb)) return false;   // reference mergeTileResults: strict less
    ShadeCtx c;
    c.u = &V.u;
    const DevMaterial mat = gld(V.materials, G.material & REC_MATERIAL_MASK);
    c.m = &mat;
    c.face_colors = V.face_colors;
    c.prim = face;
    typename S::Var var[3];
    if constexpr (kVerts) {
        if (clipped) {
            for (int q = 0; q < 3; ++q) var[q] = S::vs(ar.clip_verts[3 * (size_t)slot + q], V.u);
        } else if (VARY && V.vary) {
            const typename S::Var* vy = static_cast<const typename S::Var*>(V.vary);
            var[0] = gld(vy, i0);
            var[1] = gld(vy, i1);
            var[2] = gld(vy, i2);
        } else {
            var[0] = S::vs(v0, V.u);
            var[1] = S::vs(v1, V.u);
            var[2] = S::vs(v2, V.u);
        }
    }
    bgra = pack_bgra(S::fs(make3(al, be, ga), var, c));
    return true;
}

// Returns whether the winner passed the depth test against dfb and was
// written.
// VARY, INSIDE: as for shade_vis_pixel and k_shade.
template <class S, bool VARY, bool INSIDE>
__device__ __forceinline__ bool resolve_vis_pixel(const ViewDesc& V, const Arena& ar, unsigned long long k, int px,
                                                  int py, size_t pix, float dfb) {
    float z;
    uint32_t bgra;
    if (!shade_vis_pixel<S, VARY, INSIDE>(V, ar, k, px, py, dfb, z, bgra)) return false;
    gst(V.depth, pix, z);
    gst(V.color, pix, bgra);
    if (V.ids) gst(V.ids, pix, (uint32_t)k);
    return true;
}

// Pixels p0, p0 + step, ... of the bin at (ox, oy), row-major.
template <int T, class S, bool VARY, bool INSIDE>
__device__ __forceinline__ void resolve_vis_tile(const ViewDesc& V, const Arena& ar, int ox, int oy,
                                                 const ClearSpec& cs, int p0, int step) {
    unsigned long long* vk = ar.vkeys + V.pix_base;
    for (int p = p0; p < T * T; p += step) {
        const int px = ox + (p % T), py = oy + (p / T);
        if (px >= V.W || py >= V.H) continue;
        const size_t pix = (size_t)py * (size_t)V.W + (size_t)px;
        const unsigned long long k = vk[pix];
        bool drawn = false;
        if (k != EMPTY_KEY) {
            vk[pix] = EMPTY_KEY;
            drawn = resolve_vis_pixel<S, VARY, INSIDE>(V, ar, k, px, py, pix, cs.on ? cs.depth : gld(V.depth, pix));
        }
        if (!drawn && cs.on) clear_pixel(V, pix, cs);
    }
}

template <int T, int SK, bool VARY, bool INSIDE>
__device__ __forceinline__ void resolve_vis_tile_kind(const ViewDesc& V, const Arena& ar, int ox, int oy,
                                                      const ClearSpec& cs, int p0, int step) {
    if constexpr (SK >= 0) {
        resolve_vis_tile<T, typename ShaderOf<SK>::type, VARY, INSIDE>(V, ar, ox, oy, cs, p0, step);
    } else {
        switch (V.u.kind) {
        case SHADER_FLAT: resolve_vis_tile<T, FlatShader, VARY, INSIDE>(V, ar, ox, oy, cs, p0, step); break;
        case SHADER_PHONG: resolve_vis_tile<T, PhongShader, VARY, INSIDE>(V, ar, ox, oy, cs, p0, step); break;
        case SHADER_PBR: resolve_vis_tile<T, PBRShader, VARY, INSIDE>(V, ar, ox, oy, cs, p0, step); break;
        case SHADER_GOURAUD: resolve_vis_tile<T, GouraudShader, VARY, INSIDE>(V, ar, ox, oy, cs, p0, step); break;
        case SHADER_PHONG_POINT: resolve_vis_tile<T, PhongPointShader, VARY, INSIDE>(V, ar, ox, oy, cs, p0, step); break;
        default: resolve_vis_tile<T, FlatColorShader, VARY, INSIDE>(V, ar, ox, oy, cs, p0, step); break;
        }
    }
}

// Bins of 8 px: one wave per bin (four per workgroup, grid-stride over the
// bins), so they cost no workgroup dispatch of their own and need no barrier.
// Larger bins: one workgroup each, in k_raster's order, whose runs of
// neighbouring bins write whole cache lines of a row from one XCD (a 16 px
// bin's row is 64 bytes, half a line), and which leaves before the barrier
// where the bin has no keys.  Against bins in launch order and a barrier in
// every workgroup, at 1080p: 7-9 -> 4.8 us without keys, 11-14 -> 8.3 with a
// clear to write, 2,000 Phong faces over it 14.3 -> 9.6.  Four flags per
// workgroup instead of one: 5.9 us empty, but full bins then share one.  SK >= 0
// builds the kernel for that shader kind alone (every view uses it), so its
// register budget is that shader's and not the largest of all six; SK = -1
// picks the shader per bin.
//
// ka.clear: the framebuffers' clear (a plain draw's pending clear, a batch's
// or a server batch's clear, the same values for every view) is written here
// instead of by a pass of its own: every bin is visited, a pixel no winner
// is written to takes the clear values, and winners are depth-tested
// against the clear depth without reading the framebuffer.  If the frame
// failed (an arena overflow), only the clear is written, as a separate
// clear pass would have.
// INSIDE (plain draws only): every face lies inside the frustum
// (ka.skip_clip), so the winners' classification is left out.  Only a
// batch's views carry vertex-stage outputs (VARY = BATCH).
template <int T, bool BATCH, int SK, bool INSIDE = false>
__global__ __launch_bounds__(256) void k_resolve(KArgs ka, Arena ar) {
    // the bin's flag leaves with the error word (as in k_raster)
    const uint32_t t = ka.first_bin + bin_of_block(blockIdx.x), error = ar.counters[CNT_ERROR];
    uint32_t flag = 0;
    if (T > 8 && t < ka.total_tiles) flag = ar.tile_count[t];
    const bool failed = error != 0u;
    const ClearSpec cs{ka.clear != 0, ka.clear_bgra, ka.clear_depth};
    if (failed && !cs.on) return;
    if (!failed && blockIdx.x == 0) {
        // the per-frame counters of this mode were last needed by k_big
        reset_clip_counters(ar);
        if (threadIdx.x == 0) *big_counter(ar) = 0ull;
    }
    if constexpr (T == 8) {
        // one wave per bin
        const uint32_t nw = gridDim.x * 4u;
        for (uint32_t t = (blockIdx.x * 256u + threadIdx.x) >> 6; t < ka.total_tiles; t += nw) {
            // the same word for the whole wave; the branch waits for the
            // load, so every lane has read the flag before lane 0 clears it
            const bool keys = !failed && ar.tile_count[t] != 0u;
            if (!keys && !cs.on) continue;
            if (keys && __lane_id() == 0) ar.tile_count[t] = 0u;
            uint32_t vi = 0;
            if constexpr (BATCH) vi = ka.tile_views[t];
            const ViewDesc& V = view_at<BATCH>(ka, vi);
            const uint32_t local = t - V.tile_base;
            const int ox = (int)(local % (uint32_t)V.tiles_x) * T, oy = (int)(local / (uint32_t)V.tiles_x) * T;
            if (keys) resolve_vis_tile_kind<T, SK, BATCH, INSIDE>(V, ar, ox, oy, cs, (int)__lane_id(), 64);
            else clear_bin<T>(V, ox, oy, cs, (int)__lane_id(), 64);
        }
    } else {
        // one workgroup (four waves, a pixel or more per thread) per bin
        if (t >= ka.total_tiles) return;
        const bool keys = flag != 0u && !failed;
        if (!keys && !cs.on) return;
        uint32_t vi = 0;
        if constexpr (BATCH) vi = ka.tile_views[t];
        const ViewDesc& V = view_at<BATCH>(ka, vi);
        const uint32_t local = t - V.tile_base;
        const int ox = (int)(local % (uint32_t)V.tiles_x) * T, oy = (int)(local / (uint32_t)V.tiles_x) * T;
        if (!keys) {
            clear_bin<T>(V, ox, oy, cs, (int)threadIdx.x, 256);
            return;
        }
        // every wave has read the flag before thread 0 clears it
        __syncthreads();
        if (threadIdx.x == 0) ar.tile_count[t] = 0u;
        resolve_vis_tile_kind<T, SK, BATCH, INSIDE>(V, ar, ox, oy, cs, (int)threadIdx.x, 256);
    }
}

// ---------------------------------------------------------------------------
// The resolve of a plain draw that absorbs a clear, in two passes, so that
// the shading need not wait for an earlier draw into the same framebuffer:
// winners are tested against the clear depth, never against the planes.
// k_shade shades every winner into its own key slot (depth bits << 32 |
// packed colour; a winner behind the clear empties the slot); k_finish, the
// only pass that touches the framebuffer, writes every pixel from its slot
// or the clear and leaves the slots and bin flags empty.  For a framebuffer
// with an id plane (IDS) the slot keeps the winner's key in its low word
// and the colour goes to the arena's colour slots (vcol).

// INSIDE: as for k_vis, every face lies inside the frustum (ka.skip_clip),
// so the winners' classification is left out.  That instantiation without an
// id plane asks for seven waves per SIMD (at most 72 VGPRs, which the Phong
// kinds fit without spilling and PBR would not): the 1080p frame's k_shade
// 17.2 -> 16.3 us against six waves; eight spilled and ran 19.2 us.
template <int T, int SK, bool IDS, bool INSIDE = false>
__global__ __launch_bounds__(256, (INSIDE && !IDS && SK != SHADER_PBR) ? 7 : 1) void k_shade(KArgs ka, Arena ar) {
    using S = typename ShaderOf<SK>::type;
    if (ar.counters[CNT_ERROR]) return;
    if (blockIdx.x == 0) {
        // the per-frame counters of this mode were last needed by k_big
        reset_clip_counters(ar);
        if (threadIdx.x == 0) *big_counter(ar) = 0ull;
    }
    const ViewDesc& V = ka.one;
    unsigned long long* vk = ar.vkeys + V.pix_base;
    // one wave per 64 pixels of a bin (SUB waves per bin), one pixel per
    // lane: a bin edge of 16 or 32 gives the pass as many waves as one of 8
    constexpr uint32_t SUB = (uint32_t)(T * T + 63) / 64;
    const uint32_t nunits = ka.total_tiles * SUB;
    const int lane = (int)__lane_id();
    const uint32_t nw = gridDim.x * 4u;
    for (uint32_t u = (blockIdx.x * 256u + threadIdx.x) >> 6; u < nunits; u += nw) {
        const uint32_t t = u / SUB;
        if (ar.tile_count[t] == 0u) continue;
        const int p = (int)(u % SUB) * 64 + lane;   // row-major within the bin
        const uint32_t local = t - V.tile_base;
        const int px = (int)(local % (uint32_t)V.tiles_x) * T + (p % T);
        const int py = (int)(local / (uint32_t)V.tiles_x) * T + (p / T);
        if (p >= T * T || px >= V.W || py >= V.H) continue;
        const size_t pix = (size_t)py * (size_t)V.W + (size_t)px;
        const unsigned long long k = vk[pix];
        if (k == EMPTY_KEY) continue;
        float z;
        uint32_t bgra;
        const bool drawn = shade_vis_pixel<S, false, INSIDE>(V, ar, k, px, py, ka.clear_depth, z, bgra);
        vk[pix] = drawn ? ((unsigned long long)__float_as_uint(z) << 32) | (IDS ? (uint32_t)k : bgra) : EMPTY_KEY;
        if (IDS && drawn) ar.vcol[V.pix_base + pix] = bgra;
    }
}

// One wave per strip of 64 pixels by one bin row (64 / T bins side by
// side), one lane per column: each row of the strip is one 256-byte store
// per plane.  A slot is read only in bins that had keys.
template <int T, bool IDS>
__global__ __launch_bounds__(256) void k_finish(KArgs ka, Arena ar) {
    static_assert(64 % T == 0, "a strip holds whole bins");
    const bool failed = ar.counters[CNT_ERROR] != 0u;
    const ViewDesc& V = ka.one;
    const ClearSpec cs{true, ka.clear_bgra, ka.clear_depth};
    unsigned long long* vk = ar.vkeys + V.pix_base;
    const uint32_t lane = __lane_id();
    const uint32_t sx_n = ((uint32_t)V.W + 63u) / 64u;
    const uint32_t nstrips = sx_n * (uint32_t)V.tiles_y;
    const uint32_t nw = gridDim.x * 4u;
    for (uint32_t st = (blockIdx.x * 256u + threadIdx.x) >> 6; st < nstrips; st += nw) {
        const uint32_t sx = st % sx_n, by = st / sx_n;
        const int px = (int)(sx * 64u + lane);
        const bool in_x = px < V.W;
        const uint32_t t = V.tile_base + by * (uint32_t)V.tiles_x + (uint32_t)px / (uint32_t)T;
        const bool keys = !failed && in_x && ar.tile_count[t] != 0u;
        const int rows = imin(T, V.H - (int)by * T);
        const size_t pix0 = (size_t)by * T * (size_t)V.W + (size_t)px;
        constexpr int RB = T < 8 ? T : 8;   // rows whose slots are loaded together
        for (int r0 = 0; r0 < rows; r0 += RB) {
            // all slot loads of RB rows first: the stores below may alias
            // them for the compiler, which would otherwise wait for each
            unsigned long long sl[RB];
#pragma unroll
            for (int r = 0; r < RB; ++r)
                sl[r] = keys && r0 + r < rows ? vk[pix0 + (size_t)(r0 + r) * V.W] : EMPTY_KEY;
            if (!in_x) continue;
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                if (r0 + r >= rows) break;
                const size_t pix = pix0 + (size_t)(r0 + r) * V.W;
                if (sl[r] != EMPTY_KEY) {
                    vk[pix] = EMPTY_KEY;
                    V.color[pix] = IDS ? ar.vcol[V.pix_base + pix] : (uint32_t)sl[r];
                    V.depth[pix] = __uint_as_float((uint32_t)(sl[r] >> 32));
                    if (IDS) V.ids[pix] = (uint32_t)sl[r];
                } else {
                    clear_pixel(V, pix, cs);
                }
            }
        }
        // every lane of a bin read its flag before the loop's loads returned
        if (keys && (uint32_t)px % (uint32_t)T == 0u) ar.tile_count[t] = 0u;
    }
}

// k_finish for a width that is a multiple of 4 (every row then starts
// 16-byte aligned in the 256-byte aligned planes): one wave per strip of
// 64 pixels by one bin row, each lane four adjacent pixels of every fourth
// row, 16-byte loads and stores (each store instruction covers four rows
// of 256 contiguous bytes).
template <int T, bool IDS>
__global__ __launch_bounds__(256) void k_finish4(KArgs ka, Arena ar) {
    static_assert(64 % T == 0 && T % 4 == 0, "a strip holds whole bins, a lane's pixels one bin");
    constexpr int RL = T / 4;   // rows per lane
    const bool failed = ar.counters[CNT_ERROR] != 0u;
    const ViewDesc& V = ka.one;
    unsigned long long* vk = ar.vkeys + V.pix_base;
    const uint4 cv = make_uint4(ka.clear_bgra, ka.clear_bgra, ka.clear_bgra, ka.clear_bgra);
    const float4 dv = make_float4(ka.clear_depth, ka.clear_depth, ka.clear_depth, ka.clear_depth);
    const ulonglong2 ev2 = make_ulonglong2(EMPTY_KEY, EMPTY_KEY);
    const uint32_t lane = __lane_id();
    const uint32_t cg = lane & 15u, rg = lane >> 4;
    const uint32_t sx_n = ((uint32_t)V.W + 63u) / 64u;
    const uint32_t nstrips = sx_n * (uint32_t)V.tiles_y;
    const uint32_t nw = gridDim.x * 4u;
    for (uint32_t st = (blockIdx.x * 256u + threadIdx.x) >> 6; st < nstrips; st += nw) {
        const uint32_t sx = st % sx_n, by = st / sx_n;
        const int px = (int)(sx * 64u + 4u * cg);
        if (px >= V.W) continue;   // W % 4 == 0: the lane's four pixels are all inside or all outside
        const uint32_t t = V.tile_base + by * (uint32_t)V.tiles_x + (uint32_t)px / (uint32_t)T;
        const bool keys = !failed && ar.tile_count[t] != 0u;
        const int y0 = (int)by * T;
        // all slot loads first: the stores below may alias them for the
        // compiler, which would otherwise wait for each
        ulonglong2 a[RL], b[RL];
#pragma unroll
        for (int k = 0; k < RL; ++k) {
            a[k] = b[k] = ev2;
            const int py = y0 + (int)rg + 4 * k;
            if (keys && py < V.H) {
                const ulonglong2* q = reinterpret_cast<const ulonglong2*>(vk + (size_t)py * V.W + (size_t)px);
                a[k] = q[0];
                b[k] = q[1];
            }
        }
#pragma unroll
        for (int k = 0; k < RL; ++k) {
            const int py = y0 + (int)rg + 4 * k;
            if (py >= V.H) break;
            const size_t pix = (size_t)py * V.W + (size_t)px;
            const unsigned long long s0 = a[k].x, s1 = a[k].y, s2 = b[k].x, s3 = b[k].y;
            uint4 c = cv;
            float4 d = dv;
            uint4 id = make_uint4(~0u, ~0u, ~0u, ~0u);
            if ((s0 & s1 & s2 & s3) != EMPTY_KEY) {
                if (s0 != EMPTY_KEY) { c.x = (uint32_t)s0; d.x = __uint_as_float((uint32_t)(s0 >> 32)); }
                if (s1 != EMPTY_KEY) { c.y = (uint32_t)s1; d.y = __uint_as_float((uint32_t)(s1 >> 32)); }
                if (s2 != EMPTY_KEY) { c.z = (uint32_t)s2; d.z = __uint_as_float((uint32_t)(s2 >> 32)); }
                if (s3 != EMPTY_KEY) { c.w = (uint32_t)s3; d.w = __uint_as_float((uint32_t)(s3 >> 32)); }
                if constexpr (IDS) {
                    // the slots hold the winners' keys; their colours are in vcol
                    id = c;
                    const uint4 vc = *reinterpret_cast<const uint4*>(ar.vcol + V.pix_base + pix);
                    c = make_uint4(s0 != EMPTY_KEY ? vc.x : cv.x, s1 != EMPTY_KEY ? vc.y : cv.y,
                                   s2 != EMPTY_KEY ? vc.z : cv.z, s3 != EMPTY_KEY ? vc.w : cv.w);
                    id = make_uint4(s0 != EMPTY_KEY ? id.x : ~0u, s1 != EMPTY_KEY ? id.y : ~0u,
                                    s2 != EMPTY_KEY ? id.z : ~0u, s3 != EMPTY_KEY ? id.w : ~0u);
                }
                ulonglong2* q = reinterpret_cast<ulonglong2*>(vk + pix);
                q[0] = ev2;
                q[1] = ev2;
            }
            typedef unsigned int v4u __attribute__((ext_vector_type(4)));
            gst_nt(reinterpret_cast<v4u*>(V.color + pix), 0, v4u{c.x, c.y, c.z, c.w});
            gst_nt(reinterpret_cast<v4u*>(V.depth + pix), 0,
                   v4u{__float_as_uint(d.x), __float_as_uint(d.y), __float_as_uint(d.z), __float_as_uint(d.w)});
            if constexpr (IDS) gst_nt(reinterpret_cast<v4u*>(V.ids + pix), 0, v4u{id.x, id.y, id.z, id.w});
        }
        // every lane of a bin read its flag before the loop's loads returned
        if (keys && rg == 0u && (uint32_t)px % (uint32_t)T == 0u) ar.tile_count[t] = 0u;
    }
}

// ---------------------------------------------------------------------------
// framebuffer clear (reference framebuffer.cpp:26-42)

// Planes start 256-byte aligned (hipMalloc, or 256-byte aligned offsets in
// a server block), so four pixels go per 16-byte store; the tail is scalar.
__device__ __forceinline__ void clear_planes(uint32_t* color, float* depth, uint32_t* ids, size_t n, uint32_t bgra,
                                             float d, size_t first, size_t stride) {
    const size_t n4 = n / 4;
    // non-temporal 16-byte stores (a cache hint only): a clear streams whole
    // planes, which later passes read back at most once
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    v4u* c4 = reinterpret_cast<v4u*>(color);
    v4u* d4 = reinterpret_cast<v4u*>(depth);
    v4u* i4 = reinterpret_cast<v4u*>(ids);
    const uint32_t du = __float_as_uint(d);
    const v4u cv = {bgra, bgra, bgra, bgra}, dv = {du, du, du, du}, iv = {~0u, ~0u, ~0u, ~0u};
    for (size_t i = first; i < n4; i += stride) {
        __builtin_nontemporal_store(cv, c4 + i);
        __builtin_nontemporal_store(dv, d4 + i);
        if (ids) __builtin_nontemporal_store(iv, i4 + i);
    }
    for (size_t i = 4 * n4 + first; i < n; i += stride) {
        color[i] = bgra;
        depth[i] = d;
        if (ids) ids[i] = 0xFFFFFFFFu;
    }
}

__global__ void k_clear(uint32_t* color, float* depth, uint32_t* ids, size_t n, uint32_t bgra, float d) {
    clear_planes(color, depth, ids, n, bgra, d, blockIdx.x * (size_t)blockDim.x + threadIdx.x,
                 (size_t)gridDim.x * blockDim.x);
}

// Clear of every view of a batch: blockIdx.y picks the view (views
// [view0, view0 + gridDim.y)), the x blocks stride over its pixels.
__global__ void k_clear_views(const ViewDesc* views, uint32_t view0, uint32_t bgra, float d) {
    const ViewDesc& V = views[view0 + blockIdx.y];
    clear_planes(V.color, V.depth, V.ids, (size_t)V.W * (size_t)V.H, bgra, d, blockIdx.x * (size_t)blockDim.x + threadIdx.x,
                 (size_t)gridDim.x * blockDim.x);
}

// ---------------------------------------------------------------------------
// k_vary: the vertex stage of every vertex of every job (a mesh shared by
// views whose vertex stage reads the same uniforms), one lane per vertex;
// the resolve then reads each winner's three outputs instead of running
// the vertex stage per pixel.  The same function on the same inputs, so
// the varyings are bit for bit those the resolve would compute.

template <class S>
__device__ __forceinline__ void vary_one(const VaryJob& j, uint32_t v, const ViewDesc& V) {
    static_cast<typename S::Var*>(j.out)[v] = S::vs(j.verts[v], V.u);
}

__global__ __launch_bounds__(256) void k_vary(const VaryJob* jobs, const uint32_t* firsts, uint32_t njobs,
                                              uint32_t total, const ViewDesc* views) {
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    if (g >= total) return;
    const VaryJob& j = jobs[find_le(firsts, njobs, g)];
    const uint32_t v = g - j.first;
    const ViewDesc& V = views[j.view];
    switch (j.kind) {
    case SHADER_FLAT: vary_one<FlatShader>(j, v, V); break;
    case SHADER_PHONG: vary_one<PhongShader>(j, v, V); break;
    case SHADER_PBR: vary_one<PBRShader>(j, v, V); break;
    case SHADER_GOURAUD: vary_one<GouraudShader>(j, v, V); break;
    case SHADER_PHONG_POINT: vary_one<PhongPointShader>(j, v, V); break;
    default: break;   // FLAT_COLOR: no vertex stage
    }
}

// Bytes of the vertex stage's output per vertex for a shader kind (0: the
// shader has none).
uint32_t vary_bytes(int kind) {
    switch (kind) {
    case SHADER_FLAT: return sizeof(FlatShader::Var);
    case SHADER_PHONG: return sizeof(PhongShader::Var);
    case SHADER_PBR: return sizeof(PBRShader::Var);
    case SHADER_GOURAUD: return sizeof(GouraudShader::Var);
    case SHADER_PHONG_POINT: return sizeof(PhongPointShader::Var);
    default: return 0;
    }
}

// ---------------------------------------------------------------------------
// host-side launch wrappers

// Expects a clean arena (bin counts and per-frame counters zero) and leaves
// it clean.
constexpr int RESOLVE_MAX_BLOCKS = 16384;

// Tool ranges named after the reference's phases (its Tracy zones,
// tiled_pipeline.cpp:173, 264, 268, 273, 283, 312) around each stage's
// launches, for a profiler's marker trace; on when AXR_ROCTX=1 at library
// load.  The stages of a raster mode map onto the phases as in
// kBinnedPhases / kVisPhases (the vertex pass of a batch belongs to the
// reference's raster phase, where its fragment shading runs).
static bool phase_ranges_on() {
    static const bool on = [] {
        const char* v = getenv("AXR_ROCTX");
        return v && v[0] == '1';
    }();
    return on;
}
static const char* const kBinnedPhases[kStages] = {"ClippingAllTriangles", "ClippingAllTriangles", "TilePreparation",
                                                   "BinAllTriangles", "RasterizingTiles", "RasterizingTiles"};
static const char* const kVisPhases[kStages] = {"ClippingAllTriangles", "ClippingAllTriangles", "RasterizingTiles",
                                                "RasterizingTiles", "MergingAllTiles", "RasterizingTiles"};
static thread_local const char* const* t_phases = kBinnedPhases;

// One kernel of stage `stage`.  With kernel timing (ev), the first kernel
// of a stage carries the stage's start event and its last kernel the stop
// event, attached to the dispatches (hipExtLaunchKernel).
template <class... KA, class... A>
static void stage_launch(void (*kern)(KA...), dim3 grid, dim3 block, hipStream_t st, StageEvents* ev, int stage,
                         bool first, bool last, A... args) {
    const bool ranges = phase_ranges_on();
    if (ranges && first) roctxRangePush(t_phases[stage]);
    struct Pop {
        bool on;
        ~Pop() { if (on) roctxRangePop(); }
    } pop{ranges && last};
    if (ev) {
        hipExtLaunchKernelGGL(kern, grid, block, 0, st, first ? ev->start[stage] : nullptr,
                              last ? ev->stop[stage] : nullptr, 0, args...);
        ev->used |= 1u << stage;
    } else {
        hipLaunchKernelGGL(kern, grid, block, 0, st, args...);
    }
}
template <class... KA, class... A>
static void stage_launch1(void (*kern)(KA...), dim3 grid, dim3 block, hipStream_t st, StageEvents* ev, int stage,
                          A... args) {
    stage_launch(kern, grid, block, st, ev, stage, true, true, args...);
}

// A kernel with a workgroup of `threads` per bin, in bin_of_block's order.
static void launch_bins(void (*kern)(KArgs, Arena), uint32_t threads, hipStream_t st, StageEvents* ev, int stage,
                        const KArgs& args, const Arena& ar) {
    KArgs ka = args;
    const uint32_t n = ka.total_tiles;
    do {
        const uint32_t left = n - ka.first_bin, take = left < LAUNCH_BINS ? left : LAUNCH_BINS;
        stage_launch(kern, dim3(bin_blocks(take ? take : 1u)), dim3(threads), st, ev, stage, ka.first_bin == 0u, take == left, ka, ar);
        ka.first_bin += take;
    } while (ka.first_bin < n);
}

static hipError_t fb_wait(hipStream_t st, const FbWait& w) {
    if (w.sig) return hipStreamWaitValue64(st, w.sig, w.value, hipStreamWaitValueGte);
    if (w.ev) return hipStreamWaitEvent(st, w.ev, 0);
    return hipSuccess;
}

// The shader-specialised kernel of ka.shader (-1: the switching one).
template <template <int> class K>
static auto by_shader(int shader) -> decltype(K<-1>::fn) {
    switch (shader) {
    case SHADER_FLAT: return K<SHADER_FLAT>::fn;
    case SHADER_PHONG: return K<SHADER_PHONG>::fn;
    case SHADER_PBR: return K<SHADER_PBR>::fn;
    case SHADER_GOURAUD: return K<SHADER_GOURAUD>::fn;
    case SHADER_PHONG_POINT: return K<SHADER_PHONG_POINT>::fn;
    case SHADER_FLAT_COLOR: return K<SHADER_FLAT_COLOR>::fn;
    default: return K<-1>::fn;
    }
}
template <int T, bool IDS, bool INSIDE> struct ShadeK {
    template <int SK> struct K {
        static constexpr auto fn = &k_shade<T, (SK < 0 ? SHADER_FLAT_COLOR : SK), IDS, INSIDE>;
    };
};
// only a batch's views may differ in their shader kind
template <int T, bool BATCH, bool INSIDE> struct ResolveK {
    template <int SK> struct K {
        static constexpr auto fn = &k_resolve<T, BATCH, (!BATCH && SK < 0 ? SHADER_FLAT_COLOR : SK), INSIDE>;
    };
};
template <int T, int NT, bool BATCH> struct RasterK {
    template <int SK> struct K {
        static constexpr auto fn = &k_raster<T, NT, BATCH, (!BATCH && SK < 0 ? SHADER_FLAT_COLOR : SK)>;
    };
};

// k_shade, then (after the wait) k_finish4 or k_finish: stages 3 and 4.
template <int T, bool IDS>
static hipError_t launch_two_pass(const KArgs& ka, const Arena& ar, hipStream_t st, StageEvents* ev,
                                  const FbWait& wait) {
    const uint64_t units = (uint64_t)ka.total_tiles * (uint64_t)((T * T + 63) / 64);
    const int sb = (int)std::min<uint64_t>(std::max<uint64_t>(1, (units + 3) / 4), RESOLVE_MAX_BLOCKS);
    const auto shade = ka.skip_clip ? by_shader<ShadeK<T, IDS, true>::template K>(ka.shader)
                                    : by_shader<ShadeK<T, IDS, false>::template K>(ka.shader);
    stage_launch1(shade, dim3(sb), dim3(256), st, ev, 3, ka, ar);
    hipError_t e = fb_wait(st, wait);
    if (e != hipSuccess) return e;
    const uint32_t strips = (((uint32_t)ka.one.W + 63u) / 64u) * (uint32_t)ka.one.tiles_y;
    const int fblocks = imax(1, imin((int)((strips + 3) / 4), RESOLVE_MAX_BLOCKS));
    if (ka.one.W % 4 == 0) stage_launch1(k_finish4<T, IDS>, dim3(fblocks), dim3(256), st, ev, 4, ka, ar);
    else stage_launch1(k_finish<T, IDS>, dim3(fblocks), dim3(256), st, ev, 4, ka, ar);
    return hipGetLastError();
}

// At most this many faces go 16 to a wave (2,048 waves, two to a SIMD) instead
// of 64.
constexpr uint32_t FEW_FACES = 32768;

// Workgroups (four waves) of the passes over faces.
static uint32_t face_blocks(const KArgs& ka) {
    const uint32_t per = 4u << ka.face_shift;
    return (uint32_t)(((uint64_t)ka.total_faces + per - 1) / per);
}

// Visibility mode: stage 0 k_vis, 1 k_clip, 2 k_big, then either 4
// k_resolve or (two-pass) 3 k_shade and 4 k_finish.
template <int T, bool BATCH>
static hipError_t launch_vis_t(const KArgs& ka, const Arena& ar, hipStream_t st, StageEvents* ev, const FbWait& wait) {
    t_phases = kVisPhases;
    const uint32_t vis_blocks = face_blocks(ka);
    if (vis_blocks) {
        const bool share = (uint64_t)ka.total_faces * VIS_SHARE <= ka.total_pixels;
        if (!BATCH && ka.skip_clip)
            stage_launch1(share ? &k_vis<T, false, true, true> : &k_vis<T, false, true, false>, dim3(vis_blocks), dim3(256), st,
                          ev, 0, ka, ar);
        else
            stage_launch1(share ? &k_vis<T, BATCH, false, true> : &k_vis<T, BATCH, false, false>, dim3(vis_blocks), dim3(256), st,
                          ev, 0, ka, ar);
    }
    // passes the host showed to have no work are not launched
    if (BATCH || !ka.skip_clip) stage_launch1(k_clip<T, BATCH, true>, dim3(CLIP_BLOCKS), dim3(64 * CLIP_WAVES), st, ev, 1, ka, ar);
    if (BATCH || !ka.skip_big) stage_launch1(k_big<T, BATCH>, dim3(1024), dim3(256), st, ev, 2, ka, ar);
    if (!BATCH && ka.two_pass && ka.clear && ka.shader >= 0 && ka.shader < SHADER_COUNT) {
        // shade at once, write the framebuffer after the earlier draws
        return ka.one.ids ? launch_two_pass<T, true>(ka, ar, st, ev, wait)
                          : launch_two_pass<T, false>(ka, ar, st, ev, wait);
    }
    // the framebuffer pass waits for what other streams were asked to do first
    hipError_t e = fb_wait(st, wait);
    if (e != hipSuccess) return e;
    const auto resolve = (!BATCH && ka.skip_clip) ? by_shader<ResolveK<T, false, true>::template K>(ka.shader)
                                                  : by_shader<ResolveK<T, BATCH, false>::template K>(ka.shader);
    // T = 8: four bins per workgroup; larger bins: one bin per workgroup
    if constexpr (T == 8)
        stage_launch1(resolve, dim3(imax(1, imin((int)((ka.total_tiles + 3) / 4), RESOLVE_MAX_BLOCKS))), dim3(256), st, ev, 4, ka, ar);
    else
        launch_bins(resolve, 256, st, ev, 4, ka, ar);
    return hipGetLastError();
}

// Binned mode: stage 0 k_setup, 1 k_clip, 4 k_raster.
template <int T, int NT, bool BATCH>
static hipError_t launch_frame_t(const KArgs& ka, const Arena& ar, hipStream_t st, StageEvents* ev,
                                 const FbWait& wait) {
    if (ka.mode == RASTER_VISIBILITY) return launch_vis_t<T, BATCH>(ka, ar, st, ev, wait);
    t_phases = kBinnedPhases;
    const uint32_t setup_blocks = face_blocks(ka);
    if (setup_blocks) {
        if (ka.skip_clip) stage_launch1(k_setup<T, BATCH, true>, dim3(setup_blocks), dim3(256), st, ev, 0, ka, ar);
        else stage_launch1(k_setup<T, BATCH>, dim3(setup_blocks), dim3(256), st, ev, 0, ka, ar);
    }
    if (!ka.skip_clip) stage_launch1(k_clip<T, BATCH, false>, dim3(CLIP_BLOCKS), dim3(64 * CLIP_WAVES), st, ev, 1, ka, ar);
    hipError_t e = fb_wait(st, wait);
    if (e != hipSuccess) return e;
    launch_bins(by_shader<RasterK<T, NT, BATCH>::template K>(ka.shader), NT, st, ev, 4, ka, ar);
    return hipGetLastError();
}

// Threads per bin of k_raster: ka.raster_threads, or more.  A bin's pixels
// are shaded by its workgroup alone, and few of a single view's bins hold
// most of its pixels, so bins of 16 or 32 px take 256 threads (a 1M-triangle
// 1080p frame: 97 us at 64, 57 at 128, 39 at 256; a PBR object at 1241x719:
// 37, 24, 18).  Where there is little to shade per pixel (one colour per
// face) or a batch's many views fill the chip, 128 (a 400k-triangle soup at
// 1080p: 49, 42, 59 us; 24 mixed views at 16 px: 130, 82, 99).  A bin of 8 px
// has 64 pixels.
template <int T, bool BATCH>
static hipError_t launch_frame_nt(const KArgs& ka, const Arena& ar, hipStream_t st, StageEvents* ev, const FbWait& w) {
    if constexpr (T == 8) {
        if (ka.raster_threads <= 64) return launch_frame_t<T, 64, BATCH>(ka, ar, st, ev, w);
    }
    const int least = T == 8 || BATCH || ka.shader == SHADER_FLAT_COLOR ? 128 : 256;
    return imax(least, ka.raster_threads) <= 128 ? launch_frame_t<T, 128, BATCH>(ka, ar, st, ev, w)
                                                 : launch_frame_t<T, 256, BATCH>(ka, ar, st, ev, w);
}

template <bool BATCH>
static hipError_t launch_frame_b(const KArgs& ka, const Arena& ar, hipStream_t st, StageEvents* ev, const FbWait& w) {
    switch (ka.tile_size) {
    case 8: return launch_frame_nt<8, BATCH>(ka, ar, st, ev, w);
    case 32: return launch_frame_nt<32, BATCH>(ka, ar, st, ev, w);
    default: return launch_frame_nt<16, BATCH>(ka, ar, st, ev, w);
    }
}

hipError_t launch_frame(const KArgs& args, const Arena& ar, hipStream_t st, StageEvents* ev, const FbWait& wait) {
    KArgs ka = args;
    ka.face_shift = ka.total_faces <= FEW_FACES ? 4 : 6;
    // stage 5: a batch's vertex stage once per vertex of each shared mesh,
    // before the resolve reads it
    if (ka.table && ka.vary_total)
        stage_launch1(k_vary, dim3((ka.vary_total + 255) / 256), dim3(256), st, ev, 5, ka.vary_jobs, ka.vary_firsts,
                      ka.vary_njobs, ka.vary_total, ka.table);
    return ka.table ? launch_frame_b<true>(ka, ar, st, ev, wait) : launch_frame_b<false>(ka, ar, st, ev, wait);
}

hipError_t launch_clear_views(const ViewDesc* views, const uint32_t* pix_bases, uint32_t nviews, uint32_t total,
                              uint32_t bgra, float d, hipStream_t st) {
    (void)pix_bases;
    // about 8 Ki pixels of the average view per block, at most 64 blocks a view
    const uint32_t avg = nviews ? total / nviews : 0;
    const int bx = imax(1, imin(64, (int)((avg + 8191) / 8192)));
    for (uint32_t v0 = 0; v0 < nviews; v0 += 65535u) {
        const uint32_t nv = nviews - v0 < 65535u ? nviews - v0 : 65535u;
        k_clear_views<<<dim3(bx, nv), 256, 0, st>>>(views, v0, bgra, d);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// host waits and read-backs

// After a kernel, hipStreamSynchronize returns 4 us later than the host sees a
// word that the stream's next kernel stored (14.2 against 10.4 us for a 2 us
// kernel, on MI355X).
__global__ void k_done(uint32_t* word, uint32_t seq) {
    if (threadIdx.x == 0) __hip_atomic_store(word, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Planes of a framebuffer into pinned host memory, all in one launch whose
// last workgroup tells the host: bound by the host link (56 GB/s), which
// READ_BLOCKS workgroups fill.  Two planes of 32 KB: 9.5 us against 17.5 for a
// runtime copy each and a stream wait, two of 2 MB 84 against 91; a single
// plane is 0.5 us faster by the runtime copy and stays with it.
constexpr uint32_t READ_BLOCKS = 16;
__global__ __launch_bounds__(256) void k_read(ReadJob job, uint32_t* blocks_done, uint32_t* word, uint32_t seq) {
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    const size_t first = blockIdx.x * 256u + threadIdx.x, stride = gridDim.x * 256u;
    for (int p = 0; p < 3; ++p) {
        if (!job.dst[p]) continue;
        const v4u* src = reinterpret_cast<const v4u*>(job.src[p]);
        v4u* dst = reinterpret_cast<v4u*>(job.dst[p]);
        const size_t n4 = job.words / 4;
        for (size_t i = first; i < n4; i += stride) __builtin_nontemporal_store(src[i], dst + i);
        for (size_t i = 4 * n4 + first; i < job.words; i += stride) job.dst[p][i] = job.src[p][i];
    }
    __threadfence_system();   // this thread's stores before its workgroup counts as done
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(blocks_done, 1u) == gridDim.x - 1u) {
        *blocks_done = 0u;
        __threadfence_system();
        __hip_atomic_store(word, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

hipError_t launch_done(uint32_t* word, uint32_t seq, hipStream_t st) {
    k_done<<<1, 64, 0, st>>>(word, seq);
    return hipGetLastError();
}

hipError_t launch_read(const ReadJob& job, uint32_t* blocks_done, uint32_t* word, uint32_t seq, hipStream_t st) {
    k_read<<<READ_BLOCKS, 256, 0, st>>>(job, blocks_done, word, seq);
    return hipGetLastError();
}

hipError_t launch_prep(const Arena& ar, uint32_t ntiles, hipStream_t st) {
    k_prep<<<imax(1, imin(1024, (int)((ntiles + 255) / 256))), 256, 0, st>>>(ar, ntiles);
    return hipGetLastError();
}

hipError_t launch_clear(uint32_t* color, float* depth, uint32_t* ids, size_t n, uint32_t bgra, float d, hipStream_t st) {
    int blocks = (int)imin(2048, (int)((n / 4 + 255) / 256));
    k_clear<<<imax(1, blocks), 256, 0, st>>>(color, depth, ids, n, bgra, d);
    return hipGetLastError();
}

}  // namespace axr
