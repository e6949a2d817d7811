// grt_traverse.hip -- 3D-DDA traversal of the uniform grid
// with Moller-Trumbore intersection, on gfx950 (wave64).
//
// Reference semantics:
//   clip + DDA set-up   AabbIntersection.cpp:37-63, UniformGridAccStruct.cpp:118-149
//   DDA loop            UniformGridAccStruct.cpp:160-195 (single-axis step,
//                       ties to y then z)
//   cell loop           UniformGridAccStruct.cpp:362-378 (hits bounded by the
//                       current cell's exit)
//   Moller-Trumbore     RayTracing_kernel.cu:56-89 (no determinant epsilon)
//   any hit             shadow_FRAG.glsl:122-245
//
// Data in HBM: rays and hits are structures of arrays (coalesced 4-byte
// lanes); the grid is offsets[m+1] (uint32) plus one 48-byte record per
// reference, trir[k] = {v0.xyz, e1.x}{e1.yz, e2.xy}{e2.z, id, -, -}, stored
// contiguously per cell, so a cell's triangles stream without an index
// indirection.
//
//   k_trace_window        one-level grid, 1..16 lanes per ray (grt_window.h)
//   k_trace_batch_window  the same over the items of a batch
//   k_trace2, _split      two-level grid
#include "grt_launch.h"
#include "grt_mt.h"
#include "grt_window.h"

namespace grt {

// ---------------------------------------------------------------------------
// Ray indexing
// ---------------------------------------------------------------------------

// Slot -> ray: through the ray list when the launch has one (slots beyond
// the list's device-side count are idle), else the image-tile mapping.
__device__ __forceinline__ uint32_t trace_ray(const TraceArgs& a, uint32_t slot, bool& valid)
{
    if (a.list) {
        const uint32_t c = *a.list_count;
        valid = slot < c && slot < a.n;
        return valid ? a.list[slot] : 0u;
    }
    return slot_ray(slot, a.image_width, a.n, valid);
}

// ---------------------------------------------------------------------------
// DDA
// ---------------------------------------------------------------------------
struct Dda {
    int32_t cx, cy, cz;
    int32_t sx, sy, sz;
    int32_t ox, oy, oz;   // out-of-grid limits
    float tx, ty, tz;     // t at the next boundary per axis
    float dtx, dty, dtz;
};

__device__ __forceinline__ bool grid_ok(const DevFrame* __restrict__ fr)
{
    return (fr->status & (kStatusFrameInvalid | kStatusCellsOver | kStatusRefsOver)) == 0;
}

// Ray::update + clipRay + DDA set-up.  False when the ray misses the grid box
// (or its interval is empty).
__device__ __forceinline__ bool dda_setup(const DevFrame* __restrict__ fr, float o0, float o1,
                                          float o2, float d0, float d1, float d2, float tmin,
                                          float tmax, Dda& s)
{
    const float i0 = 1.0f / d0, i1 = 1.0f / d1, i2 = 1.0f / d2;
    float tn = tmin, tf = tmax;
    {
        const float a = (fr->bmin[0] - o0) * i0, b = (fr->bmax[0] - o0) * i0;
        tn = tmax_f(tn, tmin_f(a, b));
        tf = tmin_f(tf, tmax_f(a, b));
    }
    {
        const float a = (fr->bmin[1] - o1) * i1, b = (fr->bmax[1] - o1) * i1;
        tn = tmax_f(tn, tmin_f(a, b));
        tf = tmin_f(tf, tmax_f(a, b));
    }
    {
        const float a = (fr->bmin[2] - o2) * i2, b = (fr->bmax[2] - o2) * i2;
        tn = tmax_f(tn, tmin_f(a, b));
        tf = tmin_f(tf, tmax_f(a, b));
    }
    if (tn > tf)
        return false;
    const float p0 = o0 + d0 * tn, p1 = o1 + d1 * tn, p2 = o2 + d2 * tn;
    s.cx = vox(p0, fr->bmin[0], fr->inv[0], fr->n[0]);
    s.cy = vox(p1, fr->bmin[1], fr->inv[1], fr->n[1]);
    s.cz = vox(p2, fr->bmin[2], fr->inv[2], fr->n[2]);
    const bool n0 = __builtin_signbit(d0), n1 = __builtin_signbit(d1), n2 = __builtin_signbit(d2);
    s.sx = n0 ? -1 : 1;
    s.sy = n1 ? -1 : 1;
    s.sz = n2 ? -1 : 1;
    s.ox = n0 ? -1 : fr->n[0];
    s.oy = n1 ? -1 : fr->n[1];
    s.oz = n2 ? -1 : fr->n[2];
    const float w0 = (float)(s.cx + (n0 ? 0 : 1)) * fr->cell[0] + fr->bmin[0];
    const float w1 = (float)(s.cy + (n1 ? 0 : 1)) * fr->cell[1] + fr->bmin[1];
    const float w2 = (float)(s.cz + (n2 ? 0 : 1)) * fr->cell[2] + fr->bmin[2];
    s.tx = (w0 - o0) * i0;
    s.ty = (w1 - o1) * i1;
    s.tz = (w2 - o2) * i2;
    s.dtx = fabsf(fr->cell[0] * i0);
    s.dty = fabsf(fr->cell[1] * i1);
    s.dtz = fabsf(fr->cell[2] * i2);
    return true;
}

// ---------------------------------------------------------------------------
// One-level grid: windowed walk
// ---------------------------------------------------------------------------

// The DDA of a windowed walk: the current cell's index with one stride per
// axis, and the steps left on each axis before the ray leaves the grid.
struct DdaW {
    uint32_t ci, sx, sy, sz;
    uint32_t rx, ry, rz;
    float tx, ty, tz, dtx, dty, dtz;
};

__device__ __forceinline__ DdaW dda_window(const DevFrame* __restrict__ fr, const Dda& s)
{
    const uint32_t nx = (uint32_t)fr->n[0], ny = (uint32_t)fr->n[1], nxy = nx * ny;
    DdaW w;
    w.ci = (uint32_t)s.cx + nx * ((uint32_t)s.cy + ny * (uint32_t)s.cz);
    w.sx = s.sx < 0 ? ~0u : 1u;
    w.sy = s.sy < 0 ? 0u - nx : nx;
    w.sz = s.sz < 0 ? 0u - nxy : nxy;
    w.rx = (uint32_t)(s.sx < 0 ? s.cx : s.ox - 1 - s.cx);
    w.ry = (uint32_t)(s.sy < 0 ? s.cy : s.oy - 1 - s.cy);
    w.rz = (uint32_t)(s.sz < 0 ? s.cz : s.oz - 1 - s.cz);
    w.tx = s.tx;
    w.ty = s.ty;
    w.tz = s.tz;
    w.dtx = s.dtx;
    w.dty = s.dty;
    w.dtz = s.dtz;
    return w;
}

// One step (dda_step's tie order) when `go`; false when the ray does not go
// on (the state then stays in the grid).
__device__ __forceinline__ bool dda_window_step(DdaW& w, bool go)
{
    const bool ax = w.tx < w.ty && w.tx < w.tz;
    const bool ay = !ax && w.ty < w.tz;
    // values, not lvalues: a conditional over fields would select addresses
    // and send the walk's state to scratch memory
    const uint32_t rx = w.rx, ry = w.ry, rz = w.rz, sx = w.sx, sy = w.sy, sz = w.sz;
    const uint32_t left = ax ? uint32_t(rx) : (ay ? uint32_t(ry) : uint32_t(rz));
    go = go && left != 0;
    const bool mx = go && ax, my = go && ay, mz = go && !ax && !ay;
    const float tx = w.tx + w.dtx, ty = w.ty + w.dty, tz = w.tz + w.dtz;
    w.tx = mx ? tx : w.tx;
    w.ty = my ? ty : w.ty;
    w.tz = mz ? tz : w.tz;
    w.rx -= mx ? 1u : 0u;
    w.ry -= my ? 1u : 0u;
    w.rz -= mz ? 1u : 0u;
    const uint32_t d = ax ? uint32_t(sx) : (ay ? uint32_t(sy) : uint32_t(sz));
    w.ci += go ? d : 0u;
    return go;
}

// Sum over the `lanes`-lane group (every lane of the wave calls it).
__device__ __forceinline__ uint32_t group_sum(uint32_t v, uint32_t lanes)
{
    for (uint32_t o = 1; o < lanes; o <<= 1)
        v += (uint32_t)__shfl_xor((int)v, (int)o, 64);
    return v;
}

// Bound by VALU issue (0.70-0.85 of the cycles) with 51-60 of 64 lanes active
// per instruction; the per-lane loops this replaced ran 10-30 lanes and one
// memory latency per cell and test.  Before and after, us: 512x512 spheres
// (16k triangles) primary 121 -> 51, bounce 238 -> 43; stadium (lambda 128,
// 1280x720) primary 3294 -> 1585, shadow 3100 -> 1739; 1.2 M-slot batch
// 1197 -> 552.
//
// Ray i (valid: the whole group) against one grid, traced by a group of
// `lanes` lanes (1..16, a power of two) in windows of lanes x c cells, c =
// min(S, 16 / lanes), lane j taking the cells from j c on; every lane of the
// wave calls it together.
template <bool ANY, bool COUNT, int S>
__device__ __forceinline__ void trace_window(const DevFrame* __restrict__ fr,
                                             const uint32_t* __restrict__ offsets,
                                             const float4* __restrict__ trir, const RaySoA& rays,
                                             const HitSoA& hits, uint8_t* __restrict__ occluded,
                                             uint32_t* __restrict__ counters, uint32_t lanes,
                                             uint32_t i, bool valid, WaveWin& W)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t j = lane & (lanes - 1u), owner = lane - j;
    const uint32_t c = lanes * S <= 16u ? (uint32_t)S : 16u / lanes, cell0 = j * c;
    float4 ro = make_float4(0.0f, 0.0f, 0.0f, 0.0f), rd = ro;
    DdaW w = {};
    bool walk = false;   // the lane stands on a cell of its ray
    if (valid) {
        ro = make_float4(rays.ox[i], rays.oy[i], rays.oz[i], rays.tmin[i]);
        rd = make_float4(rays.dx[i], rays.dy[i], rays.dz[i], rays.tmax[i]);
        Dda s;
        walk = grid_ok(fr) && dda_setup(fr, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z, ro.w, rd.w, s);
        if (walk)
            w = dda_window(fr, s);
    }
    bool open = valid;   // the ray's result is not written yet
    uint32_t cells = 0, tests = 0;
    if (__ballot(walk) != 0) {
        W.ro[lane] = make_float4(ro.x, ro.y, ro.z, win_lo(ro.w));
        W.rd[lane] = make_float4(rd.x, rd.y, rd.z, ro.w);
        for (uint32_t q = 0; q < cell0; ++q)
            walk = dda_window_step(w, walk && !(tmin_f(tmin_f(w.tx, w.ty), w.tz) > rd.w));
        // The next window's steps and list bounds come before this one's
        // tests, so their latency overlaps the tests.
        WinU<S> nb, ne, nbound;
        uint32_t nvisited;
        const auto next_window = [&]() {
            nvisited = 0;
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)S; ++s) {
                const uint32_t* o = offsets + w.ci;   // in the grid also when the walk is over
                nb[s] = o[0];
                ne[s] = o[1];
                const float ex = tmin_f(tmin_f(w.tx, w.ty), w.tz);
                nbound[s] = __float_as_uint(ANY ? win_end(rd.w, INFINITY)
                                                : win_end(rd.w, ex * kExitScale));
                const bool mine = walk && s < c;
                nvisited += mine ? 1u : 0u;
                const bool on = dda_window_step(w, mine && !(ex > rd.w));
                walk = mine ? on : walk;
            }
            // the other lanes' cells, up to the lane's next window
            for (uint32_t q = c; q < lanes * c; ++q)
                walk = dda_window_step(w, walk && !(tmin_f(tmin_f(w.tx, w.ty), w.tz) > rd.w));
        };
        next_window();
        do {
            const WinU<S> b = nb, bound = nbound;
            WinU<S> n = ne;
            const uint32_t visited = nvisited;
            next_window();
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)S; ++s)
                n[s] = s < visited ? n[s] - b[s] : 0u;
            const unsigned long long key = win_tests<ANY, S>(W, trir, b, n, bound, owner, cell0);
            const bool hit = key != ~0ull;
            uint32_t hs = win_cell(key) - cell0;
            hs = hs < c ? hs : (uint32_t)S;   // S: not one of the lane's cells
            if (COUNT && open) {
                const bool after = hit && win_cell(key) < cell0;
                cells += after ? 0u : (hit && hs < (uint32_t)S) ? hs + 1u : visited;
#pragma unroll
                for (uint32_t s = 0; s < (uint32_t)S; ++s)
                    tests += after              ? 0u
                             : !hit || s < hs   ? n[s]
                             : s == hs          ? (ANY ? win_pos(key) + 1u : n[s])
                                                : 0u;
            }
            if (hit) {
                if (ANY) {
                    if (j == 0)
                        occluded[i] = 1;
                } else if (hs < (uint32_t)S) {
                    const uint64_t k = win_pick<S>(b, hs) + win_pos(key);
                    const float4 A = trir[3ull * k], B = trir[3ull * k + 1], C = trir[3ull * k + 2];
                    const MtPre m = mt_pre(A, B, C, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z);
                    float t, u, v;
                    mt_exact(m, t, u, v);
                    hits.id[i] = (int32_t)__float_as_uint(C.y);
                    hits.t[i] = t;
                    hits.u[i] = u;
                    hits.v[i] = v;
                }
                open = false;
                walk = false;
                nvisited = 0;
            }
        } while (__ballot(nvisited != 0) != 0);
    }
    if (COUNT) {
        const uint32_t sc = group_sum(cells, lanes), st = group_sum(tests, lanes);
        if (valid && j == 0) {
            counters[2ull * i] = sc;
            counters[2ull * i + 1] = st;
        }
    }
    if (open && j == 0) {
        if (ANY) {
            occluded[i] = 0;
        } else {
            hits.id[i] = -1;
            hits.t[i] = INFINITY;
            hits.u[i] = 0.0f;
            hits.v[i] = 0.0f;
        }
    }
}

extern __shared__ WaveWin win_lds[];   // one per wave of the block

template <bool ANY, bool COUNT, int S>
__global__ __launch_bounds__(256) void k_trace_window(TraceArgs a, RaySoA rays, HitSoA hits,
                                                      uint8_t* __restrict__ occluded,
                                                      uint32_t lanes)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    bool valid;
    const uint32_t i = trace_ray(a, t >> __builtin_ctz(lanes), valid);
    trace_window<ANY, COUNT, S>(a.fr, a.offsets, a.trir, rays, hits, occluded, a.counters, lanes, i,
                             valid, win_lds[threadIdx.x >> 6]);
}

// Batched multi-scene traversal: every 64-slot group belongs to one task
// (map[slot / 64]), so each wave runs its task's walk with wave-uniform scene
// data.
template <int S>
__global__ __launch_bounds__(256) void k_trace_batch_window(const BatchTask* __restrict__ tasks,
                                                            const uint32_t* __restrict__ map,
                                                            uint32_t total_slots,
                                                            uint32_t lanes)
{
    const uint32_t slot = (blockIdx.x * blockDim.x + threadIdx.x) >> __builtin_ctz(lanes);
    const uint32_t group = __builtin_amdgcn_readfirstlane(slot >> 6);
    if ((group << 6) >= total_slots)
        return;   // whole waves only: total_slots is a multiple of 64
    const uint32_t task = __builtin_amdgcn_readfirstlane(map[group]);
    const BatchTask& T = tasks[task];
    bool valid;
    const uint32_t i = slot_ray(slot - T.slot_begin, T.image_width, T.n, valid);
    WaveWin& W = win_lds[threadIdx.x >> 6];
    if (T.any)
        trace_window<true, false, S>(T.fr, T.offsets, T.trir, T.rays, T.hits, T.occluded, nullptr,
                                  lanes, i, valid, W);
    else
        trace_window<false, false, S>(T.fr, T.offsets, T.trir, T.rays, T.hits, T.occluded, nullptr,
                                   lanes, i, valid, W);
}

// ---------------------------------------------------------------------------
// Batched multi-scene traversal
// ---------------------------------------------------------------------------

// map[b] = index of the task owning slots [64b, 64b+64).
__global__ __launch_bounds__(256) void k_task_map(const BatchTask* __restrict__ tasks,
                                                  uint32_t* __restrict__ map)
{
    const BatchTask& t = tasks[blockIdx.x];
    const uint32_t b0 = t.slot_begin >> 6, nb = t.slots >> 6;
    for (uint32_t j = threadIdx.x; j < nb; j += blockDim.x)
        map[b0 + j] = blockIdx.x;
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
static uint32_t ray_grid(uint32_t n, uint32_t img_w, uint32_t block)
{
    return (uint32_t)((slot_count(n, img_w) + block - 1) / block);
}

// ---------------------------------------------------------------------------
// Two-level grid: one ray per lane
// ---------------------------------------------------------------------------
//
// The top DDA as in the one-level kernels; a top cell whose record carries a
// sub-grid resolution is walked by a DDA of its own from the point where the
// ray entered the cell (the clipped entry, then each top cell's exit), with
// hits bounded by the sub-cell's exit; other cells test their references
// bounded by the cell's exit.  The first (sub-)cell holding a hit ends a
// closest-hit ray, the first triangle in (tmin, tmax] an any-hit ray.
// Counters: top cells plus sub-cells visited, triangle tests.

// Tests records [b, e) of `rec`: closest (bound) or any.  True when the ray is
// done (a hit in this cell, or an occluder).
template <bool ANY>
__device__ __forceinline__ bool trace2_cell(const float4* __restrict__ rec, uint32_t b,
                                            uint32_t e, float o0, float o1, float o2, float d0,
                                            float d1, float d2, float tmin, float tmax,
                                            float bound, int32_t& id, float& best, float& bu,
                                            float& bv, uint32_t& tests)
{
    return test_records<ANY>(rec, b, e, o0, o1, o2, d0, d1, d2, tmin, tmax, bound, id, best, bu,
                             bv, tests);
}

__device__ __forceinline__ int32_t sub_vox(float val, float bmin, float inv, int32_t r)
{
    float x = (val - bmin) * inv;
    x = x > 0.0f ? x : 0.0f;
    const float hi = (float)(r - 1);
    x = x < hi ? x : hi;
    return (int32_t)x;
}

// Per-ray constants of the two-level walk.
struct Ray2 {
    float o0, o1, o2, d0, d1, d2, i0, i1, i2, tmin, tmax;
    bool n0, n1, n2;
};

// Sub-cell sizes and their reciprocals by resolution, staged in LDS by every
// block of a two-level kernel: sc = tab[16 a + r - 1], 1/sc = tab[48 + 16 a +
// r - 1] (the build evaluates cell_a / r and 1 / that, the frame's own
// operations, once per frame).
__device__ __forceinline__ void stage_sub_tab(const TraceArgs& a, float* tab)
{
    if (threadIdx.x < 96u)
        tab[threadIdx.x] = a.sub_tab[threadIdx.x];
    __syncthreads();
}

// DDA state inside a top cell's sub-grid: current sub-cell (and its index si
// in the sub-cell arrays, which a step along y or z changes by sy or sz; by
// +-1 along x), next boundary crossings and their increments.
struct Sub2 {
    uint32_t si, sy, sz;
    int32_t qx, qy, qz, ox, oy, oz;
    float tx, ty, tz, dtx, dty, dtz;
};

// Entry into the sub-grid of the top cell at s (record rec) at t_enter.
__device__ __forceinline__ void sub_setup(const DevFrame* __restrict__ fr, const float* tab,
                                          const Ray2& r, const Dda& s, uint2 rec, float t_enter,
                                          Sub2& q)
{
    const uint32_t base = rec.x & 0x7fffffffu;
    const int32_t r0 = (int32_t)(rec.y & 255u);
    const int32_t r1 = (int32_t)((rec.y >> 8) & 255u);
    const int32_t r2 = (int32_t)((rec.y >> 16) & 255u);
    const float sb0 = (float)s.cx * fr->cell[0] + fr->bmin[0];
    const float sb1 = (float)s.cy * fr->cell[1] + fr->bmin[1];
    const float sb2 = (float)s.cz * fr->cell[2] + fr->bmin[2];
    const float sc0 = tab[r0 - 1], sc1 = tab[16 + r1 - 1], sc2 = tab[32 + r2 - 1];
    const float si0 = tab[48 + r0 - 1], si1 = tab[64 + r1 - 1], si2 = tab[80 + r2 - 1];
    q.qx = sub_vox(r.o0 + r.d0 * t_enter, sb0, si0, r0);
    q.qy = sub_vox(r.o1 + r.d1 * t_enter, sb1, si1, r1);
    q.qz = sub_vox(r.o2 + r.d2 * t_enter, sb2, si2, r2);
    q.ox = r.n0 ? -1 : r0;
    q.oy = r.n1 ? -1 : r1;
    q.oz = r.n2 ? -1 : r2;
    q.tx = ((float)(q.qx + (r.n0 ? 0 : 1)) * sc0 + sb0 - r.o0) * r.i0;
    q.ty = ((float)(q.qy + (r.n1 ? 0 : 1)) * sc1 + sb1 - r.o1) * r.i1;
    q.tz = ((float)(q.qz + (r.n2 ? 0 : 1)) * sc2 + sb2 - r.o2) * r.i2;
    q.dtx = fabsf(sc0 * r.i0);
    q.dty = fabsf(sc1 * r.i1);
    q.dtz = fabsf(sc2 * r.i2);
    q.si = base + (uint32_t)q.qx +
           (uint32_t)r0 * ((uint32_t)q.qy + (uint32_t)r1 * (uint32_t)q.qz);
    q.sy = r.n1 ? 0u - (uint32_t)r0 : (uint32_t)r0;
    q.sz = r.n2 ? 0u - (uint32_t)(r0 * r1) : (uint32_t)(r0 * r1);
}

// One sub-grid step (the top DDA's tie order); false when it leaves the grid
// (q is then left as it was).  Branch-free: the crossed axis selects which
// coordinate, crossing and index change.
__device__ __forceinline__ bool sub_step(const Ray2& r, Sub2& q)
{
    const bool ax = q.tx < q.ty && q.tx < q.tz;
    const bool ay = !ax && q.ty < q.tz;
    const bool az = !ax && !ay;
    const int32_t dx = r.n0 ? -1 : 1;
    const int32_t qx = ax ? q.qx + dx : q.qx;
    const int32_t qy = ay ? q.qy + (r.n1 ? -1 : 1) : q.qy;
    const int32_t qz = az ? q.qz + (r.n2 ? -1 : 1) : q.qz;
    if ((ax && qx == q.ox) || (ay && qy == q.oy) || (az && qz == q.oz))
        return false;
    q.qx = qx;
    q.qy = qy;
    q.qz = qz;
    const float tx = q.tx + q.dtx, ty = q.ty + q.dty, tz = q.tz + q.dtz;
    q.tx = ax ? tx : q.tx;
    q.ty = ay ? ty : q.ty;
    q.tz = az ? tz : q.tz;
    q.si += ax ? (uint32_t)dx : (ay ? q.sy : q.sz);
    return true;
}

// One non-empty top cell (index ci, coordinates of s, record rec) of the
// two-level walk, entered at t_enter and left at exit_t: its sub-grid from t_enter when it has one and
// the second level is valid, else its own references bounded by exit_t.
// Counts the sub-cells visited and the tests.  True when the walk ends in this
// cell: a hit (closest), an occluder (any, *occ set) or a sub-cell whose exit
// lies beyond tmax.
template <bool ANY>
__device__ __forceinline__ bool top_cell2(const TraceArgs& a, const DevFrame* __restrict__ fr,
                                          const float* tab, bool sub_ok, const Ray2& r,
                                          const Dda& s, uint2 rec, uint32_t ci, float t_enter,
                                          float exit_t, bool& occ, int32_t& id, float& best,
                                          float& bu, float& bv, uint32_t& cells,
                                          uint32_t& tests)
{
    const bool has_sub = (rec.x >> 31) != 0u;
    if (!(sub_ok && has_sub)) {
        // the top cell's own list (also for a sub-grid cell when the second
        // level is not valid)
        const uint32_t kb = has_sub ? a.offsets[ci] : rec.x;
        const uint32_t ke = has_sub ? a.offsets[ci + 1] : rec.y;
        if (trace2_cell<ANY>(a.trir, kb, ke, r.o0, r.o1, r.o2, r.d0, r.d1, r.d2, r.tmin, r.tmax,
                             exit_t * kExitScale, id, best, bu, bv, tests)) {
            occ = ANY;
            return true;
        }
        return false;
    }
    Sub2 q;
    sub_setup(fr, tab, r, s, rec, t_enter, q);
    uint32_t kb = a.sub_offsets[q.si], ke = a.sub_offsets[q.si + 1];
    for (;;) {
        ++cells;
        const float sexit = tmin_f(tmin_f(q.tx, q.ty), q.tz);
        // the next sub-cell and its offsets, loaded before this one's tests
        // (unconditionally: a step out of the sub-grid leaves q.si in place)
        const uint32_t cb = kb, ce = ke;
        const bool more = sub_step(r, q);
        kb = a.sub_offsets[q.si];
        ke = a.sub_offsets[q.si + 1];
        if (trace2_cell<ANY>(a.sub_trir, cb, ce, r.o0, r.o1, r.o2, r.d0, r.d1, r.d2, r.tmin,
                             r.tmax, sexit * kExitScale, id, best, bu, bv, tests)) {
            occ = ANY;
            return true;
        }
        if (sexit > r.tmax || !more)
            return sexit > r.tmax;
    }
}

// Set-up of a two-level ray: constants, the top DDA and the clipped entry.
__device__ __forceinline__ bool ray2_setup(const DevFrame* __restrict__ fr, const RaySoA& rays,
                                           uint32_t i, Ray2& r, Dda& s, float& t_enter)
{
    r.o0 = rays.ox[i];
    r.o1 = rays.oy[i];
    r.o2 = rays.oz[i];
    r.d0 = rays.dx[i];
    r.d1 = rays.dy[i];
    r.d2 = rays.dz[i];
    r.tmin = rays.tmin[i];
    r.tmax = rays.tmax[i];
    if (!(grid_ok(fr) && dda_setup(fr, r.o0, r.o1, r.o2, r.d0, r.d1, r.d2, r.tmin, r.tmax, s)))
        return false;
    r.i0 = 1.0f / r.d0;
    r.i1 = 1.0f / r.d1;
    r.i2 = 1.0f / r.d2;
    // the clipped entry, as dda_setup computes it
    t_enter = r.tmin;
    t_enter = tmax_f(t_enter, tmin_f((fr->bmin[0] - r.o0) * r.i0, (fr->bmax[0] - r.o0) * r.i0));
    t_enter = tmax_f(t_enter, tmin_f((fr->bmin[1] - r.o1) * r.i1, (fr->bmax[1] - r.o1) * r.i1));
    t_enter = tmax_f(t_enter, tmin_f((fr->bmin[2] - r.o2) * r.i2, (fr->bmax[2] - r.o2) * r.i2));
    r.n0 = __builtin_signbit(r.d0);
    r.n1 = __builtin_signbit(r.d1);
    r.n2 = __builtin_signbit(r.d2);
    return true;
}

// The walk over the top grid goes item by item.  An item is a cell of the
// grid; for an empty cell with skip radius rr > 0 it is the cells ahead of it
// within rr on every axis (all empty), left in one step.  Each item's exit is
// its first boundary plane crossed, from the plane formula of the DDA set-up
// (t = ((float)k cell_a + bmin_a - o_a) / d_a), in the DDA's tie order.

// Skip radius of a cell record: {r, r} marks an empty cell.
__device__ __forceinline__ int32_t skip_radius(uint2 rec, bool& empty)
{
    empty = rec.x == rec.y;
    return empty && rec.x <= (uint32_t)kSkipMax ? (int32_t)rec.x : 0;
}

// Exit t of the item at the walk's cell s with radius rr; axis: the axis
// crossed.
__device__ __forceinline__ float item_exit(const DevFrame* __restrict__ fr, const Ray2& r,
                                           const Dda& s, int32_t rr, int& axis)
{
    const float t0 =
        ((float)(r.n0 ? s.cx - rr : s.cx + rr + 1) * fr->cell[0] + fr->bmin[0] - r.o0) * r.i0;
    const float t1 =
        ((float)(r.n1 ? s.cy - rr : s.cy + rr + 1) * fr->cell[1] + fr->bmin[1] - r.o1) * r.i1;
    const float t2 =
        ((float)(r.n2 ? s.cz - rr : s.cz + rr + 1) * fr->cell[2] + fr->bmin[2] - r.o2) * r.i2;
    if (t0 < t1 && t0 < t2) {
        axis = 0;
        return t0;
    }
    if (t1 < t2) {
        axis = 1;
        return t1;
    }
    axis = 2;
    return t2;
}

// v kept within the rr cells ahead of c (behind, for a negative direction).
__device__ __forceinline__ int32_t skip_cell(int32_t v, int32_t c, int32_t rr, bool neg)
{
    if (neg) {
        v = v < c ? v : c;
        return v > c - rr ? v : c - rr;
    }
    v = v > c ? v : c;
    return v < c + rr ? v : c + rr;
}

// Step to the next item across the current one's exit (axis, at t = e);
// false when that leaves the grid.  After a skip (rr > 0) the other two
// axes take the cells of the exit point, kept within the skipped cells: no
// axis ever moves backwards, and the crossed one moves by rr + 1.
__device__ __forceinline__ bool item_advance(const DevFrame* __restrict__ fr, const Ray2& r,
                                             Dda& s, int32_t rr, int axis, float e)
{
    if (axis == 0) {
        const int32_t c = r.n0 ? s.cx - rr - 1 : s.cx + rr + 1;
        if (c < 0 || c >= fr->n[0])
            return false;
        s.cx = c;
    } else if (axis == 1) {
        const int32_t c = r.n1 ? s.cy - rr - 1 : s.cy + rr + 1;
        if (c < 0 || c >= fr->n[1])
            return false;
        s.cy = c;
    } else {
        const int32_t c = r.n2 ? s.cz - rr - 1 : s.cz + rr + 1;
        if (c < 0 || c >= fr->n[2])
            return false;
        s.cz = c;
    }
    if (rr > 0) {
        if (axis != 0)
            s.cx = skip_cell(vox(r.o0 + r.d0 * e, fr->bmin[0], fr->inv[0], fr->n[0]), s.cx, rr,
                             r.n0);
        if (axis != 1)
            s.cy = skip_cell(vox(r.o1 + r.d1 * e, fr->bmin[1], fr->inv[1], fr->n[1]), s.cy, rr,
                             r.n1);
        if (axis != 2)
            s.cz = skip_cell(vox(r.o2 + r.d2 * e, fr->bmin[2], fr->inv[2], fr->n[2]), s.cz, rr,
                             r.n2);
    }
    return true;
}

template <bool ANY>
__global__ __launch_bounds__(128) void k_trace2(TraceArgs a, RaySoA rays, HitSoA hits,
                                                uint8_t* __restrict__ occluded)
{
    __shared__ float tab[96];
    stage_sub_tab(a, tab);
    const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
    bool valid;
    const uint32_t i = trace_ray(a, slot, valid);
    if (!valid)
        return;
    const DevFrame* __restrict__ fr = a.fr;
    int32_t id = -1;
    float best = INFINITY, bu = 0.0f, bv = 0.0f;
    bool occ = false;
    uint32_t cells = 0, tests = 0;
    // Over its capacity the second level's records are not complete: the top
    // grid alone then.
    const bool sub_ok = a.g2->status == 0;
    Ray2 r;
    Dda s;
    float t_enter;
    if (ray2_setup(fr, rays, i, r, s, t_enter)) {
        const uint32_t nx = (uint32_t)fr->n[0], ny = (uint32_t)fr->n[1];
        uint32_t ci = (uint32_t)s.cx + nx * ((uint32_t)s.cy + ny * (uint32_t)s.cz);
        uint2 rec = a.cellrec[ci];
        for (;;) {
            ++cells;
            bool empty;
            const int32_t rr = skip_radius(rec, empty);
            int axis;
            const float e = item_exit(fr, r, s, rr, axis);
            // the next item and its record, loaded before this cell's tests
            Dda ns = s;
            const bool more = !(e > r.tmax) && item_advance(fr, r, ns, rr, axis, e);
            const uint32_t nci =
                (uint32_t)ns.cx + nx * ((uint32_t)ns.cy + ny * (uint32_t)ns.cz);
            // ns is inside the grid whether or not the walk goes on
            const uint2 nrec = a.cellrec[nci];
            if ((!empty && top_cell2<ANY>(a, fr, tab, sub_ok, r, s, rec, ci, t_enter, e, occ, id,
                                          best, bu, bv, cells, tests)) ||
                !more)
                break;
            t_enter = e;
            s = ns;
            ci = nci;
            rec = nrec;
        }
    }
    if (ANY) {
        occluded[i] = occ ? 1 : 0;
    } else {
        hits.id[i] = id;
        hits.t[i] = best;
        hits.u[i] = bu;
        hits.v[i] = bv;
    }
    if (a.counters) {
        a.counters[2ull * i] = cells;
        a.counters[2ull * i + 1] = tests;
    }
}

// `count` items of the walk, each after checking its exit against tmax (the
// serial walk's stop); t_enter receives the exit of the last item left.
__device__ __forceinline__ bool walk_skip(const TraceArgs& a, const DevFrame* __restrict__ fr,
                                          const Ray2& r, Dda& s, uint32_t count, float& t_enter)
{
    const uint32_t nx = (uint32_t)fr->n[0], ny = (uint32_t)fr->n[1];
    for (uint32_t q = 0; q < count; ++q) {
        const uint32_t ci = (uint32_t)s.cx + nx * ((uint32_t)s.cy + ny * (uint32_t)s.cz);
        bool empty;
        const int32_t rr = skip_radius(a.cellrec[ci], empty);
        int axis;
        const float e = item_exit(fr, r, s, rr, axis);
        if (e > r.tmax || !item_advance(fr, r, s, rr, axis, e))
            return false;
        t_enter = e;
    }
    return true;
}

// Several lanes per ray (2..16, `lanes`): lane j of a ray's group walks the
// ray's top cells j, j + lanes, ... of the serial order, each one whole (its
// sub-grid included).  After every round the group's earliest cell that ends
// the walk (a hit, an occluder, a sub-cell exit beyond tmax) decides: its
// result is the serial result, and the cells after it in that round are not
// counted.  Latency of a long ray drops about `lanes`-fold; the sparse
// secondary stages are bound by it.
template <bool ANY>
__global__ __launch_bounds__(256) void k_trace2_split(TraceArgs a, RaySoA rays, HitSoA hits,
                                                      uint8_t* __restrict__ occluded,
                                                      uint32_t lanes)
{
    __shared__ float tab[96];
    stage_sub_tab(a, tab);
    const uint32_t shift = (uint32_t)__builtin_ctz(lanes);
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    bool valid;
    const uint32_t i = trace_ray(a, t >> shift, valid);
    const DevFrame* __restrict__ fr = a.fr;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t j = lane & (lanes - 1u);
    const uint32_t g0 = lane - j;
    const uint64_t gmask = (lanes >= 64u ? ~0ull : ((1ull << lanes) - 1ull)) << g0;
    const bool sub_ok = a.g2->status == 0;
    const uint32_t nx = (uint32_t)fr->n[0], ny = (uint32_t)fr->n[1];
    int32_t id = -1;
    float best = INFINITY, bu = 0.0f, bv = 0.0f;
    bool occ = false;
    uint32_t cells = 0, tests = 0;
    Ray2 r = {};
    Dda s = {};
    float t_enter = 0.0f;
    bool alive = valid && ray2_setup(fr, rays, i, r, s, t_enter) && walk_skip(a, fr, r, s, j, t_enter);
    bool winner = false;
    while (__ballot(alive) != 0) {
        const uint32_t c0 = cells, t0 = tests;
        bool stop = false;
        int32_t rr = 0;
        int axis = 0;
        float e = 0.0f;
        if (alive) {
            ++cells;
            const uint32_t ci = (uint32_t)s.cx + nx * ((uint32_t)s.cy + ny * (uint32_t)s.cz);
            const uint2 rec = a.cellrec[ci];
            bool empty;
            rr = skip_radius(rec, empty);
            e = item_exit(fr, r, s, rr, axis);
            stop = !empty && top_cell2<ANY>(a, fr, tab, sub_ok, r, s, rec, ci, t_enter, e, occ,
                                            id, best, bu, bv, cells, tests);
        }
        // The group's earliest cell that ends the walk ends the ray; cells
        // after it (higher lanes of this round) are not part of the serial walk.
        const uint64_t sm = __ballot(alive && stop) & gmask;
        if (sm != 0) {
            const uint32_t jw = (uint32_t)__builtin_ctzll(sm) - g0;
            if (alive && j > jw) {
                cells = c0;
                tests = t0;
            }
            winner = alive && j == jw && (ANY ? occ : id >= 0);
            alive = false;
        } else if (alive) {
            alive = !(e > r.tmax) && item_advance(fr, r, s, rr, axis, e);   // NaN tmax: no stop
            if (alive) {
                t_enter = e;
                alive = walk_skip(a, fr, r, s, lanes - 1u, t_enter);
            }
        }
    }
    const bool group_hit = (__ballot(winner) & gmask) != 0;
    uint32_t sc = 0, st = 0;
    if (a.counters) {
        sc = group_sum(cells, lanes);
        st = group_sum(tests, lanes);
    }
    if (!valid)
        return;
    if (ANY) {
        if (j == 0)
            occluded[i] = group_hit ? 1 : 0;
    } else if (winner || (j == 0 && !group_hit)) {
        hits.id[i] = winner ? id : -1;
        hits.t[i] = winner ? best : INFINITY;
        hits.u[i] = winner ? bu : 0.0f;
        hits.v[i] = winner ? bv : 0.0f;
    }
    if (a.counters && j == 0) {
        a.counters[2ull * i] = sc;
        a.counters[2ull * i + 1] = st;
    }
}

hipError_t launch_trace2(const TraceArgs& a, const RaySoA& rays, const HitSoA& hits,
                         uint8_t* occluded, uint32_t lanes, hipStream_t s)
{
    if (a.n == 0)
        return hipSuccess;
    if (lanes <= 1) {
        const uint32_t g = ray_grid(a.n, a.image_width, 128);
        if (occluded)
            hipLaunchKernelGGL(k_trace2<true>, dim3(g), dim3(128), 0, s, a, rays, hits, occluded);
        else
            hipLaunchKernelGGL(k_trace2<false>, dim3(g), dim3(128), 0, s, a, rays, hits,
                               occluded);
        return hipGetLastError();
    }
    if (lanes > 16 || (lanes & (lanes - 1)) != 0)
        return hipErrorInvalidValue;
    const uint64_t threads = slot_count(a.n, a.image_width) * lanes;
    if (threads > 0xffffffffull - 256)
        return hipErrorInvalidValue;
    const dim3 g((uint32_t)((threads + 255) / 256));
    if (occluded)
        hipLaunchKernelGGL(k_trace2_split<true>, g, dim3(256), 0, s, a, rays, hits, occluded,
                           lanes);
    else
        hipLaunchKernelGGL(k_trace2_split<false>, g, dim3(256), 0, s, a, rays, hits, occluded,
                           lanes);
    return hipGetLastError();
}

// Lanes per ray of a windowed launch of `slots` ray slots.  More lanes per ray
// mean more waves with less work each -- a small launch is bound by its
// longest wave -- but every lane of a group steps the whole walk, and past a
// few times 5,120 resident waves the kernel is bound by those instructions.
// Measured (us, 1 / 2 / 4 / 8 lanes): 64x64 spheres frame 129 / 115 / 111 /
// 108, 512x512 spheres bounce 70 / 56 / 43 / 44 and primary 70 / 58 / 51 / 71,
// 904x678 spheres primary 120 / 97 / 113 / 165, 1.2 M-slot batch 592 / 568 /
// 612 / 813, 1.6 M ambient-occlusion rays with their frame 1229 / 1188 / 1276
// / 1660, serving rounds of several million slots 9383 / 10080 / 11847 / -.
static uint32_t window_lanes(uint64_t slots)
{
    if (slots >= (4u << 20))
        return 1;
    if (slots >= 400000)
        return 2;
    return slots >= 100000 ? 4 : 8;
}

template <bool ANY, bool COUNT>
static void window_launch(const TraceArgs& a, const RaySoA& rays, const HitSoA& hits,
                          uint8_t* occluded, uint32_t lanes, uint32_t grid, uint32_t block,
                          hipStream_t s)
{
    const size_t lds = block / 64 * sizeof(WaveWin);
    if (lanes == 1)
        hipLaunchKernelGGL((k_trace_window<ANY, COUNT, 4>), dim3(grid), dim3(block), lds, s, a,
                           rays, hits, occluded, lanes);
    else
        hipLaunchKernelGGL((k_trace_window<ANY, COUNT, 2>), dim3(grid), dim3(block), lds, s, a,
                           rays, hits, occluded, lanes);
}

hipError_t launch_trace_window(const TraceArgs& a, const RaySoA& rays, const HitSoA& hits,
                               uint8_t* occluded, bool any, uint32_t lanes, uint32_t block,
                               hipStream_t s)
{
    if (a.n == 0)
        return hipSuccess;
    if (lanes > 16 || (lanes & (lanes - 1)) != 0)
        return hipErrorInvalidValue;
    const uint64_t slots = slot_count(a.n, a.image_width);
    if (lanes == 0)
        lanes = window_lanes(slots);
    const uint64_t threads = slots * lanes;
    if (lanes > 1 && threads > 0xffffffffull - block)
        return hipErrorInvalidValue;
    const uint32_t g = (uint32_t)((threads + block - 1) / block);
    if (any && a.counters)
        window_launch<true, true>(a, rays, hits, occluded, lanes, g, block, s);
    else if (any)
        window_launch<true, false>(a, rays, hits, occluded, lanes, g, block, s);
    else if (a.counters)
        window_launch<false, true>(a, rays, hits, occluded, lanes, g, block, s);
    else
        window_launch<false, false>(a, rays, hits, occluded, lanes, g, block, s);
    return hipGetLastError();
}

hipError_t launch_task_map(const BatchTask* tasks, uint32_t n_tasks, uint32_t* map, hipStream_t s)
{
    if (n_tasks == 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_task_map, dim3(n_tasks), dim3(256), 0, s, tasks, map);
    return hipGetLastError();
}

hipError_t launch_trace_batch(const BatchTask* tasks, const uint32_t* map, uint32_t total_slots,
                              uint32_t lanes, uint32_t block, hipStream_t s)
{
    if (total_slots == 0)
        return hipSuccess;
    if (lanes == 0)
        lanes = window_lanes(total_slots);
    if (lanes > 16 || (lanes & (lanes - 1)) != 0)
        return hipErrorInvalidValue;
    const uint64_t threads = (uint64_t)total_slots * lanes;
    if (lanes > 1 && threads > 0xffffffffull - block)
        return hipErrorInvalidValue;
    const dim3 g((uint32_t)((threads + block - 1) / block));
    const size_t lds = block / 64 * sizeof(WaveWin);
    if (lanes == 1)
        hipLaunchKernelGGL(k_trace_batch_window<4>, g, dim3(block), lds, s, tasks, map,
                           total_slots, lanes);
    else
        hipLaunchKernelGGL(k_trace_batch_window<2>, g, dim3(block), lds, s, tasks, map,
                           total_slots, lanes);
    return hipGetLastError();
}

}  // namespace grt
