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
//   k_trace2_window       two-level grid, 1..16 lanes per ray
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

// One step (on ties y before x, z before both) when `go`; false when the ray does not go
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
// wave calls it together.  SPANS: closest hits in lists of any length (a
// template of its own: in the others the search for the record took the batch
// kernel from five waves per SIMD to four, batch of 16 scenes 534 -> 560 us).
template <bool ANY, bool COUNT, int S, bool SPANS = false>
__device__ __forceinline__ void trace_window(const DevFrame* __restrict__ fr,
                                             const uint32_t* __restrict__ offsets,
                                             const float4* __restrict__ trir, const RaySoA& rays,
                                             const HitSoA& hits, uint8_t* __restrict__ occluded,
                                             uint32_t* __restrict__ counters, uint32_t lanes,
                                             uint32_t i, bool valid, WaveWin& W)
{
    const uint32_t lane = threadIdx.x & 63u;
    float4 ro = make_float4(0.0f, 0.0f, 0.0f, 0.0f), rd = ro;
    DdaW w = {};
    bool walk;   // the lane stands on a cell of its ray
    bool open;   // the ray's result is not written yet
    const auto write_miss = [&]() {
        if (ANY) {
            occluded[i] = 0;
        } else {
            hits.id[i] = -1;
            hits.t[i] = INFINITY;
            hits.u[i] = 0.0f;
            hits.v[i] = 0.0f;
        }
    };
    for (bool again = false;; again = true) {
        walk = false;
        open = valid;
        if (valid) {
            ro = make_float4(rays.ox[i], rays.oy[i], rays.oz[i], rays.tmin[i]);
            rd = make_float4(rays.dx[i], rays.dy[i], rays.dz[i], rays.tmax[i]);
            Dda s;
            walk = grid_ok(fr) && dda_setup(fr, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z, ro.w, rd.w, s);
            if (walk)
                w = dda_window(fr, s);
        }
        // Few rays to walk: the misses are written, the others share the wave.
        const bool head = (lane & (lanes - 1u)) == 0;
        const uint64_t heads = __ballot(walk && head);
        const uint32_t more = win_lanes((uint32_t)__popcll(heads), lanes, 16u / (uint32_t)S);
        if (again || heads == 0 || more == lanes)
            break;
        if (valid && !walk && head) {
            write_miss();
            if (COUNT) {
                counters[2ull * i] = 0u;
                counters[2ull * i + 1] = 0u;
            }
        }
        lanes = (uint32_t)__builtin_amdgcn_readfirstlane((int)more);
        valid = win_regroup(W, heads, lanes, i);
    }
    const uint32_t j = lane & (lanes - 1u), owner = lane - j;
    const uint32_t c = lanes * S <= 16u ? (uint32_t)S : 16u / lanes, cell0 = j * c;
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
            const unsigned long long key = win_tests<ANY, false, S, SPANS>(
                W, WinRecs{trir, trir}, b, n, bound, 0u, owner, cell0);
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
                             : s == hs          ? (ANY ? win_pos<true>(key) + 1u : n[s])
                                                : 0u;
            }
            if (hit) {
                if (ANY) {
                    if (j == 0)
                        occluded[i] = 1;
                } else if (hs < (uint32_t)S) {
                    uint64_t k = win_pick<S>(b, hs) + win_pos<false>(key);
                    float4 A = trir[3ull * k], B = trir[3ull * k + 1], C = trir[3ull * k + 2];
                    float t, u, v;
                    bool in = mt_exact(mt_pre(A, B, C, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z), t, u, v);
                    if (SPANS) {
                        // the first of the key's positions that holds a hit at
                        // its t (an earlier one would have won; the values are
                        // the test's, bit for bit)
                        while (!(in && win_t_bits(t) == win_t_bits(key)) &&
                               (k += kWinSpan) < fr->r) {
                            A = trir[3ull * k];
                            B = trir[3ull * k + 1];
                            C = trir[3ull * k + 2];
                            in = mt_exact(mt_pre(A, B, C, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z), t,
                                          u, v);
                        }
                    }
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
    if (open && j == 0)
        write_miss();
}

extern __shared__ WaveWin win_lds[];   // one per wave of the block

template <bool ANY, bool COUNT, int S, bool SPANS>
__global__ __launch_bounds__(256) void k_trace_window(TraceArgs a, RaySoA rays, HitSoA hits,
                                                      uint8_t* __restrict__ occluded,
                                                      uint32_t lanes)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    bool valid;
    const uint32_t i = trace_ray(a, t >> __builtin_ctz(lanes), valid);
    trace_window<ANY, COUNT, S, SPANS>(a.fr, a.offsets, a.trir, rays, hits, occluded, a.counters,
                                       lanes, i, valid, win_lds[threadIdx.x >> 6]);
}

// Batched multi-scene traversal: every 64-slot group belongs to one task
// (map[slot / 64]), so each wave runs its task's walk with wave-uniform scene
// data.
template <int S, bool SPANS>
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
        trace_window<false, false, S, SPANS>(T.fr, T.offsets, T.trir, T.rays, T.hits, T.occluded,
                                             nullptr, lanes, i, valid, W);
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
// Two-level grid: windowed walk
// ---------------------------------------------------------------------------
//
// The walk over the top grid goes item by item.  An item is a cell of the
// grid; for an empty cell with skip radius rr > 0 it is the cells ahead of it
// within rr on every axis (all empty), left in one step.  Each item's exit is
// its first boundary plane crossed, from the plane formula of the DDA set-up
// (t = ((float)k cell_a + bmin_a - o_a) / d_a), in the DDA's tie order.  A top
// cell whose record carries a sub-grid resolution is walked by a DDA of its
// own from the point where the ray entered the cell (the clipped entry, then
// each item's exit), with hits bounded by the sub-cell's exit; other cells
// test their references bounded by the cell's exit.  The first (sub-)cell
// holding a hit ends a closest-hit ray, the first triangle in (tmin, tmax] an
// any-hit ray, and a sub-cell whose exit lies beyond tmax ends either.
// Counters: top items plus sub-cells visited, triangle tests.

// Top items per window at most, and the lanes below which another one waits
// for the next window while other lanes stand in sub-grids (stadium at
// 1920x1080, us, primary / shadow / bounce: 692 / 666 / 1057 with 2 items a
// window, 676 / 669 / 1022 with 4, 685 / 685 / 1037 with 8; 688 / 695 / 1058
// without the wait).
constexpr int kTopSteps = 4;
constexpr int kTopMin = 16;

// Per-ray constants of the two-level walk.
struct Ray2 {
    float o0, o1, o2, d0, d1, d2, i0, i1, i2, tmin, tmax;
    int32_t m0, m1, m2;   // -1 on the axes of negative direction, else 0
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

// DDA state inside a top cell's sub-grid: the sub-cell's index in the sub-cell
// arrays, which a step along y or z changes by sy or sz (by +-1 along x), the
// steps left on each axis before the sub-grid ends (8 bits each), the next
// boundary crossings and their increments.
struct SubW {
    uint32_t si, sy, sz, left;
    float tx, ty, tz, dtx, dty, dtz;
};

// vox(): the clamp as one median (NaN goes to 0 as there).
__device__ __forceinline__ int32_t vox_median(float val, float bmin, float inv, float hi)
{
    return (int32_t)__builtin_amdgcn_fmed3f((val - bmin) * inv, 0.0f, hi);
}

// Entry into the sub-grid of the top cell at s (record rec) at t_enter.
__device__ __forceinline__ SubW sub_setup(const DevFrame* __restrict__ fr, const float* tab,
                                          const Ray2& r, const Dda& s, uint2 rec, float t_enter)
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
    const int32_t qx = vox_median(r.o0 + r.d0 * t_enter, sb0, si0, (float)(r0 - 1));
    const int32_t qy = vox_median(r.o1 + r.d1 * t_enter, sb1, si1, (float)(r1 - 1));
    const int32_t qz = vox_median(r.o2 + r.d2 * t_enter, sb2, si2, (float)(r2 - 1));
    SubW q;
    q.left = (uint32_t)(r.m0 ? qx : r0 - 1 - qx) | (uint32_t)(r.m1 ? qy : r1 - 1 - qy) << 8 |
             (uint32_t)(r.m2 ? qz : r2 - 1 - qz) << 16;
    q.tx = ((float)(qx + 1 + r.m0) * sc0 + sb0 - r.o0) * r.i0;
    q.ty = ((float)(qy + 1 + r.m1) * sc1 + sb1 - r.o1) * r.i1;
    q.tz = ((float)(qz + 1 + r.m2) * sc2 + sb2 - r.o2) * r.i2;
    q.dtx = fabsf(sc0 * r.i0);
    q.dty = fabsf(sc1 * r.i1);
    q.dtz = fabsf(sc2 * r.i2);
    q.si = base + (uint32_t)qx + (uint32_t)r0 * ((uint32_t)qy + (uint32_t)r1 * (uint32_t)qz);
    // r0 and r0 r1, negated on the axes of negative direction
    q.sy = (uint32_t)((r0 ^ r.m1) - r.m1);
    q.sz = (uint32_t)((r0 * r1 ^ r.m2) - r.m2);
    return q;
}

// Leaves the current sub-cell (the top DDA's tie order): its exit t, and
// whether the next one is in the sub-grid.  The state is meaningless once it
// is not.
__device__ __forceinline__ float sub_step(SubW& q, uint32_t sx, bool& in)
{
    const float tx = q.tx, ty = q.ty, tz = q.tz;   // values: as in dda_window_step
    const uint32_t sy = q.sy, sz = q.sz;
    const bool ax = tx < ty && tx < tz;
    const bool ay = !ax && ty < tz;
    const bool az = !ax && !ay;
    const uint32_t sh = ax ? 0u : (ay ? 8u : 16u);
    in = ((q.left >> sh) & 255u) != 0u;
    q.left -= 1u << sh;
    q.tx = ax ? tx + q.dtx : tx;
    q.ty = ay ? ty + q.dty : ty;
    q.tz = az ? tz + q.dtz : tz;
    q.si += ax ? sx : (ay ? sy : sz);
    return ax ? tx : (ay ? ty : tz);
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
    r.m0 = __float_as_int(r.d0) >> 31;
    r.m1 = __float_as_int(r.d1) >> 31;
    r.m2 = __float_as_int(r.d2) >> 31;
    return true;
}

// Skip radius of a cell record: {r, r} marks an empty cell.
__device__ __forceinline__ int32_t skip_radius(uint2 rec, bool& empty)
{
    empty = rec.x == rec.y;
    return empty && rec.x <= (uint32_t)kSkipMax ? (int32_t)rec.x : 0;
}

// The item at the walk's cell s with skip radius rr: its exit t, the axis
// crossed there, and on every axis the cell before the exit plane -- rr cells
// ahead of s (behind, for a negative direction).
struct Item {
    float e;
    bool ax, ay;
    int32_t fx, fy, fz;
};

// (rr ^ m) + c: with m = -1 for a negative direction, else 0, the cell rr
// ahead of c is that minus m and the index of its exit plane that plus 1.
__device__ __forceinline__ Item item_exit(const DevFrame* __restrict__ fr, const Ray2& r,
                                          const Dda& s, int32_t rr)
{
    const int32_t hx = (rr ^ r.m0) + s.cx, hy = (rr ^ r.m1) + s.cy, hz = (rr ^ r.m2) + s.cz;
    const float t0 = ((float)(hx + 1) * fr->cell[0] + fr->bmin[0] - r.o0) * r.i0;
    const float t1 = ((float)(hy + 1) * fr->cell[1] + fr->bmin[1] - r.o1) * r.i1;
    const float t2 = ((float)(hz + 1) * fr->cell[2] + fr->bmin[2] - r.o2) * r.i2;
    Item it;
    it.ax = t0 < t1 && t0 < t2;
    it.ay = !it.ax && t1 < t2;
    it.e = it.ax ? t0 : (it.ay ? t1 : t2);
    it.fx = hx - r.m0;
    it.fy = hy - r.m1;
    it.fz = hz - r.m2;
    return it;
}

// a, b, c's median: v kept between two cells in either order.
__device__ __forceinline__ int32_t median(int32_t a, int32_t b, int32_t c)
{
    const int32_t lo = a < b ? a : b, hi = a < b ? b : a, m = hi < c ? hi : c;
    return lo > m ? lo : m;
}

// Step to the next item across the current one's exit; false when that leaves
// the grid (s is then meaningless).  The crossed axis takes the cell beyond
// the exit plane.  After a skip (rr > 0) the other two take the cells of the
// exit point, kept within the skipped cells, so no axis ever moves backwards;
// without one those are the current cells, so no lane branches.
__device__ __forceinline__ bool item_advance(const DevFrame* __restrict__ fr, const Ray2& r,
                                             Dda& s, const Item& it)
{
    const int32_t kx = median(vox_median(r.o0 + r.d0 * it.e, fr->bmin[0], fr->inv[0],
                                         (float)(fr->n[0] - 1)), s.cx, it.fx);
    const int32_t ky = median(vox_median(r.o1 + r.d1 * it.e, fr->bmin[1], fr->inv[1],
                                         (float)(fr->n[1] - 1)), s.cy, it.fy);
    const int32_t kz = median(vox_median(r.o2 + r.d2 * it.e, fr->bmin[2], fr->inv[2],
                                         (float)(fr->n[2] - 1)), s.cz, it.fz);
    const bool az = !it.ax && !it.ay;
    s.cx = it.ax ? it.fx + 2 * r.m0 + 1 : kx;
    s.cy = it.ay ? it.fy + 2 * r.m1 + 1 : ky;
    s.cz = az ? it.fz + 2 * r.m2 + 1 : kz;
    const uint32_t n = (uint32_t)(it.ax ? fr->n[0] : (it.ay ? fr->n[1] : fr->n[2]));
    return (uint32_t)(it.ax ? s.cx : (it.ay ? s.cy : s.cz)) < n;
}

// A wave walks its rays in windows as trace_window does, `lanes` lanes per ray
// (lanes x S <= 16 units a window): a unit is a top cell's list or a
// sub-cell's, unit u of the window going to lane u / S of the group.  A window
// is a few top items, until the lane stands in a sub-grid or its units are
// used up, then sub-cells up to the window's end.
//
// Bound by VALU issue while the chip is full (0.69 of the cycles over the whole
// launch, 8.7 k instructions a wave on primary rays, of which the top walk is
// two fifths and the tests a quarter), then by the longest waves: one wave
// alone takes up to 0.42 ms with a ray per lane, 0.18 ms with 16 lanes per ray.
// The per-lane walk this replaced ran 15-32 of 64 lanes per instruction, this
// one 33-44.  Stadium of 2^20 triangles, us before -> after: 1920x1080 primary
// 821 -> 676, shadow 1110 -> 669, bounce 1463 -> 1022; 480x270 primary 768 ->
// 293, shadow 1305 -> 211.  Waves that take new rays as lanes fall idle were
// slower (primary 1229 us): rays of different image parts share fewer steps.
// The next window's loads before this one's tests cost a wave per SIMD
// (primary 854 against 746 us).
template <bool ANY, bool COUNT, int S>
__global__ __launch_bounds__(128) void k_trace2_window(TraceArgs a, RaySoA rays, HitSoA hits,
                                                       uint8_t* __restrict__ occluded,
                                                       uint32_t lanes)
{
    __shared__ float tab[96];
    stage_sub_tab(a, tab);
    WaveWin& W = win_lds[threadIdx.x >> 6];
    const uint32_t lane = threadIdx.x & 63u;
    bool valid;
    uint32_t i = trace_ray(a, (blockIdx.x * blockDim.x + threadIdx.x) >> __builtin_ctz(lanes),
                           valid);
    const DevFrame* __restrict__ fr = a.fr;
    const uint32_t nx = (uint32_t)fr->n[0], ny = (uint32_t)fr->n[1];
    // Over its capacity the second level's records are not complete: the top
    // grid alone then.
    const bool sub_ok = a.g2->status == 0;
    Ray2 r = {};
    Dda s = {};
    float t_enter = 0.0f;
    uint2 rec = make_uint2(0u, 0u);
    bool top;    // an item of the top walk is next
    bool open;   // the result is not written yet
    const auto write_miss = [&]() {
        if (ANY) {
            occluded[i] = 0;
        } else {
            hits.id[i] = -1;
            hits.t[i] = INFINITY;
            hits.u[i] = 0.0f;
            hits.v[i] = 0.0f;
        }
    };
    for (bool again = false;; again = true) {
        top = valid && ray2_setup(fr, rays, i, r, s, t_enter);
        open = valid;
        // Few rays to walk: the misses are written, the others share the wave.
        const bool head = (lane & (lanes - 1u)) == 0;
        const uint64_t heads = __ballot(top && head);
        const uint32_t more = win_lanes((uint32_t)__popcll(heads), lanes, 16u / (uint32_t)S);
        if (again || heads == 0 || more == lanes)
            break;
        if (valid && !top && head) {
            write_miss();
            if (COUNT) {
                a.counters[2ull * i] = 0u;
                a.counters[2ull * i + 1] = 0u;
            }
        }
        lanes = (uint32_t)__builtin_amdgcn_readfirstlane((int)more);
        valid = win_regroup(W, heads, lanes, i);
    }
    const uint32_t j = lane & (lanes - 1u), owner = lane - j, cell0 = j * (uint32_t)S;
    const uint32_t units = lanes * (uint32_t)S;
    uint32_t cells = 0, tests = 0;
    if (__ballot(top) != 0) {
        W.ro[lane] = make_float4(r.o0, r.o1, r.o2, win_lo(r.tmin));
        W.rd[lane] = make_float4(r.d0, r.d1, r.d2, r.tmin);
        uint32_t ci = (uint32_t)s.cx + nx * ((uint32_t)s.cy + ny * (uint32_t)s.cz);
        if (top)
            rec = a.cellrec[ci];
        const uint32_t sx = (uint32_t)(r.m0 | 1);
        bool insub = false;   // the walk stands in a sub-grid
        SubW w = {};
        WinU<S> nb, nn, nend, ncum;
        uint32_t nsubs;
        const auto next_window = [&]() {
            uint32_t u = 0, idx[S];
            nsubs = 0;
#pragma unroll
            for (int q = 0; q < S; ++q) {
                nb[q] = 0u;
                nn[q] = 0u;
                nend[q] = ANY ? __float_as_uint(r.tmax) : 0u;
                ncum[q] = 0u;
                idx[q] = 0u;
            }
            for (int k = 0; k < kTopSteps; ++k) {
                const bool need = top && !insub && u < units;
                const uint64_t m = __ballot(need);
                if (m == 0 || (k != 0 && __popcll(m) < kTopMin && __ballot(insub) != 0))
                    break;
                if (need) {
                    ++cells;
                    bool empty;
                    const int32_t rr = skip_radius(rec, empty);
                    const Item it = item_exit(fr, r, s, rr);
                    const bool has_sub = (rec.x >> 31) != 0u;
                    if (!empty && has_sub && sub_ok) {
                        w = sub_setup(fr, tab, r, s, rec, t_enter);
                        insub = true;
                    } else if (!empty) {
                        // the top cell's own list (also for a sub-grid cell
                        // when the second level is not valid)
                        if (has_sub)
                            rec = make_uint2(a.offsets[ci], a.offsets[ci + 1]);
                        const uint32_t bound = __float_as_uint(win_end(r.tmax, it.e * kExitScale));
#pragma unroll
                        for (int q = 0; q < S; ++q) {
                            const bool mine = u == cell0 + (uint32_t)q;
                            nb[q] = mine ? rec.x : uint32_t(nb[q]);
                            nn[q] = mine ? rec.y - rec.x : uint32_t(nn[q]);
                            if (!ANY)
                                nend[q] = mine ? bound : uint32_t(nend[q]);
                            if (COUNT)
                                ncum[q] = mine ? cells : uint32_t(ncum[q]);
                        }
                        ++u;
                    }
                    top = item_advance(fr, r, s, it) && !(it.e > r.tmax);
                    t_enter = it.e;
                    if (top) {
                        ci = (uint32_t)s.cx + nx * ((uint32_t)s.cy + ny * (uint32_t)s.cz);
                        rec = a.cellrec[ci];
                    }
                }
            }
            if (__ballot(insub) == 0)
                return;
            for (uint32_t jj = 0; jj < lanes; ++jj) {
#pragma unroll
                for (int q = 0; q < S; ++q) {
                    if (insub && jj * (uint32_t)S + (uint32_t)q >= u) {
                        const bool mine = lanes == 1u || jj == j;
                        ++cells;
                        idx[q] = mine ? uint32_t(w.si) : idx[q];
                        nsubs |= mine ? 1u << q : 0u;
                        if (COUNT)
                            ncum[q] = mine ? cells : uint32_t(ncum[q]);
                        const float ex = sub_step(w, sx, insub);
                        if (!ANY) {
                            const uint32_t bound =
                                __float_as_uint(win_end(r.tmax, ex * kExitScale));
                            nend[q] = mine ? bound : uint32_t(nend[q]);
                        }
                        if (ex > r.tmax) {
                            insub = false;
                            top = false;
                        }
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < S; ++q) {
                const uint32_t* o = a.sub_offsets + idx[q];
                const uint32_t b = o[0], e = o[1];
                const bool sub = (nsubs >> q) & 1u;
                nb[q] = sub ? b : uint32_t(nb[q]);
                nn[q] = sub ? e - b : uint32_t(nn[q]);
            }
        };
        do {
            next_window();
            const WinU<S> b = nb, n = nn, bound = nend, cum = ncum;
            const uint32_t subs = nsubs;
            const unsigned long long key = win_tests<ANY, true, S, false>(
                W, WinRecs{a.trir, a.sub_trir}, b, n, bound, subs, owner, cell0);
            const bool hit = key != ~0ull;
            const uint32_t hs = win_cell(key) - cell0;   // >= S: not one of the lane's units
            if (COUNT && open) {
                const bool after = hit && win_cell(key) < cell0;
#pragma unroll
                for (uint32_t q = 0; q < (uint32_t)S; ++q)
                    tests += after                         ? 0u
                             : !hit || hs >= (uint32_t)S || q < hs ? n[q]
                             : q == hs                     ? (ANY ? win_pos<true>(key) + 1u : n[q])
                                                           : 0u;
                if (hit)
                    cells = hs < (uint32_t)S ? win_pick<S>(cum, hs) : 0u;
            }
            if (hit) {
                if (ANY) {
                    if (j == 0)
                        occluded[i] = 1;
                } else if (hs < (uint32_t)S) {
                    const uint64_t k = win_pick<S>(b, hs) + win_pos<false>(key);
                    const float4* __restrict__ tri = (subs >> hs) & 1u ? a.sub_trir : a.trir;
                    const float4 A = tri[3ull * k], B = tri[3ull * k + 1], C = tri[3ull * k + 2];
                    const MtPre m = mt_pre(A, B, C, r.o0, r.o1, r.o2, r.d0, r.d1, r.d2);
                    float t, u, v;
                    mt_exact(m, t, u, v);
                    hits.id[i] = (int32_t)__float_as_uint(C.y);
                    hits.t[i] = t;
                    hits.u[i] = u;
                    hits.v[i] = v;
                }
                open = false;
                top = false;
                insub = false;
            }
        } while (__ballot(top || insub) != 0);
        if (COUNT && open && j != 0)
            cells = 0u;   // every lane of the group counted the whole walk
    }
    if (COUNT) {
        const uint32_t sc = group_sum(cells, lanes), st = group_sum(tests, lanes);
        if (valid && j == 0) {
            a.counters[2ull * i] = sc;
            a.counters[2ull * i + 1] = st;
        }
    }
    if (open && j == 0)
        write_miss();
}

template <bool ANY, bool COUNT>
static void trace2_launch(const TraceArgs& a, const RaySoA& rays, const HitSoA& hits,
                          uint8_t* occluded, uint32_t lanes, uint32_t grid, hipStream_t s)
{
    constexpr uint32_t kBlock = 128;
    const size_t lds = kBlock / 64 * sizeof(WaveWin);
    if (lanes <= 4)
        hipLaunchKernelGGL((k_trace2_window<ANY, COUNT, 4>), dim3(grid), dim3(kBlock), lds, s, a,
                           rays, hits, occluded, lanes);
    else if (lanes == 8)
        hipLaunchKernelGGL((k_trace2_window<ANY, COUNT, 2>), dim3(grid), dim3(kBlock), lds, s, a,
                           rays, hits, occluded, lanes);
    else
        hipLaunchKernelGGL((k_trace2_window<ANY, COUNT, 1>), dim3(grid), dim3(kBlock), lds, s, a,
                           rays, hits, occluded, lanes);
}

// Lanes per ray of a two-level launch of `slots` ray slots.  The top walk is
// stepped by every lane of a group, so large launches take one lane; small
// ones are bound by their longest wave.  Measured on the stadium (us, 1 / 2 /
// 4 / 8 / 16 lanes): 1360x765 primary 496 / 529 / 720 / - / -; 960x540 primary
// 434 / 393 / 447 / 628 / -, shadow 419 / 295 / 389 / 528 / -, bounce 623 / 570
// / 605 / 735 / -; 720x405 primary - / 348 / 368 / 421 / 615, shadow - / 293 /
// 268 / 363 / 505, bounce - / 476 / 496 / 516 / 673, bounce shadow - / 220 / 214
// / 197 / 218 (2 and 4 are level over the stages); 480x270 primary 432 / 315 /
// 295 / 293 / 372, shadow 417 / 298 / 239 / 211 / 282, bounce 580 / 377 / 399 /
// 365 / 411; 160x90 shadow 424 / 277 / 218 / 185 / 174.
static uint32_t trace2_lanes(uint64_t slots)
{
    if (slots >= 1000000)
        return 1;
    if (slots >= 300000)
        return 2;
    if (slots >= 150000)
        return 4;
    return slots >= 32000 ? 8 : 16;
}

// A fixed number of lanes per ray (the split schedule) holds below kFixedSlots
// ray slots, and for ray lists, which may name few of them; otherwise at most
// kFixedLanes from there on.  Every lane of a group steps the whole walk,
// sub-grids included, so more lanes do not pay there: stadium (us, 4 lanes / 2)
// 1920x1080 primary 1346 / 879, bounce 1681 / 1204; 960x540 primary 445 / 401,
// shadow 393 / 304, bounce 606 / 513, bounce shadow 238 / 230; below, at
// 720x405, shadow 268 / 293 and bounce shadow 214 / 220.  The walk in which the
// lanes of a group took sub-grids in turn had 1225 and 1700 with 4 lanes at
// 1920x1080.
constexpr uint32_t kFixedLanes = 2;
constexpr uint64_t kFixedSlots = 500000;

hipError_t launch_trace2(const TraceArgs& a, const RaySoA& rays, const HitSoA& hits,
                         uint8_t* occluded, uint32_t lanes, hipStream_t s)
{
    if (a.n == 0)
        return hipSuccess;
    if (lanes > 16 || (lanes & (lanes - 1)) != 0)
        return hipErrorInvalidValue;
    const uint64_t slots = slot_count(a.n, a.image_width);
    uint64_t threads = slots * lanes;
    if (lanes > 1 && threads > 0xffffffffull - 256)
        return hipErrorInvalidValue;
    if (lanes == 0)
        lanes = trace2_lanes(slots);
    else if (lanes > kFixedLanes && slots >= kFixedSlots && !a.list)
        lanes = kFixedLanes;
    threads = slots * lanes;
    const uint32_t g = (uint32_t)((threads + 127) / 128);
    if (occluded && a.counters)
        trace2_launch<true, true>(a, rays, hits, occluded, lanes, g, s);
    else if (occluded)
        trace2_launch<true, false>(a, rays, hits, occluded, lanes, g, s);
    else if (a.counters)
        trace2_launch<false, true>(a, rays, hits, occluded, lanes, g, s);
    else
        trace2_launch<false, false>(a, rays, hits, occluded, lanes, g, s);
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
//
// Rays that run along a flat grid cross many times the cells of the others, so
// its launches wait longer for their last waves, and up to a million slots
// twice the lanes pay: 2^20-triangle stadium (us, 2 / 4 / 8 / 16 lanes),
// 1280x720 frame at lambda 128 4026 / 3594 / 3517 / 4846; 960x540 primary at
// lambda 8 6174 / 5354 / 4359 / 3312, at 64 1538 / 1341 / 1279 / 1601, at 256
// 1044 / 907 / 1087 / 1880; 480x270 frame 2305 / 1736 / 1446 / 1419; 160x90
// frame 2174 / 1458 / 1128 / 990.  The rule knows only size and flatness, so it
// stays where a fine grid, which such a scene needs, does best (lambda 256: 4
// lanes at 960x540); a coarse one, with its long lists, would gain from more
// (lambda 64 5% with 8, lambda 8 38% with 16).
static uint32_t window_lanes(uint64_t slots, bool flat)
{
    if (slots >= (4u << 20))
        return 1;
    if (slots >= 1000000 || (slots >= 400000 && !flat))
        return 2;
    const uint32_t l = slots >= 400000 ? 2 : slots >= 100000 ? 4 : 8;
    return flat ? 2 * l : l;
}

template <bool ANY, bool COUNT>
static void window_launch(const TraceArgs& a, const RaySoA& rays, const HitSoA& hits,
                          uint8_t* occluded, uint32_t lanes, uint32_t grid, uint32_t block,
                          hipStream_t s)
{
    const size_t lds = block / 64 * sizeof(WaveWin);
    if (!ANY && a.spans)
        hipLaunchKernelGGL((k_trace_window<ANY, COUNT, 4, !ANY>), dim3(grid), dim3(block), lds, s,
                           a, rays, hits, occluded, lanes);
    else if (lanes == 1)
        hipLaunchKernelGGL((k_trace_window<ANY, COUNT, 4, false>), dim3(grid), dim3(block), lds, s,
                           a, rays, hits, occluded, lanes);
    else
        hipLaunchKernelGGL((k_trace_window<ANY, COUNT, 2, false>), dim3(grid), dim3(block), lds, s,
                           a, rays, hits, occluded, lanes);
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
        lanes = window_lanes(slots, a.flat);
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
                              bool spans, uint32_t lanes, uint32_t block, hipStream_t s)
{
    if (total_slots == 0)
        return hipSuccess;
    if (lanes == 0)
        lanes = window_lanes(total_slots, false);
    if (lanes > 16 || (lanes & (lanes - 1)) != 0)
        return hipErrorInvalidValue;
    const uint64_t threads = (uint64_t)total_slots * lanes;
    if (lanes > 1 && threads > 0xffffffffull - block)
        return hipErrorInvalidValue;
    const dim3 g((uint32_t)((threads + block - 1) / block));
    const size_t lds = block / 64 * sizeof(WaveWin);
    if (spans)
        hipLaunchKernelGGL((k_trace_batch_window<4, true>), g, dim3(block), lds, s, tasks, map,
                           total_slots, lanes);
    else if (lanes == 1)
        hipLaunchKernelGGL((k_trace_batch_window<4, false>), g, dim3(block), lds, s, tasks, map,
                           total_slots, lanes);
    else
        hipLaunchKernelGGL((k_trace_batch_window<2, false>), g, dim3(block), lds, s, tasks, map,
                           total_slots, lanes);
    return hipGetLastError();
}

}  // namespace grt
