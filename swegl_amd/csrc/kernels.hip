// kernels.hip -- gfx950 kernels of the render path.
//
// Stage map (reference loop -> kernel):
//   vertex_shaders.hpp:16-71 (v_world, normal_world, frustum coords)  -> k_vertex
//   renderer.cpp:83-185 (visibility marks), binning counts          -> k_front
//   renderer.cpp:240-460 (clip, DDA setup) for binning              -> k_front / k_bin_fill
//   renderer.cpp:462-558 (spans, z test) + pixel shading            -> k_raster (per tile)
//   post_shaders.hpp:51-131 (depth of field)                        -> k_dof
// Every kernel works on a batch of jobs (one job = one viewport of one
// scene); a block finds its job by binary search over the job table, so the
// plain path is simply a batch of one.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "jobs.h"
#include "launch.h"

namespace sw {

// ------------------------------------------------------------ job lookup
enum { JV = 0, JT = 1, JD = 2, JTILE = 3 };
template <int F>
__device__ __forceinline__ uint32_t first_block(const JobDev &j)
{
    return F == JV ? j.vblock0 : F == JT ? j.tblock0 : F == JD ? j.dblock0 : j.tile_base;
}
// Every kernel takes the job table as a `const __restrict__` argument of its
// own as well: the table is not written while kernels run, and through such
// an argument the compiler reads uniform job fields with scalar loads.
template <int F>
__device__ __forceinline__ int find_job(const BatchDev &B, const JobDev *__restrict__ jobs, uint32_t blk)
{
    int lo = 0, hi = (int)B.n_jobs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (first_block<F>(jobs[mid]) <= blk)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}
// Triangle t's vertex ids (x, y, z) and primitive (w).
__device__ __forceinline__ uint4 tri_ids(const uint4 *tri, uint32_t t)
{
    const SW_RO uint32_t *q = ro((const uint32_t *)(tri + t));
    return make_uint4(q[0], q[1], q[2], q[3]);
}

__device__ __forceinline__ f3 ld3(const float4 *a, uint32_t i)
{
    const float4 v = ro4(a, i);
    return {v.x, v.y, v.z};
}

// Wave-aggregated atomicAdd.  Lanes holding the same key are grouped with
// ballots (ALU only); then every group leader issues its atomic in the same
// instruction, so the wave waits for one round trip instead of one per key.
// Grouping costs a lane exchange per distinct key, so it stops after
// SW_WAVE_ADD_GROUPS groups: the lanes left (many distinct keys, as a large
// triangle's tiles are) add 1 on their own in that same instruction.
// Returns this lane's slot (old value + rank among same-key lanes) when
// `want_slot`; inactive lanes get 0.
#ifndef SW_WAVE_ADD_GROUPS
#define SW_WAVE_ADD_GROUPS 4
#endif
template <bool want_slot>
__device__ __forceinline__ uint32_t wave_add(uint32_t *base, uint32_t key, bool active)
{
    const int lane = __lane_id();
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint64_t pending = __ballot(active);
    int my_leader = lane;
    uint32_t my_rank = 0, count = 1;   // a lane left ungrouped adds 1 itself
    for (int g = 0; pending && g < SW_WAVE_ADD_GROUPS; g++) {
        const int leader = __ffsll((unsigned long long)pending) - 1;
        const uint32_t lkey = __shfl(key, leader);
        const uint64_t same = __ballot(active && key == lkey);
        if (active && key == lkey) {
            my_leader = leader;
            my_rank = (uint32_t)__popcll(same & below);
        }
        if (lane == leader)
            count = (uint32_t)__popcll(same);
        pending &= ~same;
    }
    const bool is_leader = active && my_leader == lane;
    if (!want_slot) {
        if (is_leader)
            atomicAdd(&base[key], count);
        return 0;
    }
    uint32_t old = 0;
    if (is_leader)
        old = atomicAdd(&base[key], count);
    old = __shfl(old, my_leader);
    return active ? old + my_rank : 0u;
}

__device__ __forceinline__ void stat_add(const BatchDev &B, int idx, unsigned long long v)
{
    unsigned long long *st = (unsigned long long *)(B.ctr + SW_CTR_STATS);   // 8-byte aligned
    atomicAdd(&st[(blockIdx.x & (SW_STAT_SLOTS - 1)) * 8 + idx], v);
}

// ------------------------------------------------------------- k_world
// original_to_world (vertex_shaders.hpp:16-33) and normal_world
// (:61-63).  Both depend only on the scene and its node poses, so they are
// computed when a scene is uploaded or re-posed, not per render.
__global__ __launch_bounds__(256) void k_world(WorldArgs W)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= W.n_vertices)
        return;
    int lo = 0, hi = (int)W.n_prims - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (W.prims[mid].first_vertex <= i)
            lo = mid;
        else
            hi = mid - 1;
    }
    const NodeDev &N = W.nodes[W.prims[lo].node];
    const f3 w = xform(N.M, f3{W.px[i], W.py[i], W.pz[i]});
    const f3 n = normal_world(N.RS, f3{W.nx[i], W.ny[i], W.nz[i]});
    // the texture coordinates, in texels, ride in the fourth lanes, so a
    // shading lane gets a vertex's position, normal and coordinates in two
    // loads
    const PrimDev &P = W.prims[lo];
    W.world[i] = make_float4(w.x, w.y, w.z, W.tu[i] * (float)P.tw);
    W.nworld[i] = make_float4(n.x, n.y, n.z, W.tv[i] * (float)P.th);
}

// ------------------------------------------------------------ k_vertex
// world_to_camera_or_frustum (vertex_shaders.hpp:35-52, 61-71) per viewport:
// frustum coordinates and cleared visibility marks.
// It also zeroes the tile counts and fill ranks and the counter words
// [w0, w0 + n_words) that the binning kernels after it accumulate into, and
// marks every tile as without an offset.
__device__ __forceinline__ void vertex_block(const BatchDev &B, uint32_t w0, uint32_t n_words, const JobDev &J)
{
    const uint32_t gi = blockIdx.x * 256u + threadIdx.x, stride = gridDim.x * 256u;
    for (uint32_t k = gi; k < B.n_tiles; k += stride) {
        B.tile_count[k * SW_TILE_PAD] = 0;
        B.tile_cursor[k * SW_TILE_PAD] = 0;
        B.tile_offset[k] = SW_NO_OFFSET;
    }
    for (uint32_t k = gi; k < n_words; k += stride)
        B.ctr[w0 + k] = 0;
    const uint32_t i = (blockIdx.x - J.vblock0) * 256u + threadIdx.x;
    if (i >= J.n_vertices)
        return;
    const float4 w4 = ro4(J.world, i);
    const f3 f = world_to_frustum(J.V, f3{w4.x, w4.y, w4.z});
    // 1 / z: the interpolators' start value (interpolator.hpp:58-62), which
    // every setup of a triangle with this vertex would divide out again
    J.ndc[i] = make_float4(f.x, f.y, f.z, 1.0f / f.z);
    J.yes[i] = 0;
}
__global__ __launch_bounds__(256) void k_vertex(BatchDev B, uint32_t w0, uint32_t n_words, const JobDev *__restrict__ jobs)
{
    vertex_block(B, w0, n_words, jobs[find_job<JV>(B, jobs, blockIdx.x)]);
}
// The same for a wave of one job, whose table arrives with the arguments (488
// bytes) and is left in memory for the kernels after it: a copy of its own
// ahead of the kernels is one more operation on the stream that every frame
// waits for (640x480 cube 39 us a frame with it, 35 without; 800x600 demo
// scene 57 and 50; 1280x720 field posed anew 119 and 114).
__global__ __launch_bounds__(256) void k_vertex_one(BatchDev B, uint32_t w0, uint32_t n_words, JobDev J)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *const_cast<JobDev *>(B.jobs) = J;
    vertex_block(B, w0, n_words, J);
}

// A triangle's three vertices carry visibility marks (renderer.cpp:248-253
// draws a triangle only then).
__device__ __forceinline__ bool marked(const JobDev &J, uint32_t t)
{
    const uint4 id = tri_ids(J.tri, t);
    return (ro(J.yes)[id.x] != 0) & (ro(J.yes)[id.y] != 0) & (ro(J.yes)[id.z] != 0);
}

// ------------------------------------------------ fill_triangle on device
__device__ SVert orig_vertex(const JobDev &J, uint32_t i)
{
    SVert v;
    v.s = frustum_to_screen(J.V, ld3(J.ndc, i));
    v.a = v.b = i;
    v.cut = 0.0f;
    v.clip = 0;
    return v;
}
// new vertex between a and b (renderer.cpp:290-297 and world_to_viewport)
__device__ SVert clip_vertex(const JobDev &J, uint32_t a, uint32_t b, float cut)
{
    f3 wa = ld3(J.world, a), wb = ld3(J.world, b);
    f3 w = wa + (wb - wa) * cut;
    SVert v;
    v.s = frustum_to_screen(J.V, world_to_frustum(J.V, w));
    v.a = a;
    v.b = b;
    v.cut = cut;
    v.clip = 1;
    return v;
}

// fill_triangle (renderer.cpp:240-359): the sub-triangles handed to
// fill_triangle_2, in call order.  Returns how many (0, 1 or 2).
// BINNED: t came out of the binning, which lists a triangle only if all
// three of its vertices are marked (quick_extent, and this function with
// marks checked on the exact path), so the marks need no second look.
// The same with triangle t's vertex ids already loaded (i0, i1, i2).
template <bool BINNED = false>
__device__ int tri_subs_v(const JobDev &J, uint32_t i0, uint32_t i1, uint32_t i2, SubTri *out)
{
    if (!BINNED && !(ro(J.yes)[i0] && ro(J.yes)[i1] && ro(J.yes)[i2]))
        return 0;
    SVert v0 = orig_vertex(J, i0), v1 = orig_vertex(J, i1), v2 = orig_vertex(J, i2);
    bool front = cross_z_sign(v1.s - v0.s, v2.s - v0.s, -1);
    bool inv = false;
    if (v1.s.z > v0.s.z) { SVert x = v0; v0 = v1; v1 = x; inv = !inv; }
    if (v2.s.z > v1.s.z) { SVert x = v1; v1 = v2; v2 = x; inv = !inv; }
    if (v1.s.z > v0.s.z) { SVert x = v0; v0 = v1; v1 = x; inv = !inv; }
    if (v2.s.z >= SW_NEAR) {
        out[0].v[0] = v0;
        out[0].v[1] = v1;
        out[0].v[2] = v2;
        out[0].front = front;
        return 1;
    }
    if (v1.s.z < SW_NEAR) {
        float cut1 = (v0.s.z - 0.001f) / (v0.s.z - v1.s.z);
        SVert n1 = clip_vertex(J, v0.a, v1.a, cut1);
        float cut2 = (v0.s.z - 0.001f) / (v0.s.z - v2.s.z);
        SVert n2 = clip_vertex(J, v0.a, v2.a, cut2);
        bool f = cross_z_sign(n1.s - v0.s, n2.s - v0.s, -1);
        out[0].v[0] = v0;
        out[0].v[1] = n1;
        out[0].v[2] = n2;
        out[0].front = inv ? !f : f;
        return 1;
    }
    if (v2.s.z < SW_NEAR) {
        float cut0 = (v0.s.z - 0.001f) / (v0.s.z - v2.s.z);
        SVert n1 = clip_vertex(J, v0.a, v2.a, cut0);
        float cut1 = (v1.s.z - 0.001f) / (v1.s.z - v2.s.z);
        SVert n2 = clip_vertex(J, v1.a, v2.a, cut1);
        bool f0 = cross_z_sign(v1.s - v0.s, n2.s - v0.s, -1);
        out[0].v[0] = v0;
        out[0].v[1] = v1;
        out[0].v[2] = n2;
        out[0].front = inv ? !f0 : f0;
        bool f1 = cross_z_sign(n2.s - v0.s, n1.s - v0.s, -1);
        out[1].v[0] = v0;
        out[1].v[1] = n2;
        out[1].v[2] = n1;
        out[1].front = inv ? !f1 : f1;
        return 2;
    }
    return 0;   // NaN depth: no branch of the reference is taken
}
template <bool BINNED = false>
__device__ __forceinline__ int tri_subs(const JobDev &J, uint32_t t, SubTri *out)
{
    const uint4 id = tri_ids(J.tri, t);
    return tri_subs_v<BINNED>(J, id.x, id.y, id.z, out);
}

// Rows a sub-triangle's halves process, and a conservative column range.
struct Extent {
    int y0, y1;   // [y0, y1)
    int x0, x1;   // [x0, x1]
};
// Columns of a triangle's tile rectangle: the vertex x range widened by
// SW_RECT_MARGIN pixels plus a bound of the DDA's accumulated rounding
// ((rows + 8) add errors of at most 2^-20 |x|max each, 16 times the float
// half-ulp).  A covered pixel x satisfies ceil(left.x) <= x < ceil(right.x)
// with both sides within the vertex x range up to that rounding, so the
// bound holds with no margin at all; the margin is spare.  A brute-force
// check against the rasteriser on adversarial triangles pins it.
#define SW_RECT_MARGIN 0.5f

__device__ bool sub_extent(const Setup &S, const ViewXf &V, Extent &E)
{
    int ya = INT32_MAX, yb = INT32_MIN;
    if (S.has_up && S.up_y1 > S.up_y0) {
        ya = min(ya, S.up_y0);
        yb = max(yb, S.up_y1);
    }
    if (S.has_lo && S.lo_y1 > S.lo_y0) {
        ya = min(ya, S.lo_y0);
        yb = max(yb, S.lo_y1);
    }
    if (ya >= yb)
        return false;
    E.y0 = ya;
    E.y1 = yb;
    float xmin = fminf(S.v[0].s.x, fminf(S.v[1].s.x, S.v[2].s.x));
    float xmax = fmaxf(S.v[0].s.x, fmaxf(S.v[1].s.x, S.v[2].s.x));
    // The DDA reaches row k after k float adds; each add is off by at most
    // half an ulp of the largest |x| on the walk.  Widen by that bound.
    float X = fmaxf(fmaxf(fabsf(xmin), fabsf(xmax)), 1.0f);
    float slack = SW_RECT_MARGIN + (float)(yb - ya + 8) * X * (1.0f / 1048576.0f);
    if (!(xmin == xmin) || !(xmax == xmax) || X > 1e30f) {
        E.x0 = V.vx;
        E.x1 = V.vx + V.vw - 1;
        return true;
    }
    float fx0 = floorf(xmin - slack), fx1 = ceilf(xmax + slack);
    E.x0 = fx0 < (float)V.vx ? V.vx : (int)fx0;
    E.x1 = fx1 > (float)(V.vx + V.vw - 1) ? V.vx + V.vw - 1 : (int)fx1;
    return E.x0 <= E.x1;
}

#define RECT_EMPTY 0xFFFFFFFFu

// ------------------------------------------------------ tile rectangles
// Tile rectangle of a triangle, conservative but never too small: rows are
// exact (ceil of vertex y, clipped to the viewport), columns are the vertex
// x range widened by the DDA's worst-case accumulated rounding.
// Near-clipped or non-finite triangles take the exact fill_triangle path.
// The extent of an unclipped, finite triangle from its screen points; sets
// `exact` when the triangle needs fill_triangle's exact path (near-clipped
// or non-finite).  `drawn`: fill_triangle_2 would draw it (y0 != y2).
__device__ bool quick_extent(const JobDev &J, f3 a, f3 b, f3 c, Extent &E, uint32_t &drawn, bool &exact)
{
    exact = false;
    drawn = 0;
    const float big = 1073741824.0f;
    bool finite = fabsf(a.x) < big && fabsf(b.x) < big && fabsf(c.x) < big && fabsf(a.y) < big &&
                  fabsf(b.y) < big && fabsf(c.y) < big;
    if (!finite || !(fminf(a.z, fminf(b.z, c.z)) >= SW_NEAR) || a.z != a.z || b.z != b.z || c.z != c.z) {
        exact = true;
        return false;
    }
    const float ymin = fminf(a.y, fminf(b.y, c.y)), ymax = fmaxf(a.y, fmaxf(b.y, c.y));
    const int iy0 = cvtt(ceilf(ymin)), iy2 = cvtt(ceilf(ymax));
    if (iy0 == iy2)
        return false;
    drawn = 1;
    const int y0 = max(iy0, J.V.vy), y1 = min(iy2, J.V.vy + J.V.vh);
    if (y0 >= y1)
        return false;
    E.y0 = y0;
    E.y1 = y1;
    const float xmin = fminf(a.x, fminf(b.x, c.x)), xmax = fmaxf(a.x, fmaxf(b.x, c.x));
    const float X = fmaxf(fmaxf(fabsf(xmin), fabsf(xmax)), 1.0f);
    const float slack = SW_RECT_MARGIN + (float)(iy2 - iy0 + 8) * X * (1.0f / 1048576.0f);
    const float fx0 = floorf(xmin - slack), fx1 = ceilf(xmax + slack);
    E.x0 = fx0 < (float)J.V.vx ? J.V.vx : (int)fx0;
    E.x1 = fx1 > (float)(J.V.vx + J.V.vw - 1) ? J.V.vx + J.V.vw - 1 : (int)fx1;
    return E.x0 <= E.x1;
}

// The exact path: the union extent of fill_triangle's sub-triangles and how
// many of them fill_triangle_2 draws.  Marks are not looked at here.
__device__ bool exact_extent(const JobDev &J, uint32_t t, Extent &E, uint32_t &drawn)
{
    SubTri st[2];
    const int ns = tri_subs<true>(J, t, st);
    int ya = INT32_MAX, yb = INT32_MIN, xa = INT32_MAX, xb = INT32_MIN;
    drawn = 0;
#pragma unroll
    for (int s = 0; s < 2; s++) {
        Setup S;
        if (s >= ns || !setup_subtri(st[s], J.V, S))
            continue;
        drawn++;
        Extent e;
        if (!sub_extent(S, J.V, e))
            continue;
        ya = min(ya, e.y0);
        yb = max(yb, e.y1);
        xa = min(xa, e.x0);
        xb = max(xb, e.x1);
    }
    E.y0 = ya;
    E.y1 = yb;
    E.x0 = xa;
    E.x1 = xb;
    return ya < yb && xa <= xb;
}

// The tile rows of the k_front/k_bin_fill rectangle, shared by both.
__device__ __forceinline__ uint2 tile_rect(const JobDev &J, const Extent &E, int &tx0, int &tx1, int &ty0, int &ty1)
{
    // tile edges are powers of two and the offsets are not negative: shifts
    const int sx = __builtin_ctz((unsigned)J.tw), sy = __builtin_ctz((unsigned)J.th);
    tx0 = (E.x0 - J.V.vx) >> sx;
    tx1 = (E.x1 - J.V.vx) >> sx;
    ty0 = (E.y0 - J.V.vy) >> sy;
    ty1 = (E.y1 - 1 - J.V.vy) >> sy;
    return make_uint2((uint32_t)tx0 | ((uint32_t)ty0 << 16), (uint32_t)tx1 | ((uint32_t)ty1 << 16));
}

// ------------------------------------------------------ tile count scan
// Exclusive scan of the tile counts by one block, in passes of NT x
// SCAN_PER tiles: each thread loads its SCAN_PER consecutive counts at once
// (one memory round trip per pass), the block scans the per-thread sums
// (shuffles within each wave, then the wave totals), and each thread writes
// its tiles' offsets (densely: the fill ranks, zeroed by k_vertex, sit in
// the padded lines and are added to the offsets by k_bin_fill).
#define SCAN_PER 16
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v)
{
    const int lane = __lane_id();
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d);
        if (lane >= d)
            v += o;
    }
    return v;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o);
    return v;
}

// Claim order of the raster's tiles: largest bin counts first (a counting
// sort on a logarithmic bucket of the count, four buckets per power of
// two), so that the costliest tiles start first and the last ones to start
// are cheap -- the persistent raster's makespan then comes close to its
// mean load instead of the heaviest tile started last.
#define SW_ORDER_BUCKETS 128
static_assert(SW_ORDER_BUCKETS == 2 * 64, "the bucket scan takes two buckets per lane of one wave");
__device__ __forceinline__ uint32_t count_bucket(uint32_t c)
{
    if (c < 4)
        return c;
    const uint32_t e = 31u - (uint32_t)__clz(c);   // >= 2
    return 4u * (e - 1u) + ((c >> (e - 2u)) & 3u);   // <= 123
}

// The counts of tiles i * step + first for SCAN_PER consecutive i from i0 on
// (zero past n), read with
// device-scope atomic loads (the counts were added at the memory side in
// this same kernel: an XCD's L2 may hold older lines), all issued before
// the first is used.
__device__ __forceinline__ void load_counts(const BatchDev &B, uint32_t i0, uint32_t n, uint32_t (&v)[SCAN_PER],
                                            uint32_t step = 1, uint32_t first = 0)
{
#pragma unroll
    for (int k = 0; k < SCAN_PER; k++)
        v[k] = i0 + k < n ? __hip_atomic_load(&B.tile_count[(size_t)((i0 + k) * step + first) * SW_TILE_PAD],
                                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                          : 0u;
}

// The exclusive scan of the tile counts into the bin offsets, by one block
// of NT threads.
template <int NT>
__device__ void scan_offsets(const BatchDev &B)
{
    constexpr int NW = NT / 64;
    __shared__ uint32_t wsum[NW];
    __shared__ uint32_t s_carry;
    const uint32_t n = B.n_tiles;
    const int lane = __lane_id(), wave = threadIdx.x >> 6;
    if (threadIdx.x == 0)
        s_carry = 0;
    __syncthreads();
    uint32_t v[SCAN_PER];
    for (uint32_t base = 0; base < n; base += (uint32_t)NT * SCAN_PER) {
        const uint32_t i0 = base + threadIdx.x * SCAN_PER;
        load_counts(B, i0, n, v);
        uint32_t sum = 0;
#pragma unroll
        for (int k = 0; k < SCAN_PER; k++)
            sum += v[k];
        const uint32_t incl = wave_incl_scan(sum);
        if (lane == 63)
            wsum[wave] = incl;
        __syncthreads();
        if (wave == 0) {
            const uint32_t w = lane < NW ? wsum[lane] : 0u;
            const uint32_t wi = wave_incl_scan(w);
            if (lane < NW)
                wsum[lane] = wi - w;   // exclusive prefix of the wave totals
        }
        __syncthreads();
        const uint32_t carry = s_carry;
        uint32_t run = carry + wsum[wave] + incl - sum;
#pragma unroll
        for (int k = 0; k < SCAN_PER; k++) {
            if (i0 + k < n) {
                B.tile_offset[i0 + k] = run;
                run += v[k];
            }
        }
        __syncthreads();   // everyone has read s_carry and wsum
        if (threadIdx.x == NT - 1)
            s_carry = run;   // the last thread's running sum ends the pass
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        B.tile_offset[n] = s_carry;
        B.ctr[SW_CTR_TOTAL] = s_carry;   // total bin entries
    }
}

// The raster's claim order, by SW_RASTER_QUEUES blocks of NT threads, block q
// for the tiles that are q mod SW_RASTER_QUEUES: one queue each, and an
// eighth of the counter lines to read (a block reads a line every 2.5 ns or
// so: one block for 8,160 tiles took 42 us).  A queue's items are sorted by
// a log bucket of their bin counts, the largest bucket first (order within a
// bucket is arbitrary: the raster's result does not depend on the claim
// order), then come its empty tiles.
// A tile of more than B.split entries is SW_BANDS items, a band of its rows
// each, so that the replay of a crowded tile -- a chain of 10 to 40 entries
// a lane -- is spread over several workgroups; an entry outside a band's
// rows costs little there.  Tiles without entries, where no job has big
// triangles either, are kept apart: the raster fills them without a claim
// each.
// Place j of queue q is slot 8 j + q; four slots lie in each tile's counter
// line, which has room (a tile is at most SW_BANDS items).
static_assert(SW_BANDS == 4 && SW_TILE_PAD >= 8, "four slots a counter line");
__device__ __forceinline__ uint32_t *item_slot(const BatchDev &B, uint32_t p)
{
    return B.tile_count + (size_t)(p >> 2) * SW_TILE_PAD + 4 + (p & 3);
}
template <int NT>
__device__ void order_tiles(const BatchDev &B, uint32_t queue)
{
    constexpr uint32_t Q = SW_RASTER_QUEUES;
    __shared__ uint32_t s_hist[SW_ORDER_BUCKETS], s_big;
    const uint32_t n = B.n_tiles > queue ? (B.n_tiles - 1u - queue) / Q + 1u : 0u;
    const int lane = __lane_id(), wave = threadIdx.x >> 6;
    if (threadIdx.x == 0)
        s_big = 0;
    for (int b = threadIdx.x; b < SW_ORDER_BUCKETS; b += NT)
        s_hist[b] = 0;
    __syncthreads();
    uint32_t big = 0;
    for (uint32_t j = threadIdx.x; j < B.n_jobs; j += NT)
        big |= B.ctr[SW_CTR_BIG0 + j];
    if (big)
        s_big = 1;
    auto bands = [&](uint32_t c) { return c > B.split ? (uint32_t)SW_BANDS : 1u; };
    uint32_t v[SCAN_PER];
    for (uint32_t base = 0; base < n; base += (uint32_t)NT * SCAN_PER) {
        const uint32_t i0 = base + threadIdx.x * SCAN_PER;
        load_counts(B, i0, n, v, Q, queue);
#pragma unroll
        for (int k = 0; k < SCAN_PER; k++)
            if (i0 + k < n)
                atomicAdd(&s_hist[count_bucket(v[k] / bands(v[k]))], bands(v[k]));
    }
    __syncthreads();
    // first place of each bucket, the largest bucket first: wave 0 scans the
    // buckets in descending order, two per lane; the last bucket holds the
    // empty tiles
    if (wave == 0) {
        const int b0 = SW_ORDER_BUCKETS - 1 - 2 * lane, b1 = b0 - 1;
        const uint32_t h0 = s_hist[b0], h1 = s_hist[b1];
        const uint32_t incl = wave_incl_scan(h0 + h1);
        s_hist[b0] = incl - h0 - h1;
        s_hist[b1] = incl - h1;
        if (lane == 63) {
            const uint32_t items = s_big ? incl : incl - h1;
            B.ctr[SW_CTR_ITEMS + 2 * queue] = items;
            B.ctr[SW_CTR_ITEMS + 2 * queue + 1] = incl - items;
        }
    }
    __syncthreads();
    // every tile takes the next places of its bucket; with one pass the
    // counts are still in registers
    for (uint32_t base = 0; base < n; base += (uint32_t)NT * SCAN_PER) {
        const uint32_t i0 = base + threadIdx.x * SCAN_PER;
        if (n > (uint32_t)NT * SCAN_PER)
            load_counts(B, i0, n, v, Q, queue);
#pragma unroll
        for (int k = 0; k < SCAN_PER; k++)
            if (i0 + k < n) {
                const uint32_t nb = bands(v[k]), tile = (i0 + k) * Q + queue;
                const uint32_t at = atomicAdd(&s_hist[count_bucket(v[k] / nb)], nb);
                if (nb == 1)
                    *item_slot(B, at * Q + queue) = tile;
                else
                    for (uint32_t q = 0; q < SW_BANDS; q++)
                        *item_slot(B, (at + q) * Q + queue) = tile | (q + 1) << SW_ITEM_BAND;
            }
    }
}

// ------------------------------------------------------------- k_front
// Tiles whose lanes take a triangle each (raster_tile): the most pixels that
// one lane replays on its own; smallest chunk (pixels) of a listed triangle.
#define SW_LANE_PIXELS 96
#define SW_CHUNK_PIXELS 8
// Per triangle, in one pass: the visibility marks (renderer.cpp:83-185: a
// triangle passing the frustum test and double-sided or front-facing marks
// its three vertices), its tile rectangle (conservative but never too small:
// rows exact from ceil of vertex y, clipped to the viewport; columns the
// vertex x range widened by the DDA's worst-case accumulated rounding;
// near-clipped or non-finite triangles take the exact fill_triangle path)
// and one bin count per covered tile.  Whether a triangle is drawn depends
// on marks other triangles set in this same pass, so every triangle with a
// rectangle is counted here; k_bin_fill, which runs after all marks are
// set, places only triangles whose three vertices are marked, and the
// raster checks the marks of big-list triangles.  The last block to finish
// gives the tiles that k_bin_fill will fill their bin offsets (the claim order
// is written by k_bin_fill's first blocks, off this kernel's critical path).
// With the fixed layout those are the tiles that passed their capacity, listed
// by the one entry that found each full; the others keep their entries where
// they are.  (Scanning every tile's count for the sake of a few took one
// workgroup 18 us for 8,160 tiles, placing every triangle of such a job again
// 10 to 15, and noting the overflow with two read-modify-writes a wave 23 on
// four 1920x1080 views of 500,000 stacked triangles: k_front + k_bin_fill 85 +
// 35 us, 45 + 24 now; the 999,698-triangle field at 3840x2160 51 + 25 and 33 +
// 13.  64 times a tile's share instead of 16 gained as much, at 240 MB a
// buffer set and 0.1 ms of a first frame.)
__global__ __launch_bounds__(256) void k_front(BatchDev B, const JobDev *__restrict__ jobs)
{
    const int jidx = find_job<JT>(B, jobs, blockIdx.x);
    const JobDev &J = jobs[jidx];
    const uint32_t t = (blockIdx.x - J.tblock0) * 256u + threadIdx.x;
    uint32_t big = 0;
    int ntiles = 0, tx0 = 0, tx1 = 0, ty0 = 0;
    bool self_marked = false;   // marked its own vertices: drawn whatever other triangles do
    bool large = false;         // may cover more than SW_LANE_PIXELS pixels of a tile
    if (t < J.n_tris) {
        const uint4 id = tri_ids(J.tri, t);
        const uint32_t i0 = id.x, i1 = id.y, i2 = id.z;
        const f3 a = ld3(J.ndc, i0), b = ld3(J.ndc, i1), c = ld3(J.ndc, i2);
        if (inside_frustum(a, b, c) &&
            (ro(J.prims)[id.w].double_sided || cross_z_sign(b - a, c - a, 1))) {
            J.yes[i0] = 1;
            J.yes[i1] = 1;
            J.yes[i2] = 1;
            self_marked = true;
        }
        Extent E;
        bool exact;
        uint32_t drawn;
        bool have = quick_extent(J, frustum_to_screen(J.V, a), frustum_to_screen(J.V, b),
                                 frustum_to_screen(J.V, c), E, drawn, exact);
        if (exact)
            have = exact_extent(J, t, E, drawn);
        uint2 r = make_uint2(RECT_EMPTY, 0);
        if (have) {
            int ty1;
            r = tile_rect(J, E, tx0, tx1, ty0, ty1);
            large = (int64_t)(E.x1 - E.x0) * (E.y1 - E.y0) > SW_LANE_PIXELS;
            ntiles = (tx1 - tx0 + 1) * (ty1 - ty0 + 1);
            if (ntiles > (int)B.big_tiles) {
                ntiles = 0;
                big = 1;
            }
        }
        J.rect[t] = r;
    }
    // big-list append, one atomic per wave (all lanes of a block share the job)
    {
        const uint32_t pos = wave_add<true>(B.ctr + SW_CTR_BIG0, (uint32_t)jidx, big != 0);
        if (big)
            J.big[pos] = t;
    }
    // one aggregated atomic per distinct tile per wave and round; with a
    // tile capacity the count's old value places the entry
    for (int k = 0; __any(k < ntiles); k++) {
        const bool act = k < ntiles;
        uint32_t key = 0;
        if (act) {
            const int w = tx1 - tx0 + 1;
            const int ky = k == 0 ? 0 : k / w, kx = k == 0 ? 0 : k % w;   // k is the same in every lane
            key = J.tile_base + (ty0 + ky) * J.tiles_x + (tx0 + kx);
        }
        if (B.fixed) {
            const uint32_t rank = wave_add<true>(B.tile_count, key * SW_TILE_PAD, act);
            if (act && rank < J.tile_cap)
                B.bins_fixed[J.bin_base + (size_t)(key - J.tile_base) * J.tile_cap + rank] =
                    t | (self_marked ? 0u : SW_BIN_CHECK) | (large ? SW_BIN_LARGE : 0u);
            if (act && rank == J.tile_cap) {
                // one entry of a tile finds it full: the tile is listed for
                // the filled layout and its job noted (seen by other XCDs)
                const uint32_t i = atomicAdd(B.ctr + SW_CTR_OVERFLOW, 1u);
                __hip_atomic_store(&B.tile_count[(size_t)i * SW_TILE_PAD + 2], key, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(B.ctr + SW_CTR_BIG0 + B.n_jobs + jidx, 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        } else {
            wave_add<false>(B.tile_count, key * SW_TILE_PAD, act);
        }
    }
    // The last block to finish scans.  The counts are device-scope atomics,
    // performed at the memory side, not in an XCD's L2: each wave waits
    // for its own to complete before the block takes its ticket, and the
    // scan reads the counts with device-scope atomic loads.  (A device-scope
    // fence here would write back and invalidate every XCD's L2 per block.)
    // Tickets are taken in two levels (the blocks of group k = index mod
    // SW_TICKET_GROUPS, then the groups), so that no counter sees more than
    // about gridDim / SW_TICKET_GROUPS atomics.
    __shared__ uint32_t s_last;
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t G = gridDim.x, k = blockIdx.x % SW_TICKET_GROUPS;
        const uint32_t in_group = (G - 1u - k) / SW_TICKET_GROUPS + 1u;   // blocks k, k + 32, ... below G
        const uint32_t groups = G < SW_TICKET_GROUPS ? G : SW_TICKET_GROUPS;
        uint32_t last = 0;
        if (atomicAdd(B.ctr + SW_CTR_TICKETS + 32 * k, 1u) == in_group - 1u)
            last = atomicAdd(B.ctr + SW_CTR_TICKETS + 32 * SW_TICKET_GROUPS, 1u) == groups - 1u ? 1u : 0u;
        s_last = last;
    }
    __syncthreads();
    if (!s_last)
        return;
    // the offsets serve the filled layout only: of every tile, or of the full
    // ones listed above
    if (!B.fixed) {
        scan_offsets<256>(B);
        return;
    }
    const uint32_t full = __hip_atomic_load(B.ctr + SW_CTR_OVERFLOW, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __shared__ uint32_t s_next;
    if (threadIdx.x == 0)
        s_next = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < full; i += 256u) {
        const uint32_t g = __hip_atomic_load(&B.tile_count[(size_t)i * SW_TILE_PAD + 2], __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t n = __hip_atomic_load(&B.tile_count[(size_t)g * SW_TILE_PAD], __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
        B.tile_offset[g] = atomicAdd(&s_next, n);
    }
}

// ----------------------------------------------------------- k_bin_fill
// The first SW_RASTER_QUEUES blocks write the raster's claim order instead
// (the counts are final once k_front has ended): dispatched first, they run
// beside the fill, not after it.  Block b after them fills for triangle block
// b - SW_RASTER_QUEUES.
__global__ __launch_bounds__(256) void k_bin_fill(BatchDev B, const JobDev *__restrict__ jobs)
{
    if (blockIdx.x < SW_RASTER_QUEUES) {
        if (B.order)
            order_tiles<256>(B, blockIdx.x);
        return;
    }
    // k_front placed every entry of a job unless one of its tiles was full;
    // otherwise only the statistics, if asked for, are counted here
    const uint32_t blk = blockIdx.x - SW_RASTER_QUEUES;
    const int jidx = find_job<JT>(B, jobs, blk);
    const bool place = !B.fixed || B.ctr[SW_CTR_BIG0 + B.n_jobs + jidx] != 0;
    if (!place && !B.stats)
        return;
    const JobDev &J = jobs[jidx];
    const uint32_t t = (blk - J.tblock0) * 256u + threadIdx.x;
    int ntiles = 0, tx0 = 0, tx1 = 0, ty0 = 0;
    uint32_t drawn = 0, big = 0;
    if (t < J.n_tris) {
        const uint2 r = ro2(J.rect, t);
        const bool m = (r.x != RECT_EMPTY || B.stats) && marked(J, t);   // every mark is set by now
        if (r.x != RECT_EMPTY && m) {
            tx0 = r.x & 0xFFFF;
            ty0 = r.x >> 16;
            tx1 = r.y & 0xFFFF;
            const int ty1 = r.y >> 16;
            ntiles = (tx1 - tx0 + 1) * (ty1 - ty0 + 1);
            if (ntiles > (int)B.big_tiles) {
                ntiles = 0;
                big = 1;
            }
        }
        if (B.stats && m) {
            // drawn sub-triangles (fill_triangle_2 calls that find a scanline)
            const uint4 id = tri_ids(J.tri, t);
            const uint32_t i0 = id.x, i1 = id.y, i2 = id.z;
            Extent E;
            bool exact;
            quick_extent(J, frustum_to_screen(J.V, ld3(J.ndc, i0)), frustum_to_screen(J.V, ld3(J.ndc, i1)),
                         frustum_to_screen(J.V, ld3(J.ndc, i2)), E, drawn, exact);
            if (exact)
                exact_extent(J, t, E, drawn);
        }
    }
    uint32_t entries = 0;
    for (int k = 0; __any(k < ntiles); k++) {
        const bool act = k < ntiles;
        if (!place) {   // (wave-uniform)
            entries += act ? 1u : 0u;
            continue;
        }
        uint32_t key = 0;
        if (act) {
            const int w = tx1 - tx0 + 1;
            const int ky = k == 0 ? 0 : k / w, kx = k == 0 ? 0 : k % w;   // k is the same in every lane
            key = J.tile_base + (ty0 + ky) * J.tiles_x + (tx0 + kx);
            entries++;
        }
        // the entry's place: the tile's offset plus its rank among the tile's
        // entries so far; tiles whose fixed layout holds them have no offset
        // (their counts would tell as well, but lie on the lines the ranks'
        // atomics work on: 45 us instead of 24 for four views of stacked
        // triangles)
        const uint32_t off = act ? ro(B.tile_offset)[key] : SW_NO_OFFSET;
        const bool put = off != SW_NO_OFFSET;
        if (!__any(put))
            continue;
        const uint32_t rank = wave_add<true>(B.tile_cursor, key * SW_TILE_PAD, put);
        const uint32_t pos = off + rank;
        if (put && pos < B.bin_capacity)
            B.bins[pos] = t;
    }
    if (!B.stats)
        return;
    __shared__ uint32_t s_acc[3];
    if (threadIdx.x < 3)
        s_acc[threadIdx.x] = 0;
    __syncthreads();
    if (drawn)
        atomicAdd(&s_acc[0], drawn);
    if (entries)
        atomicAdd(&s_acc[1], entries);
    if (big)
        atomicAdd(&s_acc[2], big);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_acc[0])
            stat_add(B, SW_ST_DRAWN, s_acc[0]);
        if (s_acc[1])
            stat_add(B, SW_ST_BINS, s_acc[1]);
        if (s_acc[2])
            stat_add(B, SW_ST_BIG, s_acc[2]);
    }
}

// `by` divides by fdepth - 1 (the same for the whole job); `fast` when
// 1 <= fdepth - 1 <= 2^20, where FDiv's quotient equals '/' (the numerator
// t - 1 lies in [2^-23, fdepth - 1] on that branch).
__device__ __forceinline__ float blur_factor(float z, float fdist, float fdepth, float rmax, const FDiv &by,
                                             bool fast)
{
    float t = fabsf(fdist - z);
    // inv_lerp_clipped(1, fdepth, t)
    float x;
    if (1.0f == fdepth)
        x = 0.5f;
    else if (t <= 1.0f)
        x = 0.0f;
    else if (t >= fdepth)
        x = 1.0f;
    else
        x = fast ? by(t - 1.0f) : (t - 1.0f) / (fdepth - 1.0f);
    // lerp_clipped(0, rmax, x)
    if (x <= 0)
        return 0.0f;
    if (x >= rmax)
        return rmax;
    return 0.0f + rmax * x;
}

// What the depth-of-field pass reads of a pixel: whether its blur factor is
// nonzero, and its radius in the bits above.
__device__ __forceinline__ uint32_t dof_code(float z, float fdist, float fdepth, int rmax, const FDiv &by, bool fast)
{
    const float bf = blur_factor(z, fdist, fdepth, (float)rmax, by, fast);
    const int radius = min(max(cvtt(bf), 0), rmax);   // bf is in [0, rmax] for finite inputs
    return (bf != 0.0f ? 1u : 0u) | (uint32_t)radius << 1;
}

// ------------------------------------------------------------- k_raster
// One workgroup per screen tile.  Phase 1 replays every binned sub-triangle's
// DDA over the tile's rows and columns (exact float sequence) and keeps the
// minimum (z, draw sequence) per pixel with an LDS 64-bit atomic min.
// Phase 2 shades each pixel's winner at its own progress and writes colour,
// depth (and the winner's sequence) once, coalesced.
struct TileRect { int x0, y0, x1, y1; };   // [x0,x1) x [y0,y1), absolute pixels

// Rows [wy0, wy1) of the tile only, so that one large triangle can be split
// over several lanes; every row of the tile belongs to exactly one call.
// Fragment payloads: when a fragment becomes its pixel's current minimum,
// it records its shading inputs -- its progress u along the span and the
// row's side progresses pl, pr -- in three 64-bit slots of the pixel, each
// tagged with its draw sequence and the half and side-order flags (an
// aligned 64-bit LDS store is single-copy atomic).  The pixel's final
// winner became the minimum when it ran and wrote all three; a later store
// by a fragment it beat carries another tag.  So where all three tags name
// the final winner, the payload is the winner's own, and the shading needs
// no replay of its setup, rows or span; elsewhere (a race, a sequence of
// 2^25 or more: triangles from 2^24 on) the pixel is shaded the long way.
// Tag: the sequence (25 bits), then the sub-triangle's vertex order in
// fill_triangle_2 as (index of S.v[0], of S.v[1]) among the triangle's
// three vertices, 3 * p0 + p1 (15: a clip vertex is among them), whether it
// is inverted, the half and the side order.
#define SW_SLOT_SEQ 0x01FFFFFFu
#define SW_SLOT_NOPERM 15u
__device__ __forceinline__ uint32_t slot_code(const Setup &S, uint32_t i0, uint32_t i1, uint32_t i2)
{
    if (S.v[0].clip | S.v[1].clip | S.v[2].clip)
        return SW_SLOT_NOPERM | (S.inverted ? 16u : 0u);
    const uint32_t p0 = S.v[0].a == i0 ? 0u : S.v[0].a == i1 ? 1u : 2u;
    const uint32_t p1 = S.v[1].a == i0 ? 0u : S.v[1].a == i1 ? 1u : 2u;
    if (p0 == p1)   // repeated vertex ids: no single order to record
        return SW_SLOT_NOPERM | (S.inverted ? 16u : 0u);
    return 3u * p0 + p1 + (S.inverted ? 16u : 0u);
}
__device__ __forceinline__ void store_slots(unsigned long long *slots, int n, int i, uint32_t tag, float u, float pl,
                                            float pr)
{
    const uint64_t hi = (uint64_t)tag << 32;
    __hip_atomic_store(&slots[i], hi | __float_as_uint(u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_store(&slots[n + i], hi | __float_as_uint(pl), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_store(&slots[2 * n + i], hi | __float_as_uint(pr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void put_slots(unsigned long long *slots, int n, int i, uint32_t seq, uint32_t code,
                                          bool lower, bool lr, float u, float pl, float pr)
{
    if (seq > SW_SLOT_SEQ)
        return;
    store_slots(slots, n, i, seq | code << 25 | (lower ? 1u << 30 : 0u) | (lr ? 1u << 31 : 0u), u, pl, pr);
}

// c ? a : b, field by field: a select of whole structs would take their
// addresses and put the setup in private memory.
__device__ __forceinline__ Side pick(bool c, const Side &a, const Side &b)
{
    Side r;
    r.ratio = c ? a.ratio : b.ratio;
    r.x = c ? a.x : b.x;
    r.it.ta = c ? a.it.ta : b.it.ta;
    r.it.ts = c ? a.it.ts : b.it.ts;
    r.it.ba = c ? a.it.ba : b.it.ba;
    r.it.bs = c ? a.it.bs : b.it.bs;
    r.it.v0 = c ? a.it.v0 : b.it.v0;
    r.it.v1 = c ? a.it.v1 : b.it.v1;
    return r;
}

// Calls row(y, R) for every row y in [wy0, wy1) that fill_triangle_2 draws
// for S (renderer.cpp:462-558), R holding the row's sides, half and side
// order.  The upper half's rows [up_y0, up_y1) and the lower half's
// [lo_y0, lo_y1) are adjacent when both exist (up_y1 == lo_y0 == iy1), so
// one loop walks them: the long side has taken y - ysL steps at row y in
// either half (row_state's two counts agree), a short side y minus its
// half's first row, and at the switch the lower short side starts from its
// setup state -- the same adds in the same order as a per-half replay,
// with every lane of a wave in one loop over its own rows.
template <typename RowF>
__device__ __forceinline__ void walk_rows(const Setup &S, int wy0, int wy1, RowF row)
{
    const bool up = S.has_up && S.up_y1 > S.up_y0, lo = S.has_lo && S.lo_y1 > S.lo_y0;
    if (!up && !lo)
        return;
    const int ya = max(wy0, up ? S.up_y0 : S.lo_y0), yb = min(wy1, lo ? S.lo_y1 : S.up_y1);
    if (ya >= yb)
        return;
    Row R;
    R.lower = !(up && ya < S.up_y1);
    {
        Side lng = S.L, sh = pick(R.lower, S.Sl, S.Su);
        lng.steps(ya - S.ysL);
        sh.steps(ya - (R.lower ? S.lo_y0 : S.up_y0));
        R.lr = R.lower ? S.lr_lo : S.lr_up;
        R.left = pick(R.lr, sh, lng);
        R.right = pick(R.lr, lng, sh);
    }
    for (int y = ya; y < yb; y++) {
        if (!R.lower && y == S.up_y1) {   // into the lower half
            const Side lng = pick(R.lr, R.right, R.left);
            R.lower = true;
            R.lr = S.lr_lo;
            R.left = pick(R.lr, S.Sl, lng);
            R.right = pick(R.lr, lng, S.Sl);
        }
        row(y, R);
        R.left.steps(1);
        R.right.steps(1);
    }
}

// Any triangle: near-clipped (two sub-triangles), non-finite, of any size.
// Its fragments in rows [wy0, wy1) and columns [wx0, wx1) of the tile.
__device__ void raster_depth_any(const JobDev &J, uint32_t t, uint32_t i0, uint32_t i1, uint32_t i2, TileRect tr,
                                 int wy0, int wy1, int wx0, int wx1, unsigned long long *keys, int TW,
                                 uint32_t &frags, uint32_t &nans, unsigned long long *slots, int nslot)
{
    SubTri st[2];
    int ns = tri_subs_v<true>(J, i0, i1, i2, st);
#pragma unroll
    for (int s = 0; s < 2; s++) {
        Setup S;
        if (s >= ns || !setup_subtri(st[s], J.V, S))
            continue;
        const uint32_t seq = 2u * t + (uint32_t)s;
        const uint32_t code = slots ? slot_code(S, i0, i1, i2) : 0u;
        walk_rows(S, wy0, wy1, [&](int y, const Row &R) {
            Span sp;
            if (!span_of(R, J.V, sp))
                return;
            int xa = max(sp.x1, wx0), xb = min(sp.x2, wx1);
            if (xa >= xb)
                return;
            Interp q = sp.q;
            q.steps(xa - sp.x1);
            const int rowi = (y - tr.y0) * TW - tr.x0;
            unsigned long long *row = keys + rowi;
            for (int x = xa; x < xb; x++, q.step()) {
                const float u = q.u();
                float z = q.value(u);
                if (z < SW_NEAR)
                    continue;
                frags++;
                if (z != z) {
                    nans++;
                    continue;
                }
                if (__float_as_uint(z) >= SW_MAX_Z_BITS)
                    continue;
                const unsigned long long key = vis_key(z, seq);
                if (slots) {
                    if (key < atomicMin(&row[x], key))
                        put_slots(slots, nslot, rowi + x, seq, code, R.lower, R.lr, u, sp.pl, sp.pr);
                } else {
                    atomicMin(&row[x], key);
                }
            }
        });
    }
}

// The job of a tile, its fields not known to have been read before: what a
// later phase of the tile needs is then read when that phase begins, not
// carried in scalar registers (and spilled to vector lanes) through the
// phase before.
__device__ __forceinline__ const JobDev &reread(const JobDev *__restrict__ jobs, int j)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(j));
    j = __builtin_amdgcn_readfirstlane(j);
#endif
    return jobs[j];
}

// ------------------------------------------------- plain triangles
// Plain triangles -- every vertex in front of the near plane, no coordinate
// beyond 2^16, no depth beyond 2^20 and none more than 4 times another: all
// but a few -- take a replay of their own.  They have one sub-triangle
// without clip vertices, and every division on the way is in the range of
// rcp_rn and div_rn (core.h): screen coordinates are multiples of 2^-26 (a
// product near -m03 plus m03 >= 1/2), so heights and widths are zero or at
// least that; over at most 2^17 adds the interpolators stay within 5 % of
// the interval their ends span, so 1 / z stays positive and depths within a
// factor of 6 of each other.  Only a span's width and first displacement,
// differences of accumulated sums, are checked, per row.  Most entries are a
// pixel or two, so the setup counts: reciprocals of the depths come with the
// vertices, those of the heights serve slope and interpolator.  With the
// shading's short forms the 999,698-triangle 1920x1080 field takes 31 M VALU
// wave-instructions instead of 42 M and 88 us instead of 94 (what is left of
// its raster is latency), four 1920x1080 views of 500,000 stacked triangles
// 257 us instead of 316.
struct PVert { float x, y, z, iz; };   // screen x and y, z, 1 / z
struct PTri { PVert a, b, c; };
__device__ __forceinline__ bool is_plain(const PTri &T)
{
    const float zmin = fminf(T.a.z, fminf(T.b.z, T.c.z)), zmax = fmaxf(T.a.z, fmaxf(T.b.z, T.c.z));
    return (T.a.z >= SW_NEAR) & (T.b.z >= SW_NEAR) & (T.c.z >= SW_NEAR) & (zmax <= 0x1p20f) &
           (zmax <= 4.0f * zmin) & (fabsf(T.a.x) <= 0x1p16f) & (fabsf(T.b.x) <= 0x1p16f) &
           (fabsf(T.c.x) <= 0x1p16f) & (fabsf(T.a.y) <= 0x1p16f) & (fabsf(T.b.y) <= 0x1p16f) &
           (fabsf(T.c.y) <= 0x1p16f);
}
// Whether fill_triangle draws the triangle whole, from finite points whose
// rows and columns convert to int (plain triangles are among these).
__device__ __forceinline__ bool is_unclipped(const PTri &T)
{
    const float big = 0x1p30f;
    return (T.a.z >= SW_NEAR) & (T.b.z >= SW_NEAR) & (T.c.z >= SW_NEAR) & (fabsf(T.a.x) < big) &
           (fabsf(T.b.x) < big) & (fabsf(T.c.x) < big) & (fabsf(T.a.y) < big) & (fabsf(T.b.y) < big) &
           (fabsf(T.c.y) < big);
}

// What the replay reads of a tile's job, held for a whole tile.
struct TileView {
    const uint4 *tri;
    const float4 *ndc;
    const uint8_t *yes;
    float m00, m03, m11, m13;
    int vx, vy;
    TileRect tr;
};
__device__ __forceinline__ PVert tile_vertex(const TileView &W, uint32_t i)
{
    const float4 f = ro4(W.ndc, i);
    return {W.m00 * f.x + W.m03, W.m11 * f.y + W.m13, f.z, f.w};
}

// One side from vertex p to q, at the row m below p: Interp::init and
// displace with 1 / z at hand and the reciprocal of the height shared by the
// slope and the interpolator.
struct PSide { float x, ratio, ta, ts, ba, bs, v0, v1; };
__device__ __forceinline__ PSide plain_side(const PVert &p, const PVert &q, float m)
{
    const float d = q.y - p.y, r = rcp_rn(d);
    PSide s;
    s.ratio = div_rn(q.x - p.x, d, r);
    s.ts = q.iz * r;
    s.bs = (q.iz - p.iz) * r;
    s.ta = s.ts * m;
    s.ba = p.iz + s.bs * m;
    s.x = p.x + s.ratio * m;
    s.v0 = p.z;
    s.v1 = q.z - p.z;
    return s;
}
__device__ __forceinline__ void side_step(PSide &s)
{
    s.x += s.ratio;
    s.ta += s.ts;
    s.ba += s.bs;
}
__device__ __forceinline__ void side_steps(PSide &s, int n)
{
    int i = 0;
    for (; i + 4 <= n; i += 4) {
        side_step(s);
        side_step(s);
        side_step(s);
        side_step(s);
    }
    for (; i < n; i++)
        side_step(s);
}

// The fragments of plain triangle t (vertices i0, i1, i2) in rows [wy0, wy1)
// and columns [wx0, wx1) of the tile.
template <int TW, bool SLOTS>
__device__ __forceinline__ void plain_depth(const TileView &W, const PTri &T, uint32_t t, uint32_t i0, uint32_t i1,
                                            uint32_t i2, int wy0, int wy1, int wx0, int wx1,
                                            unsigned long long *keys, unsigned long long *slots, int nslot,
                                            uint32_t &frags, uint32_t &nans)
{
    const PVert a = T.a, b = T.b, c = T.c;
    // fill_triangle's facing (cross_z_sign, whose product is zero or at least
    // 2^-52 here) and vertex order: the z-sort (renderer.cpp:262-279) only
    // matters to the y-sort (:375-387) where two heights are equal
    const bool front = (b.x - a.x) * (c.y - a.y) - (b.y - a.y) * (c.x - a.x) < 0.0f;
    const bool ba = b.y < a.y, cb = c.y < b.y, ca = c.y < a.y;
    bool a0 = !ba & !ca, b0 = ba & !cb, a2 = ba & ca, b2 = !ba & cb;   // a, b first; a, b last
    if ((a.y == b.y) | (b.y == c.y) | (a.y == c.y)) {
        uint32_t o0 = 0, o1 = 1, o2 = 2, x;
        float z0 = a.z, z1 = b.z, z2 = c.z, y0 = a.y, y1 = b.y, y2 = c.y, f;
        auto swap01 = [&] { x = o0; o0 = o1; o1 = x; f = z0; z0 = z1; z1 = f; f = y0; y0 = y1; y1 = f; };
        auto swap12 = [&] { x = o1; o1 = o2; o2 = x; f = z1; z1 = z2; z2 = f; f = y1; y1 = y2; y2 = f; };
        if (z1 > z0) swap01();
        if (z2 > z1) swap12();
        if (z1 > z0) swap01();
        if (y1 < y0) swap01();
        if (y2 < y1) swap12();
        if (y1 < y0) swap01();
        a0 = o0 == 0;
        b0 = o0 == 1;
        a2 = o2 == 0;
        b2 = o2 == 1;
    }
    const bool a1 = !a0 & !a2, b1 = !b0 & !b2;
    auto sel = [](bool m0, bool m1, float u, float v, float w) { return m0 ? u : m1 ? v : w; };
    const PVert p0 = {sel(a0, b0, a.x, b.x, c.x), sel(a0, b0, a.y, b.y, c.y), sel(a0, b0, a.z, b.z, c.z),
                      sel(a0, b0, a.iz, b.iz, c.iz)},
                p1 = {sel(a1, b1, a.x, b.x, c.x), sel(a1, b1, a.y, b.y, c.y), sel(a1, b1, a.z, b.z, c.z),
                      sel(a1, b1, a.iz, b.iz, c.iz)},
                p2 = {sel(a2, b2, a.x, b.x, c.x), sel(a2, b2, a.y, b.y, c.y), sel(a2, b2, a.z, b.z, c.z),
                      sel(a2, b2, a.iz, b.iz, c.iz)};
    // fill_triangle_2: rows [ys, iy2) of the viewport, the short side
    // changing at iy1 (walk_rows; the tile's rows lie inside the viewport's)
    const int iy0 = (int)ceilf(p0.y), iy1 = (int)ceilf(p1.y), iy2 = (int)ceilf(p2.y);
    const int ys = max(iy0, W.vy), ya = max(wy0, ys), yb = min(wy1, iy2);
    if (ya >= yb)
        return;
    // tag of the payload slots (put_slots), without its row's bits
    const uint32_t seq = 2u * t;
    uint32_t tag0 = 0;
    if (SLOTS) {
        const uint32_t perm = 3u * (a0 ? 0u : b0 ? 1u : 2u) + (a1 ? 0u : b1 ? 1u : 2u);
        tag0 = ((i0 == i1) | (i1 == i2) | (i0 == i2) ? SW_SLOT_NOPERM : perm) + (front ? 0u : 16u);
        tag0 = seq | tag0 << 25;
    }
    const float m = (float)ys - p0.y;
    PSide L = plain_side(p0, p2, m), S = plain_side(p0, p1, m);
    const int yl = max(iy1, W.vy);
    const PSide Sl = plain_side(p1, p2, (float)yl - p1.y);
    bool lower = ya >= iy1, lr = L.ratio > S.ratio;
    const bool lr_lo = L.ratio < Sl.ratio;
    side_steps(L, ya - ys);
    if (lower) {
        S = Sl;
        lr = lr_lo;
    }
    side_steps(S, ya - (lower ? yl : ys));
    for (int y = ya; y < yb; y++) {
        if (!lower & (y == iy1)) {
            lower = true;
            lr = lr_lo;
            S = Sl;
        }
        // span_of: the row's columns, then its sides' progresses and depths
        const float lx = lr ? S.x : L.x, rx = lr ? L.x : S.x;
        const int x1 = max((int)ceilf(lx), W.vx);
        const int xa = max(x1, wx0), xb = min((int)ceilf(rx), wx1);
        if (xa < xb) {
            const float uL = div_rn(L.ta, L.ba, rcp_rn(L.ba)), uS = div_rn(S.ta, S.ba, rcp_rn(S.ba));
            const float zL = L.v0 + L.v1 * uL, zS = S.v0 + S.v1 * uS;
            const float pl = lr ? uS : uL, pr = lr ? uL : uS, zl = lr ? zS : zL, zr = lr ? zL : zS;
            const float dist = rx - lx, dx = (float)x1 - lx;
            Interp q;
            const bool fast = (dist >= 0x1p-20f) & ((dx == 0.0f) | (dx >= 0x1p-40f));
            if (fast) {
                const float as = rcp_rn(dist), iz2 = rcp_rn(zr);
                q.ba = rcp_rn(zl);
                q.v0 = zl;
                q.v1 = zr - zl;
                q.ts = iz2 * as;
                q.bs = (iz2 - q.ba) * as;
                q.ta = 0.0f;
            } else {
                q.init(dist, zl, zr);
            }
            q.displace(dx);
            q.steps(xa - x1);
            const int rowi = (y - W.tr.y0) * TW - W.tr.x0;
            const uint32_t tag = tag0 | (lower ? 1u << 30 : 0u) | (lr ? 1u << 31 : 0u);
            for (int x = xa; x < xb; x++, q.step()) {
                const float u = fast ? div_rn(q.ta, q.ba, rcp_rn(q.ba)) : q.u();
                const float z = q.value(u);
                if (z < SW_NEAR)
                    continue;
                frags++;
                if (!fast) {
                    if (z != z) {
                        nans++;
                        continue;
                    }
                    if (__float_as_uint(z) >= SW_MAX_Z_BITS)
                        continue;
                }
                const unsigned long long key = vis_key(z, seq);
                if (SLOTS) {
                    if (key < atomicMin(&keys[rowi + x], key) && seq <= SW_SLOT_SEQ)
                        store_slots(slots, nslot, rowi + x, tag, u, pl, pr);
                } else {
                    atomicMin(&keys[rowi + x], key);
                }
            }
        }
        side_step(L);
        side_step(S);
    }
}

// What the shading reads of a primitive.
struct PrimView {
    TexView X;        // its texture (pixel_shaders.cpp:288-302)
    uint32_t color;   // its material's colour
};
__device__ __forceinline__ PrimView prim_view(const JobDev &J, const PrimDev &P)
{
    PrimView V{{nullptr, P.color, 1, 1}, P.color};
    if (P.tex >= 0) {
        V.X.p = J.texels + P.texel;
        V.X.w = P.tw;
        V.X.h = P.th;
    }
    return V;
}
// Primitive i's view; a scene of one primitive reads it with scalar loads.
__device__ __forceinline__ PrimView prim_view(const JobDev &J, uint32_t i)
{
    if (J.n_prims == 1)
        return prim_view(J, PrimDev(ro(J.prims)[0]));
    return prim_view(J, PrimDev(ro(J.prims)[i]));
}

// A fragment to shade: the shading attributes of its sub-triangle's y-sorted
// vertices (v_world, normal_world, texture coordinates in texels, the last in
// the fourth lanes), its half and side order, the side progresses and its
// progress u along the span.
struct Frag {
    float4 w[3], n[3];
    bool lower, lr, inverted;
    float pl, pr, u;
    uint32_t prim;
};

// The attributes of sub-triangle vertex v; clip vertices are rebuilt as in
// renderer.cpp:290-297.
__device__ void vertex_attr(const JobDev &J, const PrimDev &P, const SVert &v, float4 &w, float4 &n)
{
    if (!v.clip) {
        w = ro4(J.world, v.a);
        n = ro4(J.nworld, v.a);
        return;
    }
    const f3 wa = ld3(J.world, v.a), wb = ld3(J.world, v.b);
    const f3 wc = wa + (wb - wa) * v.cut;
    const f2 ta = {ro(J.tu)[v.a], ro(J.tv)[v.a]}, tb = {ro(J.tu)[v.b], ro(J.tv)[v.b]};
    const f2 tc = ta + (tb - ta) * v.cut;
    f3 na = {ro(J.nx)[v.a], ro(J.ny)[v.a], ro(J.nz)[v.a]}, nb = {ro(J.nx)[v.b], ro(J.ny)[v.b], ro(J.nz)[v.b]};
    f3 nobj = (na.x == nb.x && na.y == nb.y && na.z == nb.z) ? na : normalize(na + (nb - na) * v.cut);
    const NodeDev N = ro(J.nodes)[P.node];
    const f3 nc = normal_world(N.RS, nobj);
    w = make_float4(wc.x, wc.y, wc.z, tc.x * (float)P.tw);
    n = make_float4(nc.x, nc.y, nc.z, tc.y * (float)P.th);
}
// A fragment from its replayed setup, row and span.
__device__ __forceinline__ void frag_of(const JobDev &J, uint32_t t, const Setup &S, const Row &R, const Span &sp,
                                        float u, Frag &F)
{
    F.prim = tri_ids(J.tri, t).w;
    const PrimDev P = ro(J.prims)[F.prim];
#pragma unroll
    for (int k = 0; k < 3; k++)
        vertex_attr(J, P, S.v[k], F.w[k], F.n[k]);
    F.lower = R.lower;
    F.lr = R.lr;
    F.inverted = S.inverted;
    F.pl = sp.pl;
    F.pr = sp.pr;
    F.u = u;
}

// The texture part of a shader kind: 0 the material colour, 1 nearest, 2
// bilinear.
__device__ __forceinline__ int texture_kind(int k)
{
    return (k == 1 || k == 3 || k == 7) ? 2 : (k == 2 || k == 4 || k == 6) ? 1 : 0;
}

// The colour of a fragment before lighting: the material colour, nearest
// texel or bilinear texel of the shader's texture part.  Its alpha is the
// fragment's alpha for every shader whose light part only scales b, g, r
// (a10, pixel_shaders.hpp:121-179) -- all but the light-only ones.
template <bool GENERIC>
__device__ __forceinline__ uint32_t frag_texture(const JobDev &J, const Frag &F, const RowEnds &E, uint32_t &oob)
{
    const int tk = GENERIC ? texture_kind(J.shader) : 2;
    const PrimView P = prim_view(J, F.prim);
    if (tk == 0)
        return P.color;
    const float su = E.along(F.u);
    const f2 tc = {RowVal(E, F.w[0].w, F.w[1].w, F.w[2].w).at(su), RowVal(E, F.n[0].w, F.n[1].w, F.n[2].w).at(su)};
    return tk == 1 ? nearest(P.X, tc) : bilinear(P.X, tc, oob);
}

// GENERIC: the job's shader is any SWEGL_SHADER_* kind, decoded into a light
// part (0 none, 1 flat, 2 phong) and a texture part; otherwise it is
// SWEGL_SHADER_PHONG_BILINEAR, the kernel variant the common case runs without
// the other branches.
template <bool GENERIC>
__device__ __forceinline__ uint32_t shade_frag(const JobDev &J, const Frag &F, uint32_t &oob)
{
    int lk = 2;
    bool combined = true;
    if (GENERIC) {
        const int k = J.shader;
        lk = (k == 1 || k == 2 || k == 9) ? 2 : (k == 3 || k == 4 || k == 8) ? 1 : 0;
        combined = k >= 1 && k <= 4;
    }
    const RowEnds E(F.lower, F.lr, F.pl, F.pr);
    const uint32_t color = frag_texture<GENERIC>(J, F, E, oob);
    if (GENERIC && lk == 0)
        return color;
    int32_t light;
    if (GENERIC && lk == 1) {
        light = flat_light(f3{F.w[0].x, F.w[0].y, F.w[0].z}, f3{F.w[1].x, F.w[1].y, F.w[1].z},
                           f3{F.w[2].x, F.w[2].y, F.w[2].z}, F.inverted, J.V.cam, J.ambient, J.sun, J.sun_I,
                           J.lights, (int)J.n_lights);
    } else {
        const float su = E.along(F.u);
        const f3 center = {RowVal(E, F.w[0].x, F.w[1].x, F.w[2].x).at(su),
                           RowVal(E, F.w[0].y, F.w[1].y, F.w[2].y).at(su),
                           RowVal(E, F.w[0].z, F.w[1].z, F.w[2].z).at(su)};
        f3 normal = {RowVal(E, F.n[0].x, F.n[1].x, F.n[2].x).at(su), RowVal(E, F.n[0].y, F.n[1].y, F.n[2].y).at(su),
                     RowVal(E, F.n[0].z, F.n[1].z, F.n[2].z).at(su)};
        // an inverted triangle's vertex normals are negated
        // (pixel_shaders.cpp:88-110): the interpolation only adds, subtracts
        // and scales them, so the sign is as well applied at its end
        if (F.inverted)
            normal = neg(normal);
        light = phong(center, normalize(normal), J.V.cam, J.ambient, J.sun, J.sun_I, J.lights, (int)J.n_lights);
    }
    return combined ? combine(color, light) : (uint32_t)light;
}

// The fragment of the winning draw sequence seq at pixel (x, y): the
// sub-triangle, row and span re-derived by the same replay that produced the
// winner, so every step succeeds; false only for a corrupted key.
__device__ __forceinline__ bool frag_replayed(const JobDev &J, uint32_t seq, int x, int y, Frag &F)
{
    const uint32_t t = seq >> 1, s = seq & 1u;
    SubTri st[2];
    Setup S;
    Row R;
    Span sp;
    if ((int)s >= tri_subs<true>(J, t, st))
        return false;
    SubTri one = st[0];   // a copy, not a runtime index: st stays in registers
    if (s)
        one = st[1];
    if (!setup_subtri(one, J.V, S, y) || !row_state(S, y, R) || !span_of(R, J.V, sp) || x < sp.x1 || x >= sp.x2)
        return false;
    Interp q = sp.q;
    q.steps(x - sp.x1);
    frag_of(J, t, S, R, sp, q.u(), F);
    return true;
}
template <bool GENERIC>
__device__ uint32_t shade_pixel(const JobDev &J, uint32_t seq, int x, int y, uint32_t &oob)
{
    Frag F;
    return frag_replayed(J, seq, x, y, F) ? shade_frag<GENERIC>(J, F, oob) : 0u;
}

// The fragment of an unclipped triangle from its recorded payload
// (put_slots): the vertices in fill_triangle_2's order, the half and side
// order, the side progresses and the span progress u.  id: the triangle's
// vertices and primitive.
__device__ __forceinline__ void frag_recorded(const JobDev &J, uint4 id, uint32_t tag, float u, float pl, float pr,
                                              Frag &F)
{
    const uint32_t code = (tag >> 25) & 31u, perm = code & 15u;
    // (p0, p1) of 3 * p0 + p1; p2 is the third
    const bool a0 = perm < 3u, b0 = perm < 6u, a1 = perm == 3u || perm == 6u, b1 = perm == 1u || perm == 7u;
    const uint32_t i0 = a0 ? id.x : b0 ? id.y : id.z, i1 = a1 ? id.x : b1 ? id.y : id.z;
    const uint32_t i2 = id.x ^ id.y ^ id.z ^ i0 ^ i1;   // three different ids
    F.w[0] = ro4(J.world, i0);
    F.n[0] = ro4(J.nworld, i0);
    F.w[1] = ro4(J.world, i1);
    F.n[1] = ro4(J.nworld, i1);
    F.w[2] = ro4(J.world, i2);
    F.n[2] = ro4(J.nworld, i2);
    F.lower = (tag >> 30) & 1u;
    F.lr = (tag >> 31) & 1u;
    F.inverted = (code & 16u) != 0;
    F.pl = pl;
    F.pr = pr;
    F.u = u;
    F.prim = id.w;
}

// Whether a tile's fragments record payload slots (put_slots, 24 bytes a
// pixel): up to 64x32 pixels, whose 70 KB let two workgroups of 512 threads
// on a CU.
constexpr bool raster_slots(int tw, int th) { return tw * th <= 2048; }
// Threads of a tile's workgroup.  Four waves fit on a SIMD at the raster's 128
// registers whatever the workgroup's size; with more, smaller workgroups on a
// CU one shades while another waits on its replay's loads and barriers
// (32x32 tiles of the 999,698-triangle field at 3840x2160: 235 us with 256
// threads, 290 with 512, 462 with 1,024).  Above 32x32 the slots' LDS allows
// two workgroups, of 512.
constexpr int raster_threads(int tw, int th) { return tw * th > 1024 ? 512 : 256; }

template <int TW, int TH, int NT, bool GENERIC>
__device__ __forceinline__ uint32_t raster_tile(const BatchDev &B, const JobDev *__restrict__ jobs, uint32_t item,
                                                unsigned long long *keys, uint32_t *s_cnt,
                                                unsigned long long *slots, uint32_t *claim)
{
    item = (uint32_t)__builtin_amdgcn_readfirstlane((int)item);   // the same in every lane
    const uint32_t band = B.split == 0xFFFFFFFFu ? 0u : item >> SW_ITEM_BAND;
    const uint32_t g = band ? item & ((1u << SW_ITEM_BAND) - 1u) : item;
    constexpr int NSLOT = TW * TH;
    constexpr bool SLOTS = raster_slots(TW, TH);
    const int jidx = find_job<JTILE>(B, jobs, g);
    const JobDev &J = jobs[jidx];
    const int lt = (int)(g - J.tile_base);
    const int tx = lt % J.tiles_x, ty = lt / J.tiles_x;
    TileRect tr;
    tr.x0 = J.V.vx + tx * TW;
    tr.y0 = J.V.vy + ty * TH;
    tr.x1 = min(tr.x0 + TW, J.V.vx + J.V.vw);
    tr.y1 = min(tr.y0 + TH, J.V.vy + J.V.vh);
    // a band of the tile's rows: from here on a tile of its own, but for the
    // entries (split tiles are at least 32 rows high)
    int npix = TW * TH;
    if (band) {
        tr.y0 += (int)(band - 1u) * (TH / SW_BANDS);
        tr.y1 = min(tr.y0 + TH / SW_BANDS, tr.y1);
        npix = TW * (TH / SW_BANDS);
    }

    for (int i = threadIdx.x; i < npix; i += NT)
        keys[i] = SW_KEY_EMPTY;
    __syncthreads();

    uint32_t frags = 0, nans = 0, oob = 0;
    // Replay the tile's binned triangles, then the job's big triangles whose
    // rectangle touches this tile.  Up to NT / 2 of them are cut into chunks of
    // rows, or of parts of a row's columns, of about an equal number of pixels
    // (from the screen bounding boxes) and about as many as there are lanes, so
    // that a few large triangles occupy every lane.  With more, a lane takes a
    // triangle of its own, all rows, if it is plain and not one that covers
    // more than SW_LANE_PIXELS pixels of the tile, on which its lane would
    // spend several times what the others do; those are listed and cut up
    // after.  (Chunks of a fixed 64 pixels left a tile under 36 triangles 24 us
    // in this phase with 20-40 lanes busy, and one lane per triangle a tile
    // of 330 entries with one large among them 65 us.  The 640x480 cube's
    // raster 45 -> 31 us, the 800x600 demo scene's 78 -> 47; chunks of at
    // least 16 or 32 pixels: 34 and 40 us for the cube.  Parts of rows took
    // the cube from 28 to 24 us, where two triangles a tile kept 32 of 256
    // lanes busy with a row of 32 pixels each; lists of up to NT / 2 rather
    // than NT the demo scene from 42 to 36, of NT / 4 no further.)
    __shared__ uint32_t s_tri[NT], s_rows[NT], s_first[NT], s_wsum[NT / 64], s_n;
    // The tile's entries: placed by k_front in its job's fixed layout
    // (every triangle whose rectangle holds the tile; marks are checked
    // here), or, when they passed its capacity, by k_bin_fill at the offset
    // found for the tile (marked triangles only; the count also held unmarked
    // ones); then the job's big list.
    const uint32_t counted = B.tile_count[g * SW_TILE_PAD];
    const bool fixed = B.fixed != 0 && counted <= J.tile_cap;
    uint32_t nb;
    const uint32_t *bins;
    if (fixed) {
        nb = counted;
        bins = B.bins_fixed + J.bin_base + (size_t)lt * J.tile_cap;
    } else {
        nb = B.tile_cursor[g * SW_TILE_PAD];
        bins = B.bins + B.tile_offset[g];
    }
    const uint32_t entries = nb + B.ctr[SW_CTR_BIG0 + jidx];
    const int lane = __lane_id(), wave = threadIdx.x >> 6;
    TileView W;
    W.tri = J.tri;
    W.ndc = J.ndc;
    W.yes = J.yes;
    W.m00 = J.V.m00;
    W.m03 = J.V.m03;
    W.m11 = J.V.m11;
    W.m13 = J.V.m13;
    W.vx = J.V.vx;
    W.vy = J.V.vy;
    W.tr = tr;
    // Triangle t's vertices, and whether it is drawn: `check`, its marks are
    // still to be looked up.
    auto load = [&](uint32_t t, bool check, uint32_t &i0, uint32_t &i1, uint32_t &i2, PTri &T) {
        const uint4 id = tri_ids(W.tri, t);
        i0 = id.x;
        i1 = id.y;
        i2 = id.z;
        T.a = tile_vertex(W, i0);
        T.b = tile_vertex(W, i1);
        T.c = tile_vertex(W, i2);
        return !check || ((ro(W.yes)[i0] != 0) & (ro(W.yes)[i1] != 0) & (ro(W.yes)[i2] != 0));
    };
    // The tile rows a triangle covers and about how many of the tile's
    // pixels: rows [ceil(ymin), ceil(ymax)) are exactly the rows
    // fill_triangle_2 visits for an unclipped triangle; others (clipped,
    // non-finite) keep all rows and columns of the tile.
    auto rows_of = [&](const PTri &T, bool unclipped, int &ry0, int &ry1) {
        int w = W.tr.x1 - W.tr.x0;
        ry0 = W.tr.y0;
        ry1 = W.tr.y1;
        if (unclipped) {
            ry0 = max(ry0, (int)ceilf(fminf(T.a.y, fminf(T.b.y, T.c.y))));
            ry1 = min(ry1, (int)ceilf(fmaxf(T.a.y, fmaxf(T.b.y, T.c.y))));
            const int xa = max(W.tr.x0, (int)floorf(fminf(T.a.x, fminf(T.b.x, T.c.x))));
            const int xb = min(W.tr.x1, (int)ceilf(fmaxf(T.a.x, fmaxf(T.b.x, T.c.x))) + 1);
            w = max(xb - xa, 1);
        }
        return max(ry1 - ry0, 0) * w;
    };
    // Entry e of the tile: its triangle, whether its marks are still to be
    // looked up and whether it may cover many pixels (the filled layout holds
    // marked triangles and does not tell their sizes: there every triangle's
    // pixels are counted, without which a lane replays a large one alone,
    // 8,000 small triangles and 8 large ones in a 320x320 view 87 us by
    // swegl_render_noalloc, 67 with it); false: a big triangle elsewhere.
    auto entry = [&](uint32_t e, uint32_t &t, bool &check, bool &large) -> bool {
        if (e < nb) {
            const uint32_t k = ro(bins)[e], flags = fixed ? k & (SW_BIN_CHECK | SW_BIN_LARGE) : 0u;
            t = k ^ flags;
            check = (flags & SW_BIN_CHECK) != 0;
            large = !fixed || (flags & SW_BIN_LARGE) != 0;
            return true;
        }
        const JobDev &B1 = reread(jobs, jidx);
        t = ro(B1.big)[e - nb];
        check = large = true;
        const uint2 r = ro2(B1.rect, t);
        return (tx >= (int)(r.x & 0xFFFF)) & (tx <= (int)(r.y & 0xFFFF)) & (ty >= (int)(r.x >> 16)) &
               (ty <= (int)(r.y >> 16));
    };
    const bool many = entries > NT / 2;
    uint32_t listed = entries;
    if (many) {
        if (threadIdx.x == 0)
            s_n = 0;
        __syncthreads();
        auto list = [&](uint32_t t) {
            const uint32_t at = atomicAdd(&s_n, 1u);
            if (at < (uint32_t)NT)
                s_tri[at] = t;
        };
        // The loads of an entry are a chain of three (entry, vertex ids,
        // vertices): the next entry's ids and the one after's entry are on
        // their way while this one is replayed.
        const uint32_t flags = fixed ? SW_BIN_CHECK | SW_BIN_LARGE : 0u;
        if (threadIdx.x < nb) {
            uint32_t e = threadIdx.x, k = ro(bins)[e], kn = ro(bins)[min(e + NT, nb - 1u)];
            uint32_t t = k & ~flags;
            const uint4 id0 = tri_ids(W.tri, t);
            uint32_t i0 = id0.x, i1 = id0.y, i2 = id0.z;
            for (;; e += NT) {
                PTri T;
                T.a = tile_vertex(W, i0);
                T.b = tile_vertex(W, i1);
                T.c = tile_vertex(W, i2);
                const uint32_t tn = kn & ~flags;
                const uint4 idn = tri_ids(W.tri, tn);
                const uint32_t n0 = idn.x, n1 = idn.y, n2 = idn.z;
                const uint32_t kn2 = ro(bins)[min(e + 2u * NT, nb - 1u)];
                const bool drawn = !(k & flags & SW_BIN_CHECK) ||
                                   ((ro(W.yes)[i0] != 0) & (ro(W.yes)[i1] != 0) & (ro(W.yes)[i2] != 0));
                // In a band most entries lie in other rows, which only a plain
                // triangle's vertices tell: a near-clipped one also covers
                // rows beyond its projected vertices.
                const bool plain = is_plain(T);
                const bool here = !band || !plain || !(fmaxf(T.a.y, fmaxf(T.b.y, T.c.y)) <= (float)W.tr.y0 ||
                                                       fminf(T.a.y, fminf(T.b.y, T.c.y)) > (float)(W.tr.y1 - 1));
                if (drawn && here) {
                    int ry0, ry1;
                    if (!plain ||
                        ((!fixed || (k & SW_BIN_LARGE)) && rows_of(T, true, ry0, ry1) > SW_LANE_PIXELS))
                        list(t);
                    else
                        plain_depth<TW, SLOTS>(W, T, t, i0, i1, i2, W.tr.y0, W.tr.y1, W.tr.x0, W.tr.x1, keys, slots, NSLOT,
                                               frags, nans);
                }
                if (e + NT >= nb)
                    break;
                k = kn;
                t = tn;
                i0 = n0;
                i1 = n1;
                i2 = n2;
                kn = kn2;
            }
        }
        for (uint32_t e = nb + threadIdx.x; e < entries; e += NT) {
            uint32_t t;
            bool check, large;
            if (entry(e, t, check, large) && marked(reread(jobs, jidx), t))
                list(t);
        }
        __syncthreads();
        listed = s_n;
    }
    // The listed triangles, NT at a time.  More than NT listed out of many
    // are found again among the entries.
    const bool again = many && listed > (uint32_t)NT;
    const uint32_t last = again ? entries : listed;
    for (uint32_t base = 0; base < last; base += NT) {
        uint32_t t = 0, area = 0;
        int ry0 = tr.y0, ry1 = tr.y0;
        bool plain = false;
        if (base + threadIdx.x < last) {
            uint32_t i0, i1, i2;
            bool check = false, large = true, have = true;
            PTri T;
            if (many && !again)
                t = s_tri[threadIdx.x];
            else
                have = entry(base + threadIdx.x, t, check, large);
            if (have && load(t, check, i0, i1, i2, T)) {   // unmarked: no chunks
                plain = is_plain(T);
                // Not plain but unclipped: its own rows, unless there are
                // enough of them for every lane, where chunks by their sizes
                // cost more than the whole tile for each (600 triangles
                // reaching far outside a 320x320 view 54 -> 40 us; 2,500 of
                // depths far apart in a 64x64 view 58, 73 with their rows).
                area = (uint32_t)rows_of(T, again ? plain : is_unclipped(T), ry0, ry1);
                if (again && base + threadIdx.x < nb && plain && !(large && area > SW_LANE_PIXELS))
                    area = 0;   // done above
            }
        }
        auto block_total = [&] {
            uint32_t n = 0;
            for (int k = 0; k < NT / 64; k++)
                n += s_wsum[k];
            return n;
        };
        // pixels of a chunk: an equal share of the list's for every lane
        const uint32_t sum = wave_sum(area);
        if (lane == 0)
            s_wsum[wave] = sum;
        __syncthreads();
        const uint32_t per = max(block_total() / (uint32_t)NT, (uint32_t)SW_CHUNK_PIXELS);
        const uint32_t rows = (uint32_t)(ry1 - ry0);
        // whole rows a chunk, or 2^cols parts of one
        uint32_t nch = area ? max((uint32_t)((float)area * __builtin_amdgcn_rcpf((float)per)), 1u) : 0u, cols = 0;
        if (nch > rows) {
            while (cols < 3 && rows << (cols + 1) <= nch)
                cols++;
            nch = rows << cols;
        }
        __syncthreads();   // s_wsum read, s_tri too
        // exclusive prefix of the chunk counts over the block
        const uint32_t incl = wave_incl_scan(nch);
        if (lane == 63)
            s_wsum[wave] = incl;
        s_tri[threadIdx.x] = t;
        s_rows[threadIdx.x] = (uint32_t)(ry0 - tr.y0) | ((uint32_t)(ry1 - tr.y0) << 8) | (nch << 16) |
                             cols << 28 | (plain ? 1u << 31 : 0u);
        __syncthreads();
        uint32_t before = 0;
        for (int k = 0; k < wave; k++)
            before += s_wsum[k];
        const uint32_t total = block_total();
        s_first[threadIdx.x] = before + incl - nch;
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < total; i += NT) {
            // the entry whose chunks contain item i: last k with s_first[k] <= i and chunks
            int lo = 0, hi = NT - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (s_first[mid] <= i)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            // s_first is non-decreasing and i < total, so entry lo has a chunk holding i
            // (an entry without chunks shares its s_first with the next entry)
            const uint32_t pk = s_rows[lo], lc = pk >> 28 & 7u, n = (pk >> 16 & 0xFFFu) >> lc, part = i - s_first[lo];
            const uint32_t ch = part >> lc, col = part & ((1u << lc) - 1u);
            const int r0 = tr.y0 + (int)(pk & 0xFF), nr = (int)((pk >> 8) & 0xFF) - (int)(pk & 0xFF);
            const float rn = __builtin_amdgcn_rcpf((float)n);   // tap_mean: nr, ch and n are at most 64
            const int wy0 = r0 + (int)tap_mean((uint32_t)nr * ch, rn), wy1 = r0 + (int)tap_mean((uint32_t)nr * (ch + 1), rn);
            const int wx0 = tr.x0 + (int)(col * TW >> lc), wx1 = min(tr.x0 + (int)((col + 1u) * TW >> lc), tr.x1);
            const uint32_t tt = s_tri[lo];
            uint32_t i0, i1, i2;
            PTri T;
            load(tt, false, i0, i1, i2, T);
            if (pk >> 31)
                plain_depth<TW, SLOTS>(W, T, tt, i0, i1, i2, wy0, wy1, wx0, wx1, keys, slots, NSLOT, frags, nans);
            else
                raster_depth_any(reread(jobs, jidx), tt, i0, i1, i2, tr, wy0, wy1, wx0, wx1, keys, TW, frags, nans,
                                 SLOTS ? slots : nullptr, NSLOT);
        }
        __syncthreads();   // the LDS tables are rewritten by the next NT
    }
    __syncthreads();

    // The claim of the next item is on its way while this one is shaded (a
    // claim is a round trip to the memory side, 2-6 us with all workgroups
    // claiming; between the items nothing of the workgroup ran meanwhile).
    uint32_t next = 0;
    if (claim && threadIdx.x == 0)
        next = atomicAdd(claim, 1u);
    const JobDev &K = reread(jobs, jidx);
    const float maxz = __uint_as_float(SW_MAX_Z_BITS);
    // the winner's vertex ids are loaded one pixel ahead
    auto winner_ids = [&](int i) {
        const unsigned long long k = i < npix ? keys[i] : SW_KEY_EMPTY;
        return k != SW_KEY_EMPTY ? tri_ids(K.tri, (uint32_t)k >> 1) : make_uint4(0, 0, 0, 0);
    };
    uint4 id = winner_ids(threadIdx.x);
    for (int i = threadIdx.x; i < npix; i += NT) {
        const uint4 id_next = winner_ids(i + NT);
        const int x = tr.x0 + (i % TW), y = tr.y0 + (i / TW);
        if (x < tr.x1 && y < tr.y1) {
            const unsigned long long k = keys[i];
            uint32_t color = 0;
            float z = maxz;
            uint32_t seq = 0xFFFFFFFFu;
            if (k != SW_KEY_EMPTY) {
                seq = (uint32_t)k;
                z = __uint_as_float((uint32_t)(k >> 32));
                Frag F;
                bool have = false;
                if (SLOTS) {
                    const unsigned long long a = slots[i], b = slots[NSLOT + i], c = slots[2 * NSLOT + i];
                    const uint32_t tag = (uint32_t)(a >> 32);
                    have = (tag == (uint32_t)(b >> 32)) & (tag == (uint32_t)(c >> 32)) & ((tag & SW_SLOT_SEQ) == seq) &
                           ((tag >> 25 & 15u) < 9u);
                    if (have)
                        frag_recorded(K, id, tag, __uint_as_float((uint32_t)a), __uint_as_float((uint32_t)b),
                                      __uint_as_float((uint32_t)c), F);
                }
                if (!have)
                    have = frag_replayed(K, seq, x, y, F);
                if (have)
                    color = shade_frag<GENERIC>(K, F, oob);
            }
            // with depth of field the colour waits for its code below
            if (K.dofa)
                keys[i] = (uint64_t)__float_as_uint(z) << 32 | color;
            else
                K.out_color[(int64_t)(y - K.out_oy) * K.out_pitch + (x - K.out_ox)] = color;
            const int64_t zo = (int64_t)(y - K.V.vy) * K.V.vw + (x - K.V.vx);
            K.zbuf[zo] = z;
            if (K.tid)
                K.tid[zo] = seq;
        }
        id = id_next;
    }
    // What the depth-of-field pass reads: b, g, r with dof_code above them,
    // and alpha in a plane of its own.  A loop of its own keeps its registers
    // out of the shading loop's peak.
    const JobDev &D = reread(jobs, jidx);
    if (D.dofa) {
        const FDiv dof_by(D.fdepth - 1.0f);
        const bool dof_fast = D.fdepth - 1.0f >= 1.0f && D.fdepth - 1.0f <= 0x1p20f;
        for (int i = threadIdx.x; i < npix; i += NT) {
            const int x = tr.x0 + (i % TW), y = tr.y0 + (i / TW);
            if (x >= tr.x1 || y >= tr.y1)
                continue;
            const unsigned long long k = keys[i];   // this thread's, written above
            const uint32_t color = (uint32_t)k;
            const uint32_t code =
                dof_code(__uint_as_float((uint32_t)(k >> 32)), D.fdist, D.fdepth, D.rmax, dof_by, dof_fast);
            D.out_color[(int64_t)(y - D.out_oy) * D.out_pitch + (x - D.out_ox)] = (color & 0xFFFFFFu) | code << 24;
            D.dofa[(int64_t)(y - D.V.vy) * D.V.vw + (x - D.V.vx)] = (uint8_t)(color >> 24);
        }
    }
    if (B.stats) {
        if (frags)
            atomicAdd(&s_cnt[0], frags);
        if (nans)
            atomicAdd(&s_cnt[1], nans);
        if (oob)
            atomicAdd(&s_cnt[2], oob);
    }
    return next;
}

// A tile without entries: the clear alone (viewport.cpp:88-113) and the
// depth-of-field code of max_z.
template <int TW, int TH, int NT>
__device__ __forceinline__ void fill_empty(const BatchDev &B, const JobDev *__restrict__ jobs, uint32_t g)
{
    const JobDev &J = jobs[find_job<JTILE>(B, jobs, g)];
    const int lt = (int)(g - J.tile_base), tx = lt % J.tiles_x, ty = lt / J.tiles_x;
    const float maxz = __uint_as_float(SW_MAX_Z_BITS);
    uint32_t code = 0;
    if (J.dofa) {
        const FDiv by(J.fdepth - 1.0f);
        const bool fast = J.fdepth - 1.0f >= 1.0f && J.fdepth - 1.0f <= 0x1p20f;
        code = dof_code(maxz, J.fdist, J.fdepth, J.rmax, by, fast);
    }
    for (int i = threadIdx.x; i < TW * TH; i += NT) {
        const int x = tx * TW + i % TW, y = ty * TH + i / TW;   // viewport-relative
        if (x >= J.V.vw || y >= J.V.vh)
            continue;
        J.out_color[(int64_t)(y + J.V.vy - J.out_oy) * J.out_pitch + (x + J.V.vx - J.out_ox)] = code << 24;
        const int64_t zo = (int64_t)y * J.V.vw + x;
        J.zbuf[zo] = maxz;
        if (J.tid)
            J.tid[zo] = 0xFFFFFFFFu;
        if (J.dofa)
            J.dofa[zo] = 0;
    }
}

// Persistent: each workgroup takes tiles from the batch's work queue until
// the queue passes the last tile, so tiles of many jobs share the machine.
// At most 128 VGPRs, so four waves fit on each SIMD (512 registers a lane);
// the shading path needs about that many and one more halves the overlap.
template <int TW, int TH, bool GENERIC>
__global__ __launch_bounds__(raster_threads(TW, TH)) __attribute__((amdgpu_waves_per_eu(4))) void
k_raster(BatchDev B, const JobDev *__restrict__ jobs)
{
    constexpr int NT = raster_threads(TW, TH);
    constexpr uint32_t Q = SW_RASTER_QUEUES, NONE = 0xFFFFFFFFu;
    __shared__ unsigned long long keys[TW * TH];
    __shared__ unsigned long long slots[raster_slots(TW, TH) ? 3 * TW * TH : 1];
    __shared__ uint32_t s_cnt[3];
    __shared__ uint32_t s_place;
    if (threadIdx.x < 3)
        s_cnt[threadIdx.x] = 0;
    // Items come from SW_RASTER_QUEUES queues (order_tiles), each running from
    // costly items to cheap ones and counting on its own cache line:
    // same-address atomics are serialised where they execute, so one shared
    // queue would make every claim wait for all others.  The first B.n_static
    // workgroups, those that are resident together, begin with the places of
    // their home queue (block index mod 8) that are theirs without a claim.
    // A workgroup drains its home queue, its next claim on its way while the
    // item before is shaded; then wave 0 reads the eight counters at once,
    // one per lane (each read is a round trip to the memory side, and they
    // are read only then: the claims of others wait behind them), and takes
    // from the nearest queue that is not exhausted.  Counters only grow, so a
    // queue seen exhausted stays so and every workgroup stops after at most
    // n_items + 8 claims in total.
    const uint32_t home = blockIdx.x % Q;
    bool home_live = true;   // wave 0: the home queue was not seen exhausted
    // wave 0: the next item's slot; `claimed`: this lane 0's count of its home
    // queue, already taken
    auto next_slot = [&](bool have, uint32_t claimed) {
        // lane k: queue home + k, its items, and how many of them were given
        // out without a claim (found again per claim: kept, they would cost
        // the raster registers)
        uint32_t lane = threadIdx.x;
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+v"(lane));
#endif
        const uint32_t myq = (home + lane) % Q, cnt = B.ctr[SW_CTR_ITEMS + 2 * myq];
        const uint32_t given = B.n_static > myq ? (B.n_static - 1u - myq) / Q + 1u : 0u;
        uint32_t *const ctr = &B.ctr[SW_CTR_QUEUE0 + 64 * myq];
        uint32_t slot = NONE;
        if (home_live) {
            if (threadIdx.x == 0) {
                const uint32_t j = given + (have ? claimed : atomicAdd(ctr, 1u));
                if (j < cnt)
                    slot = j * Q + myq;
            }
            slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)slot);
            home_live = slot != NONE;
        }
        while (slot == NONE) {
            const bool live = threadIdx.x < Q && given + __hip_atomic_load(ctr, __ATOMIC_RELAXED,
                                                                           __HIP_MEMORY_SCOPE_AGENT) < cnt;
            const uint64_t any = __ballot(live);
            if (!any)
                break;
            const int l = __ffsll((unsigned long long)any) - 1;
            if ((int)threadIdx.x == l) {
                const uint32_t j = given + atomicAdd(ctr, 1u);
                if (j < cnt)
                    slot = j * Q + myq;
            }
            slot = __shfl(slot, l);
        }
        return slot;
    };
    uint32_t slot = NONE;
    if (blockIdx.x < B.n_static) {
        if (blockIdx.x / Q < (uint32_t)__builtin_amdgcn_readfirstlane((int)B.ctr[SW_CTR_ITEMS + 2 * home]))
            slot = blockIdx.x;   // place blockIdx / 8 of queue blockIdx mod 8
        else
            home_live = false;
    }
    if (slot == NONE) {
        if (threadIdx.x < 64) {
            const uint32_t n = next_slot(false, 0);
            if (threadIdx.x == 0)
                s_place = n;
        }
        __syncthreads();
        slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_place);
    }
    while (slot != NONE) {
        const bool ahead = home_live;
        const uint32_t claimed = raster_tile<TW, TH, NT, GENERIC>(
            B, jobs, *ro(item_slot(B, slot)), keys, s_cnt, slots, ahead ? &B.ctr[SW_CTR_QUEUE0 + 64 * home] : nullptr);
        if (threadIdx.x < 64) {
            const uint32_t n = next_slot(ahead, claimed);
            if (threadIdx.x == 0)
                s_place = n;
        }
        __syncthreads();   // also: the item is done with its keys
        // (the next claim writes s_place behind the item's own barriers)
        slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_place);
    }
    // The empty tiles of the home queue (of every queue where there are fewer
    // workgroups than queues), SW_EMPTY_CLAIM at a time, by whoever is done: a
    // claim each would take longer than their stores (of the 8,160 tiles of
    // four 1920x1080 views of stacked clusters 5,881 are empty).
    for (uint32_t q = home; q < (gridDim.x < Q ? home + Q : home + 1u); q++) {
        const uint32_t k = q % Q;
        const uint32_t T = (uint32_t)__builtin_amdgcn_readfirstlane((int)B.ctr[SW_CTR_ITEMS + 2 * k]),
                       E = (uint32_t)__builtin_amdgcn_readfirstlane((int)B.ctr[SW_CTR_ITEMS + 2 * k + 1]);
        while (E) {
            __syncthreads();
            if (threadIdx.x == 0)
                s_place = atomicAdd(B.ctr + SW_CTR_EMPTYQ + 64 * k, (uint32_t)SW_EMPTY_CLAIM);
            __syncthreads();
            uint32_t c = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_place);
            if (c >= E)
                break;
            for (const uint32_t end = min(c + SW_EMPTY_CLAIM, E); c < end; c++)
                fill_empty<TW, TH, NT>(B, jobs, *ro(item_slot(B, (T + c) * Q + k)));
        }
    }
    __syncthreads();
    if (B.stats && threadIdx.x == 0) {
        if (s_cnt[0])
            stat_add(B, SW_ST_FRAGMENTS, s_cnt[0]);
        if (s_cnt[1])
            stat_add(B, SW_ST_NAN, s_cnt[1]);
        if (s_cnt[2])
            stat_add(B, SW_ST_OOB, s_cnt[2]);
    }
}

// ------------------------------------------------------- k_raster_layers
// One pixel's base and layers (renderer.cpp:486-550)
struct LayerPixel {
    float bz, lz[SW_MAX_LAYERS];
    uint32_t bc, bseq, lc[SW_MAX_LAYERS];
};

// The z test, shading and base or layer update of one fragment at a pixel
// (renderer.cpp:489-550); `shade` computes the fragment's colour.
template <typename ShadeF>
__device__ __forceinline__ void layer_update(LayerPixel &P, float z, uint32_t seq, int K, bool deferred,
                                             uint32_t &frags, uint32_t &nans, ShadeF shade)
{
    constexpr int KMAX = SW_MAX_LAYERS;
    const float maxz = __uint_as_float(SW_MAX_Z_BITS);
    if (z < SW_NEAR)
        return;
    frags++;
    if (z != z) {
        nans++;
        return;
    }
    if (z >= P.bz)
        return;
    const uint32_t color = shade();
    // deferred: the slots keep the fragment's sequence, shaded at the end
    const uint32_t keep = deferred ? seq : color;
    // the first layer that is empty or nearer than z (renderer.cpp:500-505)
    int at = K;
#pragma unroll
    for (int k = KMAX - 1; k >= 0; k--)
        if (k < K && (P.lz[k] == maxz || P.lz[k] < z))
            at = k;
    if ((color >> 24) == 255) {
        // opaque: the new base; layers behind it drop out (:506-522)
        P.bz = z;
        P.bc = keep;
        P.bseq = seq;
        float nz[KMAX];
        uint32_t nc[KMAX];
#pragma unroll
        for (int k = 0; k < KMAX; k++) {
            const int from = k + at;
            nz[k] = maxz;
            nc[k] = 0u;
#pragma unroll
            for (int m = 0; m < KMAX; m++)
                if (m == from && m < K) {
                    nz[k] = P.lz[m];
                    nc[k] = P.lc[m];
                }
        }
#pragma unroll
        for (int k = 0; k < KMAX; k++) {
            P.lz[k] = nz[k];
            P.lc[k] = nc[k];
        }
        return;
    }
    // transparent: insert at `at` (:523-550)
    bool all_used = false;
#pragma unroll
    for (int k = 0; k < KMAX; k++)
        if (k == K - 1)
            all_used = P.lz[k] != maxz;
    float cz = z;
    uint32_t cc = keep;
    if (all_used) {
        // shift toward layer 0: the new fragment lands at at-1, layer 0 falls out
#pragma unroll
        for (int k = KMAX - 1; k >= 0; k--)
            if (k < at) {
                const float tz = P.lz[k];
                const uint32_t tc = P.lc[k];
                P.lz[k] = cz;
                P.lc[k] = cc;
                cz = tz;
                cc = tc;
            }
    } else {
        // shift away from layer 0 up to the first empty layer
        bool done = false;
#pragma unroll
        for (int k = 0; k < KMAX; k++)
            if (!done && k >= at && k < K) {
                const float tz = P.lz[k];
                const uint32_t tc = P.lc[k];
                P.lz[k] = cz;
                P.lc[k] = cc;
                cz = tz;
                cc = tc;
                done = cz == maxz;
            }
    }
}

// A chunk entry's sub-triangle staged in LDS: the vertices after
// fill_triangle's z-sort when the triangle is drawn unclipped (the common
// case); clipped triangles are re-derived by the lanes that need them.
struct LayerSub {
    float sx[3], sy[3], sz[3];
    uint32_t a[3];
    uint32_t kind;   // 0: not drawn, 1: one unclipped sub-triangle (+2: front), 4: re-derive
};

// Viewports with transparency layers (renderer.cpp:486-550).  The layer
// updates depend on the order of the fragments at a pixel, so each 8x8 tile
// (one wave) applies its triangles in draw order: the tile's bin entries
// and the job's big triangles whose rectangle holds the tile are gathered in
// LDS and sorted by triangle index (bitonic sort; the index is the draw
// order).  A tile with more than SW_LAYER_LIST such entries walks all of the
// job's triangles instead, a chunk at a time through their tile rectangles,
// compacted in order.  Entries go in chunks of SW_LAYER_CHUNK (layer_chunk):
// each lane
// walks one entry's rows over the tile (the costly, independent part), then
// each lane takes one pixel through the chunk's fragments in order -- z test
// against the base, shade, then the base write (opaque, alpha 255) with the
// farther layers dropped, or the layer insertion (transparent).  The base and
// the K layers of each pixel live in registers.  At the end the lane writes
// the base colour, depth and sequence and the layers flattened into layer 0
// (viewport.cpp:80-84); k_tflatten/k_tcopy finish the flatten and
// post_shader_t's copy (viewport.cpp:53-67, post_shaders.hpp:22-47).
#define SW_LAYER_LIST 1024
#define SW_LAYER_CHUNK 64
__device__ __forceinline__ uint32_t blend_colors(uint32_t back, uint32_t front)
{
    // colors.cpp:39-57: alpha from the front, integer alpha union, channels
    // mixed in double and truncated to 8 bits
    const int a = (int)(front >> 24), ba = (int)(back >> 24);
    const uint32_t na = (uint32_t)(255 - ((255 - a) * (255 - ba) / 255));
    if (a == 255)
        return (front & 0xFFFFFFu) | (na << 24);
    if (a == 0)
        return (back & 0xFFFFFFu) | (na << 24);
    uint32_t out = na << 24;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const double v = (double)((back >> (8 * c)) & 0xFF) * ((256 - a) / 256.0) +
                         (double)((front >> (8 * c)) & 0xFF) * (a / 256.0);
        out |= (uint32_t)(uint8_t)(int)v << (8 * c);   // v in [0, 255]
    }
    return out;
}

// The fragments of triangle t's unclipped sub-triangle over the tile's rows
// [row0, row1) and columns [tx0, tx0 + TW): the same row walk and span
// stepping as raster_depth_any (renderer.cpp:462-558), writing each covered
// pixel's depth to z[py * TW + px] and its bit to the returned mask.  With
// `opaque`, also the bit of every covered pixel whose texture-part colour
// (frag_texture: material colour, nearest or bilinear texel) has alpha 255,
// from the same row and span state a re-derivation for that pixel gives.
template <bool GENERIC>
__device__ uint64_t layer_walk(const JobDev &J, uint32_t t, const SubTri &st, int tx0, int ty0, int row0, int row1,
                               float *z, uint64_t *opaque)
{
    constexpr int TW = SW_LAYER_TW;
    Setup S;
    if (!setup_subtri(st, J.V, S))
        return 0ull;
    // texture part of the colour (frag_texture)
    const int tk = GENERIC ? texture_kind(J.shader) : 2;
    const PrimView P = prim_view(J, tri_ids(J.tri, t).w);
    const TexView &X = P.X;
    f2 tc[3];
    uint64_t opq = 0ull;
    const bool textured = opaque != nullptr && tk != 0;
    if (textured) {
#pragma unroll
        for (int k = 0; k < 3; k++)
            tc[k] = f2{ro4(J.world, S.v[k].a).w, ro4(J.nworld, S.v[k].a).w};
    }
    const bool flat_opaque = (P.color >> 24) == 255;   // tk == 0: the material colour
    const int wy0 = ty0 + row0, wy1 = min(ty0 + row1, J.V.vy + J.V.vh), wx1 = min(tx0 + TW, J.V.vx + J.V.vw);
    uint64_t mask = 0ull;
    walk_rows(S, wy0, wy1, [&](int y, const Row &R) {
        Span sp;
        if (!span_of(R, J.V, sp))
            return;
        const int xa = max(sp.x1, tx0), xb = min(sp.x2, wx1);
        if (xa >= xb)
            return;
        Interp q = sp.q;
        q.steps(xa - sp.x1);
        const RowEnds E(R.lower, R.lr, sp.pl, sp.pr);
        RowVal tx, ty;
        if (textured) {
            tx = RowVal(E, tc[0].x, tc[1].x, tc[2].x);
            ty = RowVal(E, tc[0].y, tc[1].y, tc[2].y);
        }
        for (int x = xa; x < xb; x++, q.step()) {
            const int p = (y - ty0) * TW + (x - tx0);
            const float u = q.u();
            z[p] = q.value(u);
            mask |= 1ull << p;
            bool op = flat_opaque;
            if (textured) {
                const f2 at = {tx.at(E.along(u)), ty.at(E.along(u))};
                uint32_t no_count = 0;   // texel reads are counted where the survivors are shaded
                op = tk == 1 ? (nearest(X, at) >> 24) == 255
                             : bilinear_channel(bilinear_taps(X, at, no_count), 3) == 255;
            }
            opq |= (uint64_t)op << p;
        }
    });
    if (opaque)
        *opaque = opq;
    return mask;
}

// Apply the entries list[0, n) (n <= SW_LAYER_CHUNK, in draw order) to the
// tile.  Phase one, one lane per entry: the depth of every pixel the entry
// covers goes to LDS (s_z, 64 depths per entry, and a coverage mask).
// Phase two, one lane per pixel: the entries in order, each covered pixel's
// fragment applied to the pixel's base and layers; a fragment that passes the
// z test is shaded after setting its sub-triangle up again for its row.
// Near-clipped triangles (two sub-triangles or clip vertices) are set up by
// the pixel lanes themselves.
template <bool GENERIC>
__device__ __forceinline__ void layer_chunk(const JobDev &J, const uint32_t *list, uint32_t n, LayerSub *s_sub,
                                            float *s_z, uint64_t *s_mask, uint64_t *s_opq, int tx0, int ty0,
                                            int px, int py, bool mine, int K, bool deferred, LayerPixel &P,
                                            uint32_t &frags, uint32_t &nans, uint32_t &oob)
{
    constexpr int TW = SW_LAYER_TW, TH = SW_LAYER_TH;
    // With few entries, 2, 4 or 8 lanes share an entry's rows: what a lane
    // takes longest over are the replays from a large triangle's first row
    // and from each span's first pixel.
    const uint32_t sh = n <= 8 ? 3u : n <= 16 ? 2u : n <= 32 ? 1u : 0u;
    const uint32_t e = threadIdx.x >> sh, part = threadIdx.x & ((1u << sh) - 1u);
    if (threadIdx.x < n)
        s_mask[threadIdx.x] = s_opq[threadIdx.x] = 0ull;
    __syncthreads();
    if (e < n) {
        const uint32_t t = list[e];
        SubTri st[2];
        const int ns = tri_subs<true>(J, t, st);
        LayerSub &L = s_sub[e];
        uint64_t m = 0ull, o = 0ull;
        if (ns == 1 && !st[0].v[0].clip && !st[0].v[1].clip && !st[0].v[2].clip) {
            if (part == 0) {
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    L.sx[k] = st[0].v[k].s.x;
                    L.sy[k] = st[0].v[k].s.y;
                    L.sz[k] = st[0].v[k].s.z;
                    L.a[k] = st[0].v[k].a;
                }
                L.kind = st[0].front ? 3u : 1u;
            }
            m = layer_walk<GENERIC>(J, t, st[0], tx0, ty0, (int)(part * (TH >> sh)), (int)((part + 1) * (TH >> sh)),
                                    s_z + e * 64, deferred ? &o : nullptr);
        } else if (part == 0) {
            L.kind = ns == 0 ? 0u : 4u;
            m = ns == 0 ? 0ull : ~0ull;   // near-clipped: every pixel lane sets it up itself
        }
        if (m)
            atomicOr((unsigned long long *)&s_mask[e], (unsigned long long)m);
        if (o)
            atomicOr((unsigned long long *)&s_opq[e], (unsigned long long)o);
    }
    __syncthreads();
    const int x = tx0 + px, y = ty0 + py, p = py * TW + px;
    for (uint32_t i = 0; i < n && mine; i++) {
        if (!((s_mask[i] >> p) & 1ull))
            continue;
        const LayerSub &L = s_sub[i];
        const uint32_t tt = list[i];
        if (L.kind & 1u) {
            layer_update(P, s_z[i * 64 + p], 2u * tt, K, deferred, frags, nans, [&] {
                // deferred: only the alpha matters here, found by the walk
                if (deferred)
                    return ((s_opq[i] >> p) & 1ull) ? 0xFF000000u : 0u;
                SubTri st;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    st.v[k].s = f3{L.sx[k], L.sy[k], L.sz[k]};
                    st.v[k].a = st.v[k].b = L.a[k];
                    st.v[k].cut = 0.0f;
                    st.v[k].clip = 0;
                }
                st.front = (L.kind & 2u) != 0;
                Setup S;
                Row R;
                Span sp;
                // the walk above produced this fragment, so these succeed
                if (!setup_subtri(st, J.V, S, y) || !row_state(S, y, R) || !span_of(R, J.V, sp))
                    return 0u;
                Interp q = sp.q;
                q.steps(x - sp.x1);
                Frag F;
                frag_of(J, tt, S, R, sp, q.u(), F);
                return shade_frag<GENERIC>(J, F, oob);
            });
        } else if (L.kind == 4u) {
            SubTri st[2];
            const int ns = tri_subs<true>(J, tt, st);
#pragma unroll
            for (int sub = 0; sub < 2; sub++) {   // unrolled: st is indexed by constants
                if (sub >= ns)
                    break;
                Setup S;
                Row R;
                Span sp;
                if (!setup_subtri(st[sub], J.V, S, y) || !row_state(S, y, R) || !span_of(R, J.V, sp) ||
                    x < sp.x1 || x >= sp.x2)
                    continue;
                Interp q = sp.q;
                q.steps(x - sp.x1);
                const float u = q.u();
                layer_update(P, q.value(u), 2u * tt + (uint32_t)sub, K, deferred, frags, nans, [&] {
                    uint32_t no_count = 0;
                    Frag F;
                    frag_of(J, tt, S, R, sp, u, F);
                    return deferred ? frag_texture<GENERIC>(J, F, RowEnds(F.lower, F.lr, F.pl, F.pr), no_count)
                                    : shade_frag<GENERIC>(J, F, oob);
                });
            }
        }
    }
    __syncthreads();   // s_sub, s_z and s_mask are rewritten by the next chunk
}

template <bool GENERIC>
__global__ __launch_bounds__(SW_LAYER_THREADS) void k_raster_layers(BatchDev B, const JobDev *__restrict__ jobs)
{
    constexpr int TW = SW_LAYER_TW, TH = SW_LAYER_TH, KMAX = SW_MAX_LAYERS, NT = SW_LAYER_THREADS;
    static_assert(TW * TH == 64 && NT == 64, "the layer raster works on 64-pixel tiles, one wave each");
    constexpr uint32_t CH = SW_LAYER_CHUNK;
    __shared__ uint32_t s_list[SW_LAYER_LIST], s_wcount[NT / 64];
    __shared__ LayerSub s_sub[CH];
    __shared__ float s_z[CH * 64];
    __shared__ uint64_t s_mask[CH], s_opq[CH];
    const uint32_t g = blockIdx.x;
    const int jidx = find_job<JTILE>(B, jobs, g);
    const JobDev &J = jobs[jidx];
    const int lt = (int)(g - J.tile_base);
    const int tx = lt % J.tiles_x, ty = lt / J.tiles_x;
    const int tx0 = J.V.vx + tx * TW, ty0 = J.V.vy + ty * TH;
    // this lane's pixel
    const int px = (int)(threadIdx.x % TW), py = (int)(threadIdx.x / TW);
    const bool mine = tx0 + px < J.V.vx + J.V.vw && ty0 + py < J.V.vy + J.V.vh;
    const int K = J.layers;
    // every shader but the light-only ones takes its alpha from the texture
    // part: only the alpha is needed in order, the survivors are shaded last
    const bool deferred = !GENERIC || (J.shader != 8 && J.shader != 9);   // 8, 9: lights_flat, lights_phong alone
    const float maxz = __uint_as_float(SW_MAX_Z_BITS);
    LayerPixel P;
    P.bz = maxz;
    P.bc = 0u;
    P.bseq = 0xFFFFFFFFu;
#pragma unroll
    for (int k = 0; k < KMAX; k++) {
        P.lz[k] = maxz;
        P.lc[k] = 0u;
    }
    uint32_t frags = 0, nans = 0, oob = 0;
    const int lane = __lane_id();
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    // a drawn triangle (all three vertices marked) whose rectangle holds this tile
    auto covers = [&](uint32_t t) {
        const uint2 r = ro2(J.rect, t);
        return r.x != RECT_EMPTY && tx >= (int)(r.x & 0xFFFF) && tx <= (int)(r.y & 0xFFFF) &&
               ty >= (int)(r.x >> 16) && ty <= (int)(r.y >> 16) && marked(J, t);
    };
    const uint32_t nb = B.tile_cursor[g * SW_TILE_PAD], off = B.tile_offset[g];
    const uint32_t nbig = B.ctr[SW_CTR_BIG0 + jidx];
    // the tile's triangles: bin entries, then the job's big ones whose
    // rectangle holds this tile, while they fit in LDS
    bool listed = nb <= SW_LAYER_LIST;
    uint32_t total = 0;
    if (listed) {
        for (uint32_t e = threadIdx.x; e < nb; e += NT)
            s_list[e] = ro(B.bins)[off + e];
        total = nb;
        const int wave = (int)(threadIdx.x >> 6);
        for (uint32_t base = 0; base < nbig && listed; base += NT) {
            const uint32_t e = base + threadIdx.x;
            const uint32_t t = e < nbig ? ro(J.big)[e] : 0u;
            const bool cov = e < nbig && covers(t);
            const uint64_t bal = __ballot(cov);
            if (lane == 0)
                s_wcount[wave] = (uint32_t)__popcll(bal);
            __syncthreads();
            uint32_t before = 0, sum = 0;
            for (int k = 0; k < NT / 64; k++) {
                before += k < wave ? s_wcount[k] : 0u;
                sum += s_wcount[k];
            }
            const uint32_t at = total + before + (uint32_t)__popcll(bal & lt_mask);
            if (cov && at < SW_LAYER_LIST)
                s_list[at] = t;
            total += sum;
            listed = total <= SW_LAYER_LIST;   // the same for every lane
            __syncthreads();   // s_wcount is rewritten by the next pass
        }
    }
    if (listed) {
        // bitonic sort of the first n2 >= total entries (padding sorts last)
        uint32_t n2 = 1;
        while (n2 < total)
            n2 <<= 1;
        for (uint32_t e = total + threadIdx.x; e < n2; e += NT)
            s_list[e] = 0xFFFFFFFFu;
        __syncthreads();
        for (uint32_t k = 2; k <= n2; k <<= 1)
            for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                for (uint32_t i = threadIdx.x; i < n2; i += NT) {
                    const uint32_t o = i ^ j;
                    if (o > i) {
                        const uint32_t a = s_list[i], b = s_list[o];
                        if ((a > b) == ((i & k) == 0)) {
                            s_list[i] = b;
                            s_list[o] = a;
                        }
                    }
                }
                __syncthreads();
            }
    }
    // the tile's list, or, too long for LDS, every triangle of the job in draw
    // order, CH at a time (one loop: layer_chunk's code is there once)
    for (uint32_t pos = 0; pos < (listed ? total : J.n_tris); pos += CH) {
        const uint32_t *list = s_list;
        uint32_t n = 0;
        if (listed) {
            list += pos;
            n = min(CH, total - pos);
        } else {
            const int wave = (int)(threadIdx.x >> 6);
            const uint32_t t = pos + threadIdx.x;
            const bool cov = threadIdx.x < CH && t < J.n_tris && covers(t);
            const uint64_t bal = __ballot(cov);
            if (lane == 0)
                s_wcount[wave] = (uint32_t)__popcll(bal);
            __syncthreads();
            uint32_t before = 0;
            for (int k = 0; k < NT / 64; k++) {
                before += k < wave ? s_wcount[k] : 0u;
                n += s_wcount[k];
            }
            if (cov)
                s_list[before + (uint32_t)__popcll(bal & lt_mask)] = t;
            __syncthreads();
        }
        layer_chunk<GENERIC>(J, list, n, s_sub, s_z, s_mask, s_opq, tx0, ty0, px, py, mine, K, deferred, P, frags, nans,
                             oob);
    }
    if (mine && deferred) {
        // shade the base and the surviving layers (sequences in the slots)
        const int x = tx0 + px, y = ty0 + py;
        // (one copy of the shading's code for the base, k = K, and the layers)
        for (int k = K; k >= 0; k--) {
            uint32_t seq = P.bseq;
            bool used = P.bseq != 0xFFFFFFFFu;
#pragma unroll
            for (int m = 0; m < KMAX; m++)
                if (m == k && m < K) {
                    seq = P.lc[m];
                    used = P.lz[m] != maxz;
                }
            const uint32_t color = used ? shade_pixel<GENERIC>(J, seq, x, y, oob) : 0u;
            if (k == K)
                P.bc = color;
#pragma unroll
            for (int m = 0; m < KMAX; m++)
                if (m == k && m < K)
                    P.lc[m] = color;
        }
    }
    if (mine) {
        const int x = tx0 + px, y = ty0 + py;
        J.out_color[(int64_t)(y - J.out_oy) * J.out_pitch + (x - J.out_ox)] = P.bc;
        const int64_t zo = (int64_t)(y - J.V.vy) * J.V.vw + (x - J.V.vx);
        J.zbuf[zo] = P.bz;
        if (J.tid)
            J.tid[zo] = P.bseq;
        // layers 1..K-1 flattened into layer 0 (viewport.cpp:43-51, 80-82)
        uint32_t f = P.lc[0];
#pragma unroll
        for (int k = 1; k < KMAX; k++)
            if (k < K && (P.lc[k] >> 24) != 0)
                f = blend_colors(f, P.lc[k]);
        J.tflat[zo] = f;
    }
    if (B.stats) {
        // a wave sum, one atomic per counter and wave
        const uint32_t f = wave_sum(frags), nn = wave_sum(nans), o = wave_sum(oob);
        if (lane == 0) {
            if (f)
                stat_add(B, SW_ST_FRAGMENTS, f);
            if (nn)
                stat_add(B, SW_ST_NAN, nn);
            if (o)
                stat_add(B, SW_ST_OOB, o);
        }
    }
}

// viewport_t::flatten(layer 0) (viewport.cpp:53-67): layer 0 over the screen
// pixel at (i, j) from the surface's origin -- the reference ignores the
// viewport's offset here -- or the screen pixel where layer 0 is empty.
__global__ __launch_bounds__(256) void k_tflatten(BatchDev B, uint32_t job, const JobDev *__restrict__ jobs)
{
    const JobDev &J = jobs[job];
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    if (p >= (uint32_t)(J.V.vw * J.V.vh))
        return;
    const int i = (int)(p % (uint32_t)J.V.vw), j = (int)(p / (uint32_t)J.V.vw);
    const uint32_t back = J.surface[(int64_t)j * J.surface_pitch + i];
    const uint32_t f = J.tflat[p];
    J.tflat[p] = (f >> 24) != 0 ? blend_colors(back, f) : back;
}
// post_shader_t::shade with layers (post_shaders.hpp:22-47): layer 0 to the
// screen rows y + j, columns from 0 (the reference ignores the x offset).
__global__ __launch_bounds__(256) void k_tcopy(BatchDev B, uint32_t job, const JobDev *__restrict__ jobs)
{
    const JobDev &J = jobs[job];
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    if (p >= (uint32_t)(J.V.vw * J.V.vh))
        return;
    const int i = (int)(p % (uint32_t)J.V.vw), j = (int)(p / (uint32_t)J.V.vw);
    J.surface[(int64_t)(j + J.V.vy) * J.surface_pitch + i] = J.tflat[p];
}

// ---------------------------------------------------------------- k_dof
// Depth of field (build spec of post_shader_depth_box, post_shaders.hpp:51-131
// with remap_clipped, lerp.hpp:24-43): 64x32 output pixels per block, colour
// and blur factor of the tile plus a halo staged in LDS.
// LDS bytes of a k_dof<RMAX> workgroup: two tap words per cell of the
// output tile plus an RMAX halo on every side (30 KB for RMAX 8).
__host__ __device__ inline size_t dof_lds_bytes(int RMAX)
{
    return (size_t)(SW_DOF_TW + 2 * RMAX) * (SW_DOF_TH + 2 * RMAX) * 8;
}

// SW_DOF_NT threads as 64 columns x 8 rows.  Bound by the instructions a
// pixel and by one round of loads: at 3840x2160 with radii to 16 it takes
// 29 us (75 MB, 14 us of copy), 68 before; at 1920x1080 with radii to 8 10 us,
// 15 before; four such views 24, 39 before; a 1231x717 box 16, 22 before.  What
// it gained from: a row a wave (58 to 37 us at 3840x2160; a window dealt out
// cell by cell costs a division a cell), means from one reciprocal rather than
// a gathered table (37 to 29), one word a pixel, the taller tile.  A halo as
// wide as the tile's own largest radius was no faster: the radii are read
// before the halo then.
// Consecutive workgroups run on different XCDs (round robin over 8), so the
// job's tiles are dealt out in 8 contiguous runs, one per XCD: neighbouring
// tiles, whose halos overlap, then share that XCD's L2.  The raster left b, g, r and
// dof_code in one word a pixel -- whether it is an "unfocused" tap, and its
// clamped radius -- and alpha apart, which only copied pixels need.
// RMAX bounds the job's halo (the loads below are unrolled for it, and the
// LDS window has its pitch): the launch picks 8 when no job of the launch
// has a larger radius.  The halo's cells are much of the work, so the tile is
// 64x32 (1.9 cells a pixel at radius 8, 3.0 at 16; 64x16: 2.5 and 4.5, and 26
// us against 24 for four views, 38 against 29 at 3840x2160).  64x64 on
// 1,024 threads gains at radius 16 (26) and costs at 8.
// The window is loaded a row of the tile a wave, so that a row's address and
// its bounds are scalar: the tile's own rows, which the output needs in any
// case, the rows above and below it, and the columns beside it, several rows
// a wave.
// Each LDS cell holds a tap as two words, (b, r) and (g, 1) as 16-bit
// halves for an unfocused pixel, zeros for a focused pixel or a cell
// outside the viewport (never an unfocused tap, which is what the
// reference's clipped loops give): a tap is one 64-bit LDS read and two
// adds, its count coming with the colour.
// The box's (2r)^2 taps come from exclusive prefix sums along the rows of
// the window, two reads a row (a row's sums stay below 2^16: at most 96 cells
// of 255), from SW_DOF_PREFIX on, where two reads a row beat six taps (the
// 1231x717 box of radius 5: 22.7 to 19.3 us when this went in).
#define SW_DOF_PREFIX 3
template <int RMAX>
__global__ __launch_bounds__(SW_DOF_NT) void k_dof(BatchDev B, const JobDev *__restrict__ jobs)
{
    extern __shared__ uint2 s_tap[];
    constexpr int TW = SW_DOF_TW, TH = SW_DOF_TH, ROWS = SW_DOF_NT / TW, PER = TH / ROWS, P = TW + 2 * RMAX;
    static_assert(TW == 64 && TH % ROWS == 0 && 64 % (2 * RMAX) == 0, "a wave loads whole rows");
    const JobDev &J = jobs[find_job<JD>(B, jobs, blockIdx.x)];
    const uint32_t n = dof_blocks(J.V.vw, J.V.vh), q = n / 8;
    uint32_t lb = blockIdx.x - J.dblock0;
    if (lb < 8 * q)
        lb = (lb % 8) * q + lb / 8;
    const int bx = (J.V.vw + TW - 1) / TW;
    const int ox = (int)(lb % bx) * TW, oy = (int)(lb / bx) * TH;   // viewport-relative
    const int R = J.rmax, vw = J.V.vw, vh = J.V.vh, pitch = J.out_pitch;
    const int tx = threadIdx.x & 63, ty = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Offsets are 32-bit: a surface holds at most 2^30 words.  A cell outside
    // the viewport loads one inside and is zeroed after (no branch per cell);
    // every load is issued before the first is used.
    const SW_RO uint32_t *colr = ro(J.out_color) + ((J.V.vy - J.out_oy) * pitch + (J.V.vx - J.out_ox));
    const SW_RO uint8_t *alpha = ro(J.dofa);
    const int x = ox + tx, xin = min(x, vw - 1);
    uint32_t own[PER], al[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int y = min(oy + ty + ROWS * j, vh - 1);
        own[j] = colr[y * pitch + xin];
        al[j] = alpha[y * vw + xin];
    }
    // the rows above and below: row h of 2R is -R + h, past the tile from R on
    constexpr int NV = (2 * RMAX + ROWS - 1) / ROWS;
    uint32_t vert[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int h = ty + ROWS * k, y = oy + (h < R ? h - R : h - R + TH);
        vert[k] = 0;
        if (h < 2 * R && y >= 0 && y < vh)   // the same in every lane
            vert[k] = colr[y * pitch + xin];
    }
    // the columns beside: SIDE lanes a row, RMAX on either side
    constexpr int SIDE = 2 * RMAX, SROWS = 64 / SIDE, NS = (TH + 2 * RMAX + ROWS * SROWS - 1) / (ROWS * SROWS);
    const int e = tx % SIDE, scol = e < RMAX ? e - RMAX : e - RMAX + TW;   // tile-relative
    const int sx = ox + scol, sxin = min(max(sx, 0), vw - 1);
    const bool sok = sx >= 0 && sx < vw;
    uint32_t side[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) {
        const int y = oy - R + (ty + ROWS * k) * SROWS + tx / SIDE;
        side[k] = colr[min(max(y, 0), vh - 1) * pitch + sxin];
        if (!sok || y < 0 || y >= vh)
            side[k] = 0;
    }
    auto put = [&](int row, int col, uint32_t v) {   // tile-relative cell
        const uint32_t w = v & 1u << 24 ? v : 0u;     // bit 24: unfocused
        s_tap[(row + RMAX) * P + col + RMAX] = make_uint2(w & 0x00FF00FFu, w >> 8 & 0x000100FFu);
    };
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int row = ty + ROWS * j;
        put(row, tx, x < vw && oy + row < vh ? own[j] : 0u);
    }
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int h = ty + ROWS * k;
        if (h < 2 * R)
            put(h < R ? h - R : h - R + TH, tx, x < vw ? vert[k] : 0u);
    }
#pragma unroll
    for (int k = 0; k < NS; k++) {
        const int h = (ty + ROWS * k) * SROWS + tx / SIDE;
        if (h < TH + 2 * R)
            put(h - R, scol, side[k]);
    }
    __syncthreads();
    const bool prefix = J.post == 1 && R >= SW_DOF_PREFIX;
    if (prefix) {
        // exclusive prefix sums along each row, one wave a row, 64 cells at a time
        for (int r = ty; r < TH + 2 * R; r += ROWS) {
            uint2 carry = make_uint2(0, 0);
            for (int c0 = 0; c0 < P; c0 += 64) {
                const int i = (r + RMAX - R) * P + c0 + tx;
                const bool in = c0 + tx < P;
                const uint2 v = in ? s_tap[i] : make_uint2(0, 0);
                const uint2 t = make_uint2(carry.x + wave_incl_scan(v.x), carry.y + wave_incl_scan(v.y));
                if (in)
                    s_tap[i] = make_uint2(t.x - v.x, t.y - v.y);
                carry = make_uint2(__shfl(t.x, 63), __shfl(t.y, 63));
            }
        }
        __syncthreads();
    }
    if (x >= vw)
        return;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int py = ty + ROWS * j, y = oy + py;
        if (y >= vh)
            break;
        const int c = (py + RMAX) * P + tx + RMAX;
        const int radius = (int)(own[j] >> 25);
        uint32_t out = (own[j] & 0xFFFFFFu) | al[j] << 24;
        if (radius != 0) {
            // Blue and red add as the halves of one word, green and the count
            // as the halves of another: nine taps of 255, or the 256 of a box
            // of radius 8, stay below 2^16.  A larger box adds them apart.
            uint32_t br = 0, gc = 0, b = 0, g = 0, r = 0, count = 0;
            auto add = [&](uint2 w) {
                br += w.x;
                gc += w.y;
            };
            auto unpack = [&] {
                b += br & 0xFFFFu;
                r += br >> 16;
                g += gc & 0xFFFFu;
                count += gc >> 16;
                br = gc = 0;
            };
            if (prefix) {   // box, [x-r, x+r) x [y-r, y+r)
                for (int a = -radius; a < radius; a++) {
                    const uint2 lo = s_tap[c + a * P - radius], hi = s_tap[c + a * P + radius];
                    add(make_uint2(hi.x - lo.x, hi.y - lo.y));
                    if (RMAX > 8)
                        unpack();
                }
            } else if (J.post == 1) {
                for (int a = -radius; a < radius; a++)
                    for (int f = -radius; f < radius; f++)
                        add(s_tap[c + a * P + f]);
            } else {             // 3x3 taps at {-r, 0, r}
                const int dr = radius * P;
#pragma unroll
                for (int a = -1; a <= 1; a++)
#pragma unroll
                    for (int f = -1; f <= 1; f++)
                        add(s_tap[c + a * dr + f * radius]);
            }
            unpack();
            if (count) {
                const float rc = __builtin_amdgcn_rcpf((float)count);
                out = tap_mean(b, rc) | tap_mean(g, rc) << 8 | tap_mean(r, rc) << 16 | 255u << 24;
            }
        }
        J.surface[(int64_t)(y + J.V.vy) * J.surface_pitch + (x + J.V.vx)] = out;
    }
}

__global__ void k_fill32(uint32_t *p, uint64_t n, uint32_t w)
{
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = w;
}

// ----------------------------------------------------------- launchers
#define LAUNCH_CHECK(...)                                                      \
    do {                                                                       \
        hipLaunchKernelGGL(__VA_ARGS__);                                       \
        hipError_t e_ = hipGetLastError();                                     \
        if (e_ != hipSuccess)                                                  \
            return e_;                                                         \
    } while (0)

hipError_t launch_world(const WorldArgs &W, hipStream_t s)
{
    if (W.n_vertices)
        LAUNCH_CHECK(k_world, dim3((W.n_vertices + 255) / 256), dim3(256), 0, s, W);
    return hipSuccess;
}
hipError_t launch_vertex(const BatchDev &B, uint32_t blocks, uint32_t w0, uint32_t n_words, const JobDev *one,
                         hipStream_t s)
{
    // at least one block: the kernel also zeroes the counters
    if (one) {
        LAUNCH_CHECK(k_vertex_one, dim3(blocks ? blocks : 1), dim3(256), 0, s, B, w0, n_words, *one);
        return hipSuccess;
    }
    LAUNCH_CHECK(k_vertex, dim3(blocks ? blocks : 1), dim3(256), 0, s, B, w0, n_words, B.jobs);
    return hipSuccess;
}
hipError_t launch_front(const BatchDev &B, uint32_t blocks, hipStream_t s)
{
    // at least one block: the last block to finish scans the tile counts
    // into the bin offsets
    LAUNCH_CHECK(k_front, dim3(blocks ? blocks : 1), dim3(256), 0, s, B, B.jobs);
    return hipSuccess;
}
hipError_t launch_bin_fill(const BatchDev &B, uint32_t blocks, hipStream_t s, hipEvent_t done)
{
    // SW_RASTER_QUEUES more blocks than the fill needs: the first ones write the claim order
    if (!B.n_tiles)
        return done ? hipEventRecord(done, s) : hipSuccess;
    if (done) {
        // the kernel's own completion signals `done`: no marker after it
        hipExtLaunchKernelGGL(k_bin_fill, dim3(blocks + SW_RASTER_QUEUES), dim3(256), 0, s, nullptr, done, 0, B, B.jobs);
        return hipGetLastError();
    }
    LAUNCH_CHECK(k_bin_fill, dim3(blocks + SW_RASTER_QUEUES), dim3(256), 0, s, B, B.jobs);
    return hipSuccess;
}
template <int TW, int TH, bool G>
static hipError_t launch_raster_t(BatchDev B, uint32_t max_groups, uint32_t n_cus, hipStream_t s)
{
    constexpr int NT = raster_threads(TW, TH);
    // max_groups counts groups of 256 threads
    max_groups = std::max(1u, max_groups / (NT / 256));
    // split tiles are several items (only k_bin_fill knows how many)
    const uint64_t items = B.split == 0xFFFFFFFFu ? B.n_tiles : (uint64_t)B.n_tiles * SW_BANDS;
    const uint32_t g = items < max_groups ? (uint32_t)items : max_groups;
    B.n_static = std::min(g, n_cus * (1024 / NT));   // four waves a SIMD
    LAUNCH_CHECK((k_raster<TW, TH, G>), dim3(g), dim3(NT), 0, s, B, B.jobs);
    return hipSuccess;
}
template <bool G>
static hipError_t launch_raster_g(const BatchDev &B, int tw, int th, uint32_t max_groups, uint32_t n_cus, hipStream_t s)
{
    if (tw == 8 && th == 8)
        return launch_raster_t<8, 8, G>(B, max_groups, n_cus, s);
    if (tw == 16 && th == 16)
        return launch_raster_t<16, 16, G>(B, max_groups, n_cus, s);
    if (tw == 32 && th == 16)
        return launch_raster_t<32, 16, G>(B, max_groups, n_cus, s);
    if (tw == 32 && th == 32)
        return launch_raster_t<32, 32, G>(B, max_groups, n_cus, s);
    if (tw == 64 && th == 32)
        return launch_raster_t<64, 32, G>(B, max_groups, n_cus, s);
    if (tw == 64 && th == 64)
        return launch_raster_t<64, 64, G>(B, max_groups, n_cus, s);
    return hipErrorInvalidValue;
}
hipError_t launch_raster(const BatchDev &B, int tw, int th, uint32_t max_groups, uint32_t n_cus, bool generic,
                         hipStream_t s)
{
    if (!B.n_tiles)
        return hipSuccess;
    return generic ? launch_raster_g<true>(B, tw, th, max_groups, n_cus, s)
                   : launch_raster_g<false>(B, tw, th, max_groups, n_cus, s);
}

hipError_t launch_layers(const BatchDev &B, bool generic, uint32_t pixels, hipStream_t s)
{
    if (!B.n_tiles)
        return hipSuccess;
    // one block per layer tile
    if (generic)
        LAUNCH_CHECK(k_raster_layers<true>, dim3(B.n_tiles), dim3(SW_LAYER_THREADS), 0, s, B, B.jobs);
    else
        LAUNCH_CHECK(k_raster_layers<false>, dim3(B.n_tiles), dim3(SW_LAYER_THREADS), 0, s, B, B.jobs);
    const uint32_t blocks = (pixels + 255) / 256;
    LAUNCH_CHECK(k_tflatten, dim3(blocks), dim3(256), 0, s, B, 0u, B.jobs);
    LAUNCH_CHECK(k_tcopy, dim3(blocks), dim3(256), 0, s, B, 0u, B.jobs);
    return hipSuccess;
}
hipError_t launch_dof(const BatchDev &B, uint32_t blocks, int max_radius, hipStream_t s)
{
    if (!blocks)
        return hipSuccess;
    if (max_radius <= 8)
        LAUNCH_CHECK(k_dof<8>, dim3(blocks), dim3(SW_DOF_NT), dof_lds_bytes(8), s, B, B.jobs);
    else
        LAUNCH_CHECK(k_dof<SW_MAX_DOF_RADIUS>, dim3(blocks), dim3(SW_DOF_NT), dof_lds_bytes(SW_MAX_DOF_RADIUS), s, B,
                     B.jobs);
    return hipSuccess;
}

hipError_t resolve_kernels()
{
    const void *k[] = {
        (const void *)k_world, (const void *)k_vertex, (const void *)k_vertex_one, (const void *)k_front, (const void *)k_bin_fill,
        (const void *)k_raster<8, 8, false>, (const void *)k_raster<16, 16, false>,
        (const void *)k_raster<32, 16, false>, (const void *)k_raster<32, 32, false>,
        (const void *)k_raster<64, 32, false>, (const void *)k_raster<64, 64, false>,
        (const void *)k_raster<8, 8, true>, (const void *)k_raster<16, 16, true>,
        (const void *)k_raster<32, 16, true>, (const void *)k_raster<32, 32, true>,
        (const void *)k_raster<64, 32, true>, (const void *)k_raster<64, 64, true>,
        (const void *)k_raster_layers<false>, (const void *)k_raster_layers<true>,
        (const void *)k_tflatten, (const void *)k_tcopy,
        (const void *)k_dof<8>, (const void *)k_dof<SW_MAX_DOF_RADIUS>, (const void *)k_fill32,
    };
    for (const void *f : k) {
        hipFuncAttributes a;
        hipError_t e = hipFuncGetAttributes(&a, f);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

hipError_t launch_fill32(uint32_t *p, uint64_t n, uint32_t word, hipStream_t s)
{
    uint64_t blocks = (n + 255) / 256;
    if (blocks > 65536)
        blocks = 65536;
    if (blocks)
        LAUNCH_CHECK(k_fill32, dim3((uint32_t)blocks), dim3(256), 0, s, p, n, word);
    return hipSuccess;
}

}  // namespace sw
