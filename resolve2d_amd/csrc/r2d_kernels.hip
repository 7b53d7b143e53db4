// HIP kernels of one resolve2d step (Solver.process, src/core/lib.zig:189-299)
// for gfx950, over a batch of independent worlds.
//
// Small worlds take every step of a call in one kernel (k_fused, a workgroup
// per world).  The others take separate launches (every kernel reads its
// element counts from device memory so the whole step is a fixed launch
// sequence that can be captured in a hipGraph):
//
//   k_begin_step    counters, bucket and body counts, the scans' states cleared
//   k_prep          per body: cos/sin of the angle, cell range of the stale AABB
//   k_scan          cell counts -> entry offsets                (E entries)
//   k_entries       per entry: bucket = hash(cell) % table, bucket counts
//   k_scan          bucket counts -> bucket offsets
//   k_bucket_fill   per entry: scatter body into its bucket
//   k_bucket_rank   per entry: its place in descending body order, without duplicates
//   k_ent_cnt       per entry: bodies in the bucket with a higher slot
//   k_scan          -> raw candidate offsets                    (R candidates)
//   k_cand_emit     per entry: (a, b) raw candidates in the reference's query order
//   k_narrow        per candidate: first occurrence, filters, SAT
//   k_scan          collides flags -> manifold index and list   (M manifolds)
//   k_man_build     per manifold: contact points (identifyCollisionPoints);
//                   per world: manifold / item ranges
//   k_items         solver items and their ordering resources
//   k_scan, k_list_*  per-body ordered item lists -> ranks
//   k_color, k_world_order  coloured order only
//   k_chain_build   per item: its points' records
//   k_chain_plan    per world: the program of rows, records in its order
//   k_chain_bodies, k_chain_run  per sub-step: forces, integration, pre-step;
//                   then the world's program, which reproduces the
//                   reference's sequential order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "r2d_device.h"
#include "r2d_chain.h"
#include "r2d_kernels.h"

namespace r2d {

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ uint32_t grid_tid() { return blockIdx.x * blockDim.x + threadIdx.x; }
__device__ __forceinline__ uint32_t grid_stride() { return gridDim.x * blockDim.x; }
__device__ __forceinline__ uint32_t umin(uint32_t a, uint32_t b) { return a < b ? a : b; }
__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a < b ? b : a; }

// number of valid elements given a device count clamped to capacity
__device__ __forceinline__ uint32_t dev_count(const uint32_t* c, uint32_t cap)
{
    uint32_t v = *c;
    return v < cap ? v : cap;
}

// largest i in [0, n) with off[i] <= x (off ascending)
__device__ __forceinline__ uint32_t upper_idx(const uint32_t* off, uint32_t n, uint32_t x)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= x) lo = mid; else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    return x;
}

// exclusive block scan; blockDim multiple of 64, <= 1024
__device__ uint32_t block_excl_scan(uint32_t v, uint32_t* sm, uint32_t* total)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint32_t x = wave_incl_scan(v);
    if (lane == 63) sm[wid] = x;
    __syncthreads();
    if (wid == 0) {
        uint32_t t = lane < nw ? sm[lane] : 0u;
        t = wave_incl_scan(t);
        if (lane < nw) sm[lane] = t;
    }
    __syncthreads();
    uint32_t base = wid ? sm[wid - 1] : 0u;
    *total = sm[nw - 1];
    __syncthreads();
    return base + x - v;
}

// ------------------------------------------------------------- scan (u32)
// Exclusive scan of n = min(*n_dev, cap) (or n_const) values into out[0..n],
// out[n] = total.  Of flags it also lists, in `where`, the places that are set
// (the first where_cap of them).  One kernel for arrays of up to SCAN_TILES tiles (k_scan);
// three fixed-grid kernels for larger ones.
constexpr int SCAN_BLOCKS = 256;
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 4;

__device__ __forceinline__ uint32_t scan_n(const uint32_t* n_dev, uint32_t n_const, uint32_t cap)
{
    return n_dev ? dev_count(n_dev, cap) : n_const;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_reduce(const uint32_t* in, const uint32_t* n_dev,
                                                               uint32_t n_const, uint32_t cap, uint32_t* partials)
{
    __shared__ uint32_t sm[16];
    uint32_t n = scan_n(n_dev, n_const, cap);
    uint32_t chunk = (n + SCAN_BLOCKS - 1) / SCAN_BLOCKS;
    uint32_t b0 = blockIdx.x * chunk, b1 = umin(n, b0 + chunk);
    uint32_t s = 0;
    for (uint32_t i = b0 + threadIdx.x; i < b1; i += blockDim.x) s += in[i];
    uint32_t tot;
    block_excl_scan(s, sm, &tot);
    if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_partials(uint32_t* partials, uint32_t* out,
                                                                 const uint32_t* n_dev, uint32_t n_const,
                                                                 uint32_t cap, uint32_t* total_dev)
{
    __shared__ uint32_t sm[16];
    uint32_t n = scan_n(n_dev, n_const, cap);
    uint32_t v = threadIdx.x < SCAN_BLOCKS ? partials[threadIdx.x] : 0u;
    uint32_t tot;
    uint32_t ex = block_excl_scan(v, sm, &tot);
    if (threadIdx.x < SCAN_BLOCKS) partials[threadIdx.x] = ex;
    if (threadIdx.x == 0) {
        out[n] = tot;
        if (total_dev) *total_dev = tot;
    }
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_down(const uint32_t* in, uint32_t* out,
                                                             const uint32_t* n_dev, uint32_t n_const,
                                                             uint32_t cap, const uint32_t* partials, uint32_t* where,
                                                             uint32_t where_cap)
{
    __shared__ uint32_t sm[16];
    uint32_t n = scan_n(n_dev, n_const, cap);
    uint32_t chunk = (n + SCAN_BLOCKS - 1) / SCAN_BLOCKS;
    uint32_t b0 = blockIdx.x * chunk, b1 = umin(n, b0 + chunk);
    uint32_t base = partials[blockIdx.x];
    const uint32_t tile = SCAN_THREADS * SCAN_ITEMS;
    for (uint32_t t0 = b0; t0 < b1; t0 += tile) {
        uint32_t v[SCAN_ITEMS];
        uint32_t s = 0;
        uint32_t i0 = t0 + threadIdx.x * SCAN_ITEMS;
#pragma unroll
        for (int j = 0; j < SCAN_ITEMS; ++j) {
            v[j] = (i0 + j < b1) ? in[i0 + j] : 0u;
            s += v[j];
        }
        uint32_t tot;
        uint32_t ex = block_excl_scan(s, sm, &tot);
        uint32_t run = base + ex;
#pragma unroll
        for (int j = 0; j < SCAN_ITEMS; ++j) {
            if (i0 + j < b1) {
                out[i0 + j] = run;
                if (where && v[j] && run < where_cap) where[run] = i0 + j;
            }
            run += v[j];
        }
        base += tot;
    }
}

// The single-pass scan with decoupled look-back (Merrill and Garland).  Tiles
// taken in the order of a ticket.  A tile publishes its sum, adds up its
// predecessors' (64 at a time, each a sum or, from some tile on, a prefix) and
// publishes its prefix: value and kind in one 64-bit word.  Every tile it waits
// for has its ticket and runs, so the wait ends; the limit only bounds it.
// One launch where the three kernels took 4.7 us each, almost all of it the
// launch: a step has five scans (4,096-body pile, 20 launches fewer with the
// kernels that clear and prepare folded together: 813 -> 720 us a frame).
constexpr uint32_t SCAN_EACH = 16, SCAN_TILE = SCAN_THREADS * SCAN_EACH;
constexpr uint32_t SCAN_SPIN = 1u << 22;
__global__ __launch_bounds__(SCAN_THREADS) void k_scan(const uint32_t* in, uint32_t* out, const uint32_t* n_dev,
                                                        uint32_t n_const, uint32_t cap, uint32_t* total_dev,
                                                        uint64_t* state, uint32_t* ticket, uint32_t* overflow,
                                                        uint32_t* where, uint32_t where_cap)
{
    __shared__ uint32_t sm[16], s_tile, s_before;
    const uint32_t t = threadIdx.x, lane = t & 63u;
    if (t == 0) s_tile = atomicAdd(ticket, 1u);
    __syncthreads();
    const uint32_t tile = s_tile, n = scan_n(n_dev, n_const, cap);
    const uint32_t tiles = n ? (n + SCAN_TILE - 1u) / SCAN_TILE : 1u;
    if (tile >= tiles) return;
    const uint32_t i0 = tile * SCAN_TILE + t * SCAN_EACH;
    uint32_t v[SCAN_EACH], sum = 0;
    if (i0 + SCAN_EACH <= n) {
        const uint4* q = reinterpret_cast<const uint4*>(in + i0);   // arrays start at 256-byte bounds
#pragma unroll
        for (uint32_t k = 0; k < SCAN_EACH / 4; ++k) {
            const uint4 x = q[k];
            v[4 * k] = x.x; v[4 * k + 1] = x.y; v[4 * k + 2] = x.z; v[4 * k + 3] = x.w;
        }
    } else {
#pragma unroll
        for (uint32_t k = 0; k < SCAN_EACH; ++k) v[k] = i0 + k < n ? in[i0 + k] : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < SCAN_EACH; ++k) sum += v[k];
    uint32_t tot;
    const uint32_t ex = block_excl_scan(sum, sm, &tot);
    if (t < 64u) {
        auto put = [&](uint32_t kind, uint32_t x) {
            if (lane == 0)
                __hip_atomic_store(&state[tile], ((uint64_t)kind << 32) | x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        uint32_t before = 0;
        if (tile > 0u) {
            put(1u, tot);
            uint32_t spins = 0;
            for (int32_t base = (int32_t)tile - 1; base >= 0;) {
                const int32_t at = base - (int32_t)lane;
                const uint64_t x = at >= 0 ? __hip_atomic_load(&state[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                           : (uint64_t)2u << 32;
                const uint32_t kind = (uint32_t)(x >> 32);
                if (__ballot(kind == 0u)) {
                    if (++spins > SCAN_SPIN) {
                        if (lane == 0) atomicOr(overflow, 16u);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                const uint64_t ends = __ballot(kind == 2u);
                const uint32_t last = ends ? (uint32_t)__builtin_ctzll(ends) : 63u;   // the nearest prefix ends the sum
                before += (uint32_t)__shfl((int)wave_incl_scan(lane <= last ? (uint32_t)x : 0u), 63);
                if (ends) break;
                base -= 64;
            }
        }
        put(2u, before + tot);
        if (lane == 0) s_before = before;
    }
    __syncthreads();
    uint32_t run = s_before + ex;
#pragma unroll
    for (uint32_t k = 0; k < SCAN_EACH; ++k) {
        if (i0 + k < n) {
            out[i0 + k] = run;
            if (where && v[k] && run < where_cap) where[run] = i0 + k;
        }
        run += v[k];
    }
    if (tile == tiles - 1u && t == 0) {
        out[n] = s_before + tot;
        if (total_dev) *total_dev = s_before + tot;
    }
}

void scan_u32(const uint32_t* in, uint32_t* out, const uint32_t* n_dev, uint32_t n_const, uint32_t cap,
              uint32_t* total_dev, const StepDev& S, int which, hipStream_t st, uint32_t* where, uint32_t where_cap)
{
    uint32_t* partials = S.partials;
    const uint64_t tiles = ((uint64_t)cap + SCAN_TILE - 1u) / SCAN_TILE;
    if (tiles <= SCAN_TILES) {
        hipLaunchKernelGGL(k_scan, dim3((unsigned)std::max<uint64_t>(tiles, 1u)), dim3(SCAN_THREADS), 0, st, in, out, n_dev, n_const,
                           cap, total_dev, S.scan_state + (size_t)which * SCAN_TILES, S.scan_ticket + which,
                           S.counters + C_OVERFLOW, where, where_cap);
        return;
    }
    hipLaunchKernelGGL(k_scan_reduce, dim3(SCAN_BLOCKS), dim3(SCAN_THREADS), 0, st, in, n_dev, n_const, cap, partials);
    hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(SCAN_THREADS), 0, st, partials, out, n_dev, n_const, cap,
                       total_dev);
    hipLaunchKernelGGL(k_scan_down, dim3(SCAN_BLOCKS), dim3(SCAN_THREADS), 0, st, in, out, n_dev, n_const, cap,
                       partials, where, where_cap);
}

// ---------------------------------------------------------- body geometry
// The parts of a body that SAT and contact generation read.  World vertices
// are add2(rotate2(local_vertex, angle), pos) with the angle's cos/sin taken
// once per step (identical bits to recomputing them per call).
struct Geo {
    v2 pos;
    float r;          // disc radius
    bool rect;
    uint32_t id;
    v2 lv[4];         // Rectangle.local_vertices (Rectangle.zig:40)
    v2 wv[4];         // world vertices
    float c, s;       // cos / sin of the angle
};

// B: a type with the body arrays of WorldDev (px, py, flags, rad, id, hw, hh)
template <class B>
__device__ __forceinline__ Geo load_geo(const B& D, uint32_t slot, float c, float s)
{
    Geo g;
    g.pos = mk(D.px[slot], D.py[slot]);
    uint32_t f = D.flags[slot];
    g.rect = (f & BF_RECT) != 0;
    g.r = D.rad[slot];
    g.id = D.id[slot];
    g.c = c; g.s = s;
    float hw = D.hw[slot], hh = D.hh[slot];
    g.lv[0] = mk(-hw, -hh); g.lv[1] = mk(-hw, hh); g.lv[2] = mk(hw, hh); g.lv[3] = mk(hw, -hh);
#pragma unroll
    for (int i = 0; i < 4; ++i) g.wv[i] = add2(rotcs(g.lv[i], c, s), g.pos);
    return g;
}

// Disc.closestPoint (Disc.zig:80-84); Rectangle.closestPoint (Rectangle.zig:114-130)
__device__ __forceinline__ v2 closest_point(const Geo& b, v2 p)
{
    if (!b.rect) {
        v2 n = normalize2(sub2(p, b.pos));
        return addmult2(b.pos, n, b.r);
    }
    float best = __builtin_inff();
    v2 bp = p;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float d2 = length2sq(sub2(b.wv[i], p));
        if (d2 < best) { best = d2; bp = b.wv[i]; }
    }
    return bp;
}

struct Edge {
    v2 dir, a, b;
};

// a[i] for a run-time i with the array kept in registers (selects, not a
// dynamically indexed private array, which would live in scratch memory)
__device__ __forceinline__ v2 pick4(const v2 (&a)[4], int i)
{
    v2 r = a[0];
    r = i == 1 ? a[1] : r;
    r = i == 2 ? a[2] : r;
    r = i == 3 ? a[3] : r;
    return r;
}

// Disc.getNormal (Disc.zig:86-90); Rectangle.getNormal (Rectangle.zig:132-151)
__device__ __forceinline__ Edge get_normal(const Geo& self, const Geo& other, int iter)
{
    Edge e;
    if (!self.rect) {
        v2 closest = closest_point(other, self.pos);
        e.dir = normalize2(sub2(closest, self.pos));
        e.a = e.b = mk(0.f, 0.f);
        return e;
    }
    int nx = (iter == 3) ? 0 : iter + 1;
    v2 a1 = pick4(self.wv, iter), a2 = pick4(self.wv, nx);
    e.dir = rot90ccw(normalize2(sub2(a2, a1)));
    e.a = a1; e.b = a2;
    return e;
}

// projectAlongAxis: Disc.zig:92-97, Rectangle.zig:153-169
__device__ __forceinline__ void project(const Geo& b, v2 n, float& lo, float& hi)
{
    if (!b.rect) {
        float mid = dot2(b.pos, n);
        lo = mid - b.r; hi = mid + b.r;
        return;
    }
    lo = __builtin_inff(); hi = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float d = dot2(b.wv[i], n);
        if (d < lo) lo = d;
        if (d > hi) hi = d;
    }
}

__device__ __forceinline__ bool should_flip(v2 n, const Geo& ref, const Geo& inc)
{
    return dot2(n, sub2(inc.pos, ref.pos)) < 0.0f;   // collision.zig:221-226
}

struct Sat {
    v2 normal;
    float pen;
    int nid;
    int ref;          // 0: first argument of performNarrowSAT's pair order, 1: second
    bool set;
};

// overlapSAT (collision.zig:228-289); `which` tags the reference body
__device__ __forceinline__ bool overlap_sat(Sat& ret, const Geo& ref, const Geo& inc, int which)
{
    const float EPS = SAT_OVERLAP_THRESHOLD;
    int nn = ref.rect ? 4 : 1;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        if (it >= nn) break;
        Edge e = get_normal(ref, inc, it);
        v2 normal = e.dir;
        bool flipped = false;
        if (should_flip(normal, ref, inc)) { normal = negself(normal); flipped = true; }
        float p1lo, p1hi, p2lo, p2hi;
        project(ref, normal, p1lo, p1hi);
        project(inc, normal, p2lo, p2hi);
        float d1 = p1hi - p2lo;
        float d2 = p2hi - p1lo;
        float d = minn(d1, d2);
        if (d <= -COLLISION_MARGIN) return false;
        if (!flipped && approx2(normal, ret.normal, EPS)) {
            float tref = dot2(ref.pos, normal);
            float tinc = dot2(inc.pos, normal);
            if (tref < tinc - EPS) { ret.pen = d; ret.normal = normal; ret.nid = it; ret.ref = which; ret.set = true; }
        }
        if (!flipped && approx2(normal, negate2(ret.normal), EPS)) {
            v2 diff = sub2(inc.pos, ref.pos);
            if (dot2(diff, normal) > dot2(diff, ret.normal) + EPS) {
                ret.pen = d; ret.normal = normal; ret.nid = it; ret.ref = which; ret.set = true;
            }
        }
        if (d + EPS < ret.pen) { ret.pen = d; ret.normal = normal; ret.nid = it; ret.ref = which; ret.set = true; }
    }
    return true;
}

// aabb.intersects (aabb.zig:12-19)
template <class B>
__device__ __forceinline__ bool aabb_hit(const B& D, uint32_t a, uint32_t b)
{
    float dx = absf(D.ax[b] - D.ax[a]);
    float dy = absf(D.ay[b] - D.ay[a]);
    return (dx <= (D.ahw[a] + D.ahw[b]) + AABB_EPS_OVERLAP) && (dy <= (D.ahh[a] + D.ahh[b]) + AABB_EPS_OVERLAP);
}

__device__ __forceinline__ bool excluded(const WorldDev& D, uint32_t ida, uint32_t idb)
{
    uint64_t key = ida < idb ? (((uint64_t)ida << 32) | idb) : (((uint64_t)idb << 32) | ida);
    int lo = 0, hi = D.nexcl;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        uint64_t v = D.excl[mid];
        if (v == key) return true;
        if (v < key) lo = mid + 1; else hi = mid;
    }
    return false;
}

// ------------------------------------------------------------ broadphase
// One body's broadphase preparation: cos / sin of the angle, the scheduling
// flag (a static body orders contacts only if a contact's "+= 0" could change
// it: a -0 component; joint-touched bodies are added later) and the cell
// range of SpatialHash.iterateAABBHashes (SpatialHash.zig:83-96) from the
// stale AABB.  err: 3 cell range too large to enumerate, 4 non-finite AABB
// (@intFromFloat is undefined in the reference), 0 otherwise.
struct Prep {
    float c, s;
    uint32_t res;
    int64_t x0, y0;
    uint32_t nx, ny, ncell;
    int err;
};

__device__ __forceinline__ Prep prep_body(const WorldDev& D, uint32_t sl)
{
    Prep o;
    float a = D.ang[sl];
    o.c = cosf_r(a);
    o.s = sinf_r(a);
    uint32_t f = D.flags[sl];
    o.res = 1u;
    if (f & BF_STATIC) {
        float m0 = D.mx[sl], m1 = D.my[sl], m2 = D.L[sl];
        bool negz = (m0 == 0.0f && __builtin_signbit(m0)) || (m1 == 0.0f && __builtin_signbit(m1)) ||
                    (m2 == 0.0f && __builtin_signbit(m2));
        o.res = negz ? 1u : 0u;
    }
    o.err = 0;
    o.ncell = 0;
    o.x0 = o.y0 = 0;
    o.nx = o.ny = 0;
    float cell = D.cell;
    float ax = D.ax[sl], ay = D.ay[sl], hw = D.ahw[sl], hh = D.ahh[sl];
    float v0 = floorf((ax - hw) / cell), v1 = floorf((ay - hh) / cell);
    float v2f = floorf((ax + hw) / cell), v3 = floorf((ay + hh) / cell);
    const float LIM = 4.0e18f;
    bool ok = (v0 > -LIM && v0 < LIM) && (v1 > -LIM && v1 < LIM) && (v2f > -LIM && v2f < LIM) &&
              (v3 > -LIM && v3 < LIM);
    if (ok) {
        int64_t x0 = (int64_t)v0, y0 = (int64_t)v1, x1 = (int64_t)v2f, y1 = (int64_t)v3;
        uint64_t nx = (x1 >= x0) ? (uint64_t)(x1 - x0 + 1) : 0u;
        uint64_t ny = (y1 >= y0) ? (uint64_t)(y1 - y0 + 1) : 0u;
        uint64_t tot = nx * ny;
        if (nx > (1u << 30) || ny > (1u << 30) || tot > (1u << 30)) {
            o.err = 3;
        } else {
            o.ncell = (uint32_t)tot;
            o.x0 = x0; o.y0 = y0; o.nx = (uint32_t)nx; o.ny = (uint32_t)ny;
        }
    } else {
        o.err = 4;
    }
    return o;
}

// A step's counters, statuses and counts at zero.  The overflow flag is sticky
// (it is cleared by the host), so a replayed sequence of steps stops
// committing at the first step whose scratch did not fit.
__global__ __launch_bounds__(256) void k_begin_step(StepDev S)
{
    const uint32_t top = umax(umax(S.nb, S.nbuckets), umax(S.nworlds, SCANS * SCAN_TILES));
    for (uint32_t x = grid_tid(); x <= top; x += grid_stride()) {
        if (x < C_OVERFLOW) S.counters[x] = 0u;
        if (x < SCANS) S.scan_ticket[x] = 0u;
        if (x < SCANS * SCAN_TILES) S.scan_state[x] = 0ull;
        if (x <= S.nbuckets) { S.bkt_cnt[x] = 0u; S.bkt_fill[x] = 0u; }
        if (x <= S.nworlds) {
            S.w_status[x] = 0;
            S.w_chain[x] = WorldChain{};
            if (S.nworlds == 1u) S.w_order[0] = 0u;   // k_world_order is for more
        }
        if (x <= S.nb) {
            S.deg[x] = 0u;
            S.deg_fill[x] = 0u;
            if (x < S.nb) S.cmap[x] = UNTOUCHED;
        }
    }
}

__global__ void k_prep(StepDev S)
{
    for (uint32_t i = grid_tid(); i < S.nb; i += grid_stride()) {
        uint32_t w = 0, hi = S.nworlds;   // the body's world: the last whose bodies start at or before it
        while (hi - w > 1) {
            const uint32_t mid = (w + hi) >> 1;
            if (S.worlds[mid].body_base <= i) w = mid; else hi = mid;
        }
        S.bworld[i] = w;
        const WorldDev& D = S.worlds[w];
        const Prep o = prep_body(D, i - D.body_base);
        S.cc[i] = o.c;
        S.cs[i] = o.s;
        S.sflag[i] = o.res;
        if (o.err) S.w_status[w] = o.err;
        if (!o.err && o.ncell) { S.cx0[i] = o.x0; S.cy0[i] = o.y0; S.cnx[i] = o.nx; S.cny[i] = o.ny; }
        S.ncell[i] = o.ncell;
    }
}

// the world of batch joint j
__device__ __forceinline__ uint32_t joint_world(const StepDev& S, uint32_t j)
{
    uint32_t lo = 0, hi = S.nworlds;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (S.worlds[mid].joint_base <= j) lo = mid; else hi = mid;
    }
    return lo;
}

// per cell entry: its body, its bucket; bucket occupancy counts.  And the
// bodies of distance / offset joints, which write both even when static
// (DistanceJoint.zig:72-74, OffsetDistanceJoint.zig:100-104): such a static
// body orders every item that touches it.
__global__ void k_entries(StepDev S)
{
    for (uint32_t j = grid_tid(); j < S.njoints; j += grid_stride()) {
        const WorldDev& D = S.worlds[joint_world(S, j)];
        const Joint& J = D.joints[j - D.joint_base];
        if (J.type <= 1) {
            if (J.s1 >= 0) atomicOr(&S.sflag[D.body_base + J.s1], SF_RESOURCE);
            if (J.s2 >= 0) atomicOr(&S.sflag[D.body_base + J.s2], SF_RESOURCE);
        }
    }
    uint32_t E = dev_count(&S.counters[C_ENTRIES], S.cap_e);
    if (S.counters[C_ENTRIES] > S.cap_e) { if (grid_tid() == 0) atomicOr(&S.counters[C_OVERFLOW], 1u); return; }
    for (uint32_t e = grid_tid(); e < E; e += grid_stride()) {
        uint32_t i = upper_idx(S.cell_off, S.nb, e);   // body whose cell range holds entry e
        uint32_t k = e - S.cell_off[i];
        const WorldDev& D = S.worlds[S.bworld[i]];
        uint32_t nx = S.cnx[i];
        int64_t yi = S.cy0[i] + (int64_t)(k / nx);
        int64_t xi = S.cx0[i] + (int64_t)(k % nx);
        uint32_t gb = D.bucket_base + (uint32_t)cell_hash((uint64_t)D.table, xi, yi);
        S.ent_body[e] = i;
        S.ent_bkt[e] = gb;
        atomicAdd(&S.bkt_cnt[gb], 1u);
    }
}

__global__ void k_bucket_fill(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    uint32_t E = dev_count(&S.counters[C_ENTRIES], S.cap_e);
    for (uint32_t e = grid_tid(); e < E; e += grid_stride()) {
        uint32_t gb = S.ent_bkt[e];
        uint32_t pos = atomicAdd(&S.bkt_fill[gb], 1u);
        S.bkt_items[S.bkt_off[gb] + pos] = S.ent_body[e];
    }
}

// How many of l[0, c) are below v: four entries per iteration, their loads
// in flight together
__device__ __forceinline__ uint32_t count_below(const uint32_t* l, uint32_t c, uint32_t v)
{
    uint32_t r = 0, i = 0;
    for (; i + 4 <= c; i += 4) {
        const uint32_t a0 = l[i], a1 = l[i + 1], a2 = l[i + 2], a3 = l[i + 3];
        r += (a0 < v) + (a1 < v) + (a2 < v) + (a3 < v);
    }
    for (; i < c; ++i) r += l[i] < v;
    return r;
}

// Walks of long cell lists: a wall has hundreds of cells, and one thread walks
// them while the kernel waits for it.  Sixteen loads are in flight at a time
// (four for the usual body of up to four cells).
template <uint32_t W, class F>
__device__ __forceinline__ bool walk(const uint32_t* l, uint32_t i, uint32_t c, F stop)
{
    uint32_t x[W];
    bool hit = false;
#pragma unroll
    for (uint32_t q = 0; q < W; ++q) x[q] = l[umin(i + q, c - 1u)];
#pragma unroll
    for (uint32_t q = 0; q < W; ++q) hit = stop(x[q], i + q < c) || hit;
    return hit;
}

// how many of l[0, c) equal v
__device__ __forceinline__ uint32_t count_equal(const uint32_t* l, uint32_t c, uint32_t v)
{
    uint32_t r = 0;
    for (uint32_t i = 0; i < c; i += 16)
        walk<16>(l, i, c, [&](uint32_t x, bool in) { r += in && x == v; return false; });
    return r;
}

// whether some of l[0, c) is one of h[0, n), n of 1 to 4
__device__ __forceinline__ bool any_equal(const uint32_t* l, uint32_t c, const uint32_t* h, uint32_t n)
{
    if (c == 0u) return false;
    const uint32_t h0 = h[0], h1 = h[umin(1u, n - 1u)], h2 = h[umin(2u, n - 1u)], h3 = h[n - 1u];
    auto same = [&](uint32_t x, bool) { return x == h0 || x == h1 || x == h2 || x == h3; };   // (the last one may repeat)
    if (walk<4>(l, 0u, c, same)) return true;
    for (uint32_t i = 4; i < c; i += 16)
        if (walk<16>(l, i, c, same)) return true;
    return false;
}

// A cell entry's rank among its bucket's members it[0, c): how many are
// greater than its body a and how many equal it.  Four members per
// iteration, so their loads are in flight together.
__device__ __forceinline__ void bucket_rank_of(const uint32_t* it, uint32_t c, uint32_t a, uint32_t& greater,
                                               uint32_t& same)
{
    uint32_t g = 0, e = 0, j = 0;
    for (; j + 4 <= c; j += 4) {
        const uint32_t v0 = it[j], v1 = it[j + 1], v2 = it[j + 2], v3 = it[j + 3];
        g += (v0 > a) + (v1 > a) + (v2 > a) + (v3 > a);
        e += (v0 == a) + (v1 == a) + (v2 == a) + (v3 == a);
    }
    for (; j < c; ++j) {
        const uint32_t v = it[j];
        g += v > a;
        e += v == a;
    }
    greater = g;
    same = e;
}

// Within a bucket the reference stores entries in reverse insertion order
// (pre-decrement scatter, SpatialHash.zig:36-40, 59-68): descending body slot.
// Each entry's place is the number of bucket members with a higher slot plus
// its rank among its own body's earlier entries in the same bucket (a body
// listed twice in one bucket -- two of its cells hash alike -- sits in
// adjacent places; readers skip the repeat, which cannot change which pair
// appears first).
__global__ void k_bucket_rank(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    uint32_t E = dev_count(&S.counters[C_ENTRIES], S.cap_e);
    for (uint32_t e = grid_tid(); e < E; e += grid_stride()) {
        uint32_t a = S.ent_body[e], gb = S.ent_bkt[e];
        uint32_t o = S.bkt_off[gb], n = S.bkt_cnt[gb];
        const uint32_t* it = S.bkt_items + o;
        uint32_t greater, same;
        bucket_rank_of(it, n, a, greater, same);
        uint32_t dup = 0;
        if (same > 1) {
            const uint32_t x = S.cell_off[a];
            dup = count_equal(S.ent_bkt + x, e - x, gb);
        }
        S.bkt_sorted[o + greater + dup] = a;
    }
}

// raw candidates per entry: distinct bucket members with a higher slot than
// the entry's body
__global__ void k_ent_cnt(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    uint32_t E = dev_count(&S.counters[C_ENTRIES], S.cap_e);
    for (uint32_t e = grid_tid(); e < E; e += grid_stride()) {
        uint32_t a = S.ent_body[e], gb = S.ent_bkt[e];
        const uint32_t* it = S.bkt_sorted + S.bkt_off[gb];
        uint32_t n = S.bkt_cnt[gb], c = 0;
        for (uint32_t j = 0; j < n && it[j] > a; ++j) c += (j == 0 || it[j] != it[j - 1]);
        S.ent_cnt[e] = c;
    }
}

__global__ void k_cand_emit(StepDev S)
{
    uint32_t E = dev_count(&S.counters[C_ENTRIES], S.cap_e);
    if (S.counters[C_OVERFLOW]) return;
    if (S.counters[C_RAW] > S.cap_r) { if (grid_tid() == 0) atomicOr(&S.counters[C_OVERFLOW], 2u); return; }
    for (uint32_t e = grid_tid(); e < E; e += grid_stride()) {
        uint32_t a = S.ent_body[e], gb = S.ent_bkt[e];
        const uint32_t* it = S.bkt_sorted + S.bkt_off[gb];
        uint32_t o = S.ent_off[e], c = S.ent_cnt[e];
        uint32_t k = e - S.cell_off[a];
        for (uint32_t j = 0, q = 0; q < c; ++j) {
            if (j > 0 && it[j] == it[j - 1]) continue;
            S.cand[o + q] = make_uint4(a, it[j], k, 0u);   // one 16-byte store per candidate
            ++q;
        }
    }
}

// Solver.updateManifolds filters + performNarrowSAT (lib.zig:272-285,
// collision.zig:299-320) for one raw candidate: bodies sa < sb (world slots),
// found at cell k of sa.  ba: bucket of each cell of sa; bb: of each of the nb
// cells of sb.  A candidate counts only at the first position of its partner
// in the lower body's query list; later occurrences are the reference's
// "already a manifold / already rejected".  Returns whether it collides, with
// the reference face id | ref-is-sa << 2 in info and the normal.
// PREFILTERED: the both-static and AABB filters were applied when the
// candidate was emitted (the filters are pure predicates of the pair, so
// their order does not change which pairs pass)
template <bool PREFILTERED = false, class B>
__device__ __forceinline__ bool narrow_pair(const WorldDev& D, const B& bodies, uint32_t sa, uint32_t sb, uint32_t k,
                                            const uint32_t* ba, const uint32_t* bb, uint32_t nb, float ca, float sa_sin,
                                            float cb, float sb_sin, uint32_t& info, float& nx, float& ny)
{
    // the pair filters of updateManifolds (lib.zig:273-282) depend on the
    // pair only, so they run first: the first-occurrence test below costs
    // (cells of a before k) x (cells of b), large for wall-sized bodies
    bool ok = true;
    if (!PREFILTERED) {
        uint32_t fa = bodies.flags[sa], fb = bodies.flags[sb];
        ok = !((fa & BF_STATIC) && (fb & BF_STATIC));
    }
    if (ok && D.nexcl) ok = !excluded(D, bodies.id[sa], bodies.id[sb]);
    if (!PREFILTERED && ok) ok = aabb_hit(bodies, sa, sb);
    // b first appears in a's query list at cell k unless an earlier cell of a
    // hashes to a bucket b also occupies (buckets are deduplicated, so
    // within one bucket b appears once)
    for (uint32_t j = 0; j < nb && ok; j += 4) ok = !any_equal(ba, k, bb + j, umin(nb - j, 4u));
    if (!ok) return false;
    Geo ga = load_geo(bodies, sa, ca, sa_sin);
    Geo gb = load_geo(bodies, sb, cb, sb_sin);
    // performNarrowSAT: lower id is the first reference body
    bool a_first = ga.id < gb.id;
    const Geo o1 = a_first ? ga : gb;   // by value: selecting references would put both in scratch
    const Geo o2 = a_first ? gb : ga;
    Sat sat;
    const float undef = -3.0316488252093987e-13f;   // Zig Debug fill of `undefined` (0xAA)
    sat.normal = mk(undef, undef);
    sat.pen = __builtin_inff();
    sat.nid = 0; sat.ref = 0; sat.set = false;
    if (overlap_sat(sat, o1, o2, 0) && overlap_sat(sat, o2, o1, 1)) {
        // ref body expressed relative to (a, b)
        bool ref_is_a = (sat.ref == 0) == a_first;
        info = (uint32_t)sat.nid | (ref_is_a ? 4u : 0u);
        nx = sat.normal.x; ny = sat.normal.y;
        return true;
    }
    return false;
}

__global__ void k_narrow(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    uint32_t R = dev_count(&S.counters[C_RAW], S.cap_r);
    for (uint32_t q = grid_tid(); q < R; q += grid_stride()) {
        const uint4 cq = S.cand[q];
        const uint32_t a = cq.x, b = cq.y, k = cq.z;
        uint32_t info = 0;
        float nx = 0.f, ny = 0.f;
        const WorldDev& D = S.worlds[S.bworld[a]];
        bool hit = narrow_pair(D, D, a - D.body_base, b - D.body_base, k, S.ent_bkt + S.cell_off[a],
                               S.ent_bkt + S.cell_off[b], S.ncell[b], S.cc[a], S.cs[a], S.cc[b], S.cs[b], info, nx, ny);
        S.cand_flag[q] = hit ? 1u : 0u;
        if (hit) {
            S.sat_info[q] = info;
            S.sat_nx[q] = nx;
            S.sat_ny[q] = ny;
        }
    }
}

// CollisionPoint.init (collision.zig:38-51)
__device__ __forceinline__ void write_point(const StepDev& S, uint32_t m, int p, v2 pos, float depth,
                                            const Geo& ref, const Geo& inc, v2 normal)
{
    v2 middle = sub2(pos, scale2(normal, depth / 2));
    v2 r1 = sub2(middle, ref.pos), r2 = sub2(middle, inc.pos);
    float* P = S.m_pt;
    size_t cm = S.cap_m;
    P[(MP_ACC_PN * 2 + p) * cm + m] = 0.f;
    P[(MP_ACC_PT * 2 + p) * cm + m] = 0.f;
    P[(MP_R1X * 2 + p) * cm + m] = r1.x;
    P[(MP_R1Y * 2 + p) * cm + m] = r1.y;
    P[(MP_R2X * 2 + p) * cm + m] = r2.x;
    P[(MP_R2Y * 2 + p) * cm + m] = r2.y;
    P[(MP_POSX * 2 + p) * cm + m] = middle.x;
    P[(MP_POSY * 2 + p) * cm + m] = middle.y;
    P[(MP_DEPTH * 2 + p) * cm + m] = depth;
    P[(MP_ODEPTH * 2 + p) * cm + m] = depth;
    P[(MP_MASS_N * 2 + p) * cm + m] = 0.f;
    P[(MP_MASS_T * 2 + p) * cm + m] = 0.f;
}

// clipLineToLine (collision.zig:330-363): b clipped onto a
__device__ __forceinline__ void clip_line(v2 aa, v2 ab, v2 ba, v2 bb, v2& o1, v2& o2)
{
    v2 delta_a = sub2(ab, aa);
    float a_len = length2(delta_a);
    v2 tang = scale2(delta_a, 1.0f / a_len);
    v2 p1 = ba, p2 = bb;
    {
        float sc = dot2(sub2(ba, aa), tang);
        if (!(sc > 0.f && sc < a_len)) {
            v2 clos = (sc < 0.5f * a_len) ? aa : ab;
            v2 dp = sub2(ba, bb);
            float t = -dot2(tang, sub2(bb, clos)) / dot2(tang, dp);
            p1 = addmult2(bb, dp, t);
        }
    }
    {
        float sc = dot2(sub2(bb, aa), tang);
        if (!(sc > 0.f && sc < a_len)) {
            v2 clos = (sc < 0.5f * a_len) ? aa : ab;
            v2 dp = sub2(bb, ba);
            float t = -dot2(tang, sub2(ba, clos)) / dot2(tang, dp);
            p2 = addmult2(ba, dp, t);
        }
    }
    o1 = p1; o2 = p2;
}

// identifyCollisionPoints: Disc (Disc.zig:99-123), Rectangle (Rectangle.zig:171-211),
// with clipAgainstEdge (Rectangle.zig:213-238, Disc.zig:125-130), for the
// collision of world slots sa, sb (narrow_pair's info and normal) into
// manifold m; base: the world's first batch body index
template <class B>
__device__ __forceinline__ void man_build_one(const StepDev& S, const WorldDev& D, const B& bodies, uint32_t m,
                                              uint32_t base, uint32_t sa, uint32_t sb, uint32_t info, v2 normal,
                                              float ca, float sa_sin, float cb, float sb_sin)
{
    int nid = (int)(info & 3u);
    bool ref_is_a = (info & 4u) != 0;
    uint32_t sr = ref_is_a ? sa : sb, si = ref_is_a ? sb : sa;
    Geo gr = ref_is_a ? load_geo(bodies, sr, ca, sa_sin) : load_geo(bodies, sr, cb, sb_sin);
    Geo gi = ref_is_a ? load_geo(bodies, si, cb, sb_sin) : load_geo(bodies, si, ca, sa_sin);
    S.m_ref[m] = base + sr;
    S.m_inc[m] = base + si;
    S.m_nx[m] = normal.x;
    S.m_ny[m] = normal.y;
    S.m_fric[m] = 0.f;
    S.m_prev1[m] = D.ang[sr];
    S.m_prev2[m] = D.ang[si];
    uint32_t valid = 0;
    if (!gr.rect) {
        v2 pos = closest_point(gi, gr.pos);
        Edge e = get_normal(gr, gi, nid);
        v2 n = e.dir;
        if (should_flip(n, gr, gi)) n = negself(n);
        float d = dot2(n, sub2(pos, gr.pos));
        write_point(S, m, 0, pos, d - gr.r, gr, gi, n);
        valid = 1;
    } else {
        Edge e = get_normal(gr, gi, nid);
        if (!gi.rect) {
            v2 pos = addmult2(gi.pos, e.dir, -gi.r);
            float d = dot2(sub2(pos, e.a), e.dir);
            write_point(S, m, 0, pos, d, gr, gi, e.dir);
            valid = 1;
        } else {
            // incident edge: first i minimising dot(normal, rot90ccw(normalize(v[i+1]-v[i])))
            v2 ba = gi.wv[0], bb = gi.wv[1];
            float best = __builtin_inff();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                int nx = (i == 3) ? 0 : i + 1;
                v2 tn = rot90ccw(normalize2(sub2(gi.wv[nx], gi.wv[i])));
                float d = dot2(e.dir, tn);
                if (d < best) { best = d; ba = gi.wv[i]; bb = gi.wv[nx]; }
            }
            v2 ca2, cb2;
            clip_line(e.a, e.b, ba, bb, ca2, cb2);
            int i = 0;
            float d = dot2(sub2(ca2, e.a), e.dir);
            if (d < COLLISION_MARGIN) { write_point(S, m, i, ca2, d, gr, gi, e.dir); valid |= 1u << i; i += 1; }
            d = dot2(sub2(cb2, e.b), e.dir);
            if (d < COLLISION_MARGIN) { write_point(S, m, i, cb2, d, gr, gi, e.dir); valid |= 1u << i; }
        }
    }
    S.m_valid[m] = valid;
}

// each world's range of manifolds and of items
__device__ __forceinline__ void world_ranges(const StepDev& S)
{
    uint32_t M = dev_count(&S.counters[C_MANIFOLDS], S.cap_m);
    uint32_t R = dev_count(&S.counters[C_RAW], S.cap_r);
    uint32_t E = dev_count(&S.counters[C_ENTRIES], S.cap_e);
    for (uint32_t w = grid_tid(); w <= S.nworlds; w += grid_stride()) {
        uint32_t mb;
        if (w == S.nworlds) {
            mb = M;
        } else {
            const WorldDev& D = S.worlds[w];
            uint32_t fb = D.body_base;
            uint32_t e = (fb < S.nb) ? S.cell_off[fb] : E;
            if (e > E) e = E;
            uint32_t r = S.ent_off[e];
            if (r > R) r = R;
            mb = S.cand_idx[r];
            if (mb > M) mb = M;
        }
        S.w_man_begin[w] = mb;
        uint32_t jb = (w == S.nworlds) ? S.njoints : S.worlds[w].joint_base;
        S.w_item_base[w] = jb + mb;
        if (w == S.nworlds) S.counters[C_ITEMS] = jb + mb;
    }
}

// One manifold a lane, from the list of candidates that collide: of 24 piles'
// 1.2 M candidates 80,000 do.  (A lane per candidate, most of them without
// work in a wave that waits for the rest: the 24 piles' narrowphase 104 us a
// step, with the list and k_narrow's stores for collisions only 92.)
__global__ void k_man_build(StepDev S, const uint32_t* hits)
{
    if (S.counters[C_OVERFLOW]) return;
    const uint32_t M = S.counters[C_MANIFOLDS];
    if (M > S.cap_m) { if (grid_tid() == 0) atomicOr(&S.counters[C_OVERFLOW], 4u); return; }
    world_ranges(S);
    for (uint32_t m = grid_tid(); m < M; m += grid_stride()) {
        const uint32_t q = hits[m];
        const uint4 cq = S.cand[q];
        const uint32_t a = cq.x, b = cq.y;
        const WorldDev& D = S.worlds[S.bworld[a]];
        man_build_one(S, D, D, m, D.body_base, a - D.body_base, b - D.body_base, S.sat_info[q],
                      mk(S.sat_nx[q], S.sat_ny[q]), S.cc[a], S.cs[a], S.cc[b], S.cs[b]);
    }
}

// Order in which the solve kernels' workgroups take worlds: most items first
// (longest-processing-time first shortens the tail of the launch).  Worlds
// are binned by log2 of their item count; any order gives the same results.
__global__ __launch_bounds__(1024) void k_world_order(StepDev S)
{
    __shared__ uint32_t hist[33];
    if (S.counters[C_OVERFLOW]) return;
    const uint32_t nw = S.nworlds;
    if (threadIdx.x < 33) hist[threadIdx.x] = 0u;
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < nw; w += blockDim.x) {
        uint32_t items = S.w_item_base[w + 1] - S.w_item_base[w];
        atomicAdd(&hist[(uint32_t)__builtin_clz(items + 1u)], 1u);   // fewer leading zeros = more items
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t acc = 0;
        for (int b = 0; b < 33; ++b) { uint32_t c = hist[b]; hist[b] = acc; acc += c; }
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < nw; w += blockDim.x) {
        uint32_t items = S.w_item_base[w + 1] - S.w_item_base[w];
        uint32_t pos = atomicAdd(&hist[(uint32_t)__builtin_clz(items + 1u)], 1u);
        S.w_order[pos] = w;
    }
}

// A rank among the active lanes of a wave that are `on`, added to the counter
// of each one's world: one atomic per world and wave.
__device__ __forceinline__ uint32_t world_rank(const StepDev& S, bool on, uint32_t w, uint32_t WorldChain::* counter)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t rank = 0;
    for (uint64_t todo = __ballot(on); todo;) {
        const uint32_t lead = (uint32_t)__builtin_ctzll(todo);
        const uint64_t same = __ballot(on && w == (uint32_t)__shfl((int)w, (int)lead)) & todo;
        uint32_t at = 0;
        if (lane == lead) at = atomicAdd(&(S.w_chain[w].*counter), (uint32_t)__popcll(same));
        at = (uint32_t)__shfl((int)at, (int)lead);
        if ((same >> lane) & 1u) rank = at + lanes_below(same);
        todo &= ~same;
    }
    return rank;
}

// batch body x of world w takes part in the step's items: its place in the
// world's chain (any numbering gives the same results)
__device__ __forceinline__ void chain_touch(const StepDev& S, bool on, uint32_t w, uint32_t x)
{
    bool mine = false;
    if (on && S.cmap[x] == UNTOUCHED) mine = atomicCAS(&S.cmap[x], UNTOUCHED, UNTOUCHED - 1u) == UNTOUCHED;
    const uint32_t c = world_rank(S, mine, w, &WorldChain::bodies);
    if (mine) S.cmap[x] = c;
}

// the step's solver items: their ordering bodies, and the items of each
__global__ void k_items(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    if (S.counters[C_ITEMS] > S.cap_i) { if (grid_tid() == 0) atomicOr(&S.counters[C_OVERFLOW], 8u); return; }
    auto put = [&](uint32_t w, uint32_t item, int32_t r0, int32_t r1) {
        S.it_r0[item] = r0;
        S.it_r1[item] = r1;
        if (r0 >= 0) atomicAdd(&S.deg[r0], 1u);
        if (r1 >= 0) atomicAdd(&S.deg[r1], 1u);
    };
    for (uint32_t j = grid_tid(); j < S.njoints; j += grid_stride()) {
        const uint32_t w = joint_world(S, j);
        const WorldDev& D = S.worlds[w];
        const uint32_t jl = j - D.joint_base;
        const Joint& J = D.joints[jl];
        const int32_t r0 = J.s1 >= 0 ? (int32_t)(D.body_base + J.s1) : -1;
        int32_t r1 = -1;
        if (J.type <= 1 && J.s2 >= 0 && J.s2 != J.s1) r1 = (int32_t)(D.body_base + J.s2);
        put(w, S.w_item_base[w] + jl, r0, r1);
        chain_touch(S, r0 >= 0, w, (uint32_t)r0);
        chain_touch(S, r1 >= 0, w, (uint32_t)r1);
    }
    const uint32_t M = dev_count(&S.counters[C_MANIFOLDS], S.cap_m);
    for (uint32_t m = grid_tid(); m < M; m += grid_stride()) {
        const uint32_t ref = S.m_ref[m], inc = S.m_inc[m], w = S.bworld[ref];
        put(w, S.w_item_base[w] + S.worlds[w].njoints + (m - S.w_man_begin[w]),
            (S.sflag[ref] & SF_RESOURCE) ? (int32_t)ref : -1, (S.sflag[inc] & SF_RESOURCE) ? (int32_t)inc : -1);
        chain_touch(S, true, w, ref);
        chain_touch(S, true, w, inc);
    }
}

__global__ void k_list_fill(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    uint32_t I = dev_count(&S.counters[C_ITEMS], S.cap_i);
    for (uint32_t it = grid_tid(); it < I; it += grid_stride()) {
        int32_t r0 = S.it_r0[it], r1 = S.it_r1[it];
        if (r0 >= 0) { uint32_t p = atomicAdd(&S.deg_fill[r0], 1u); S.lists[S.deg_off[r0] + p] = it * 2u; }
        if (r1 >= 0) { uint32_t p = atomicAdd(&S.deg_fill[r1], 1u); S.lists[S.deg_off[r1] + p] = it * 2u + 1u; }
    }
}

__device__ __forceinline__ uint32_t ld_acq(uint32_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void st_rel(uint32_t* p, uint32_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// the colouring polls global memory (~1 us a poll): its own, smaller limit
constexpr uint32_t COLOR_SPIN_LIMIT = 1u << 22;

// Coloured schedule (a world with r2d_set_schedule(w, 1)): greedy colouring
// of the world's items in item order -- an item takes the smallest colour
// unused by earlier items sharing one of its ordering bodies; past 127
// colours an item takes 128 + its index, a colour of its own.  One workgroup
// per world.  The colouring runs as a dataflow over per-body counters in item
// order: an item waits until every earlier item on its bodies has taken its
// colour.  Worlds in the reference order take no part.
// The counters and the colours used (20 bytes a body) are in LDS under the
// bodies' chain places when they fit, and 1,024 lanes take items in turn: an
// item waits behind its lane's earlier ones, and a poll of global memory is
// about a microsecond (4,096-body pile: 128 -> 34 us).
constexpr uint32_t COLOR_THREADS = 1024;
constexpr size_t COLOR_LDS = 159 * 1024;
__global__ __launch_bounds__(COLOR_THREADS) void k_color(StepDev S, uint32_t lds_words)
{
    extern __shared__ __align__(16) uint32_t smem[];
    __shared__ uint32_t s_abort;
    if (S.counters[C_OVERFLOW]) return;
    const uint32_t w = blockIdx.x;
    const WorldDev& D = S.worlds[w];
    if (D.sched == 0) return;
    const uint32_t i0 = S.w_item_base[w], nit = S.w_item_base[w + 1] - i0, base = D.body_base, t = threadIdx.x;
    const uint32_t nc = S.w_chain[w].bodies;
    auto run = [&](auto mask, auto count, uint32_t n, auto place) {
        for (uint32_t b = t; b < n; b += COLOR_THREADS) {
            mask[2 * b] = 0ull;
            mask[2 * b + 1] = 0ull;
            count[b] = 0u;
        }
        if (t == 0) s_abort = 0u;
        __syncthreads();
        uint32_t spins = 0, cur = ~0u, b0 = 0, b1 = 0, k0 = 0, k1 = 0;
        int32_t r0 = -1, r1 = -1;
        for (uint32_t p = t; p < nit;) {
            const uint32_t it = i0 + p;
            if (p != cur) {
                cur = p;
                r0 = S.it_r0[it]; r1 = S.it_r1[it];
                k0 = S.it_k0[it]; k1 = S.it_k1[it];
                b0 = r0 >= 0 ? place((uint32_t)r0) : 0u;
                b1 = r1 >= 0 ? place((uint32_t)r1) : 0u;
            }
            bool ready = r0 < 0 || ld_acq(&count[b0]) == k0;
            if (ready && r1 >= 0) ready = ld_acq(&count[b1]) == k1;
            if (ready) {
                uint64_t m0 = 0, m1 = 0;
                if (r0 >= 0) { m0 |= mask[2 * b0]; m1 |= mask[2 * b0 + 1]; }
                if (r1 >= 0) { m0 |= mask[2 * b1]; m1 |= mask[2 * b1 + 1]; }
                uint32_t c;
                if (~m0) c = (uint32_t)__builtin_ctzll(~m0);
                else if (~m1) c = 64u + (uint32_t)__builtin_ctzll(~m1);
                else c = 128u + p;
                S.it_color[it] = c;
                if (c < 128) {
                    const uint32_t hi = c >> 6;
                    const uint64_t bit = 1ull << (c & 63u);
                    if (r0 >= 0) mask[2 * b0 + hi] |= bit;
                    if (r1 >= 0) mask[2 * b1 + hi] |= bit;
                }
                if (r0 >= 0) st_rel(&count[b0], k0 + 1u);
                if (r1 >= 0) st_rel(&count[b1], k1 + 1u);
                p += COLOR_THREADS;
                spins = 0;
            } else {
                // every item's predecessors come first, so some item is always ready
                if (__hip_atomic_load(&s_abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) break;
                if (++spins > COLOR_SPIN_LIMIT) {
                    __hip_atomic_store(&s_abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    S.w_status[w] = 5;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
    };
    if (5u * nc <= lds_words)
        run((uint64_t*)smem, smem + 4u * nc, nc, [&](uint32_t r) { return S.cmap[r]; });
    else
        run(S.cmask + 2 * (size_t)base, S.g_cnt + base, (uint32_t)D.nbodies, [&](uint32_t r) { return r - base; });
}

// rank of each item among the items sharing one of its resources: in item
// order (the reference's sequential order: constraints, then manifolds in
// discovery order); with BY_COLOR, for bodies of coloured worlds, in
// (colour, item) order
template <bool BY_COLOR>
__global__ void k_list_rank(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    for (uint32_t x = grid_tid(); x < S.nb; x += grid_stride()) {
        if (BY_COLOR && S.worlds[S.bworld[x]].sched == 0) continue;
        uint32_t o = S.deg_off[x], n = S.deg_off[x + 1] - o;
        uint32_t* l = S.lists + o;
        auto key = [&](uint32_t v) -> uint64_t {
            return BY_COLOR ? (((uint64_t)S.it_color[v >> 1] << 32) | v) : (uint64_t)v;
        };
        for (uint32_t i = 1; i < n; ++i) {
            uint32_t v = l[i];
            uint64_t kv = key(v);
            uint32_t j = i;
            while (j > 0 && key(l[j - 1]) > kv) { l[j] = l[j - 1]; --j; }
            l[j] = v;
        }
        for (uint32_t p = 0; p < n; ++p) {
            uint32_t v = l[p];
            if (v & 1u) S.it_k1[v >> 1] = p; else S.it_k0[v >> 1] = p;
        }
    }
}

// ---------------------------------------------------------------- solver
// The body arrays that the per-body passes of a sub-step read and write,
// copied out of the world's descriptor once per pass and typed by address
// space: global for the body arrays (their loads and stores then wait on the
// memory counter alone; a generic pointer's wait also covers LDS operations),
// constant for the force generators, which no kernel writes (scalar loads,
// one per generator for the whole wave).  Through a reference to the
// descriptor in global memory the compiler reloads every pointer for every
// body, since it cannot tell that the pass's own stores leave it unchanged.
typedef __attribute__((address_space(1))) float* GlbF;
typedef const __attribute__((address_space(1))) float* GlbCF;
typedef const __attribute__((address_space(1))) uint32_t* GlbCU;
typedef const __attribute__((address_space(4))) Gen* ConstGen;
struct BodyArrays {
    GlbF px, py, ang, fx, fy, tq, ax, ay, ahw, ahh;
    GlbCF mass, inertia, rad, hw, hh;
    GlbCU flags;
    GlbCF wsum;                      // the world's float4 warm sums, as floats
    ConstGen gens;
    int32_t ngens;
    float warm;
};
__device__ __forceinline__ BodyArrays body_arrays(const WorldDev& D)
{
    return BodyArrays{(GlbF)D.px, (GlbF)D.py, (GlbF)D.ang, (GlbF)D.fx, (GlbF)D.fy, (GlbF)D.tq, (GlbF)D.ax,
                      (GlbF)D.ay, (GlbF)D.ahw, (GlbF)D.ahh, (GlbCF)D.mass, (GlbCF)D.inertia, (GlbCF)D.rad,
                      (GlbCF)D.hw, (GlbCF)D.hh, (GlbCU)D.flags, (GlbCF)(const float*)D.wsum, (ConstGen)D.gens,
                      D.ngens, D.warm};
}

// body i's warm impulse per sub-step (momentum x, y, angular: the first
// three floats of its float4)
__device__ __forceinline__ GlbCF warm_sum(const BodyArrays& D, int i) { return D.wsum + 4 * i; }

// ------------------------------------------------------------ warm starting
// Opt-in, not in the reference (its roadmap item "persist manifolds across
// frames by keying with stable body IDs", README.md:60-61).  After a step
// every manifold is kept under the lower slot of its two bodies (WARM_K
// entries per body, discovery order); at the next step a manifold with the
// same (ref id, inc id), the same points, a normal within WARM_DOT of the old
// one and no live updateTGSDepth point carries warm * acc / sub_steps of each
// point's impulses into every sub-step: added to its accumulators before the
// iterations, and applied to its bodies with the forces.

// manifold m (step index): match against its lower body's table; the points'
// impulses per sub-step to MP_WARM_N / MP_WARM_T, MV_WARM on a match
__device__ __forceinline__ void warm_match(const StepDev& S, const WorldDev& D, uint32_t m, uint32_t base,
                                           uint32_t sub_steps)
{
    const size_t cm = S.cap_m;
    float* P = S.m_pt;
    const uint32_t valid = S.m_valid[m] & 3u;
    const uint32_t a = S.m_ref[m] - base, b = S.m_inc[m] - base;
    const uint32_t lo = umin(a, b);
    const v2 n = mk(S.m_nx[m], S.m_ny[m]);
    bool live = false;
#pragma unroll
    for (int p = 0; p < 2; ++p)
        if (valid & (1u << p)) live |= !approx(P[(MP_DEPTH * 2 + p) * cm + m], P[(MP_ODEPTH * 2 + p) * cm + m], 1e-4f);
    float g[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    bool hit = false;
    if (!live) {
        const uint32_t ida = D.id[a], idb = D.id[b];
        const uint32_t c = umin(D.wcnt[lo], WARM_K);
        const uint4* e = D.wtab + (size_t)lo * WARM_K * 3;
        for (uint32_t k = 0; k < c; ++k, e += 3) {
            const uint4 h = e[0];
            if (h.x != ida || h.y != idb) continue;
            const uint4 q = e[1], r = e[2];
            const float d = dot2(n, mk(__uint_as_float(h.w), __uint_as_float(q.x)));
            if (h.z == valid && d >= WARM_DOT) {
                hit = true;
                const float acc[4] = {__uint_as_float(q.y), __uint_as_float(q.z), __uint_as_float(q.w),
                                      __uint_as_float(r.x)};
                const float ss = (float)sub_steps;
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    if (!(valid & (1u << p)) || !(P[(MP_DEPTH * 2 + p) * cm + m] < 0.0f)) continue;
                    g[2 * p] = (D.warm * acc[2 * p]) / ss;
                    g[2 * p + 1] = (D.warm * acc[2 * p + 1]) / ss;
                }
            }
            break;
        }
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        P[(MP_WARM_N * 2 + p) * cm + m] = g[2 * p];
        P[(MP_WARM_T * 2 + p) * cm + m] = g[2 * p + 1];
    }
    if (hit) S.m_valid[m] = valid | MV_WARM;
}

// body x (world slot) from its item list (entries item * 2 + side, items
// counted from ibase, in item order): the sum, in that order, of its matched
// manifolds' carried impulses, as calculateImpulses applies them
// (collision.zig:200-217): the reference body gets -dp, -r1 x dp, the
// incident body +dp, +r2 x dp
__device__ __forceinline__ void warm_body_sum(const StepDev& S, const WorldDev& D, const uint32_t* list, uint32_t cnt,
                                              uint32_t x, uint32_t ibase, uint32_t nj, uint32_t mbeg)
{
    const size_t cm = S.cap_m;
    const float* P = S.m_pt;
    float sx = 0.0f, sy = 0.0f, sl = 0.0f;
    for (uint32_t i = 0; i < cnt; ++i) {
        const uint32_t v = list[i], j = (v >> 1) - ibase;
        if (j < nj) continue;
        const uint32_t m = mbeg + (j - nj);
        const uint32_t valid = S.m_valid[m];
        if (!(valid & MV_WARM)) continue;
        const v2 n = mk(S.m_nx[m], S.m_ny[m]), t = rot90cw(n);
        for (int p = 0; p < 2; ++p) {
            if (!(valid & (1u << p))) continue;
            const v2 dp = add2(scale2(n, P[(MP_WARM_N * 2 + p) * cm + m]), scale2(t, P[(MP_WARM_T * 2 + p) * cm + m]));
            if (v & 1u) {
                const v2 r2 = mk(P[(MP_R2X * 2 + p) * cm + m], P[(MP_R2Y * 2 + p) * cm + m]);
                sx += dp.x; sy += dp.y; sl += cross2(r2, dp);
            } else {
                const v2 r1 = mk(P[(MP_R1X * 2 + p) * cm + m], P[(MP_R1Y * 2 + p) * cm + m]);
                sx -= dp.x; sy -= dp.y; sl -= cross2(r1, dp);
            }
        }
    }
    D.wsum[x] = make_float4(sx, sy, sl, 0.0f);
}

// after the step: manifold m of the world's [mbeg, mend) into its lower
// body's table at its rank among that body's manifolds (contiguous in
// discovery order: a pair is found from its lower slot); the last of them
// sets the count.  The world's counts are zero beforehand.
__device__ __forceinline__ void warm_save(const StepDev& S, const WorldDev& D, uint32_t m, uint32_t mbeg,
                                          uint32_t mend, uint32_t base)
{
    auto lo_of = [&](uint32_t k) { return umin(S.m_ref[k], S.m_inc[k]) - base; };
    const uint32_t lo = lo_of(m);
    uint32_t k = 0;
    while (k < WARM_K && m - k > mbeg && lo_of(m - k - 1) == lo) ++k;
    if (m + 1 == mend || lo_of(m + 1) != lo) D.wcnt[lo] = umin(k + 1, WARM_K);
    if (k >= WARM_K) return;
    const size_t cm = S.cap_m;
    const float* P = S.m_pt;
    uint4* e = D.wtab + ((size_t)lo * WARM_K + k) * 3;
    const uint32_t a = S.m_ref[m] - base, b = S.m_inc[m] - base;
    e[0] = make_uint4(D.id[a], D.id[b], S.m_valid[m] & 3u, __float_as_uint(S.m_nx[m]));
    e[1] = make_uint4(__float_as_uint(S.m_ny[m]), __float_as_uint(P[(MP_ACC_PN * 2 + 0) * cm + m]),
                      __float_as_uint(P[(MP_ACC_PT * 2 + 0) * cm + m]), __float_as_uint(P[(MP_ACC_PN * 2 + 1) * cm + m]));
    e[2] = make_uint4(__float_as_uint(P[(MP_ACC_PT * 2 + 1) * cm + m]), 0u, 0u, 0u);
}

// ---------------------------------- warm starting in the phase kernels
// grid-wide over the step's manifolds / bodies; worlds without warm starting
// (and stopped worlds) are skipped

// after the per-body item lists: the matches, then each body's sum
__global__ void k_warm_match(StepDev S, uint32_t sub_steps)
{
    if (S.counters[C_OVERFLOW]) return;
    const uint32_t M = dev_count(&S.counters[C_MANIFOLDS], S.cap_m);
    for (uint32_t m = grid_tid(); m < M; m += grid_stride()) {
        const uint32_t w = S.bworld[S.m_ref[m]];
        const WorldDev& D = S.worlds[w];
        if (D.warm > 0.0f && S.w_status[w] == 0) warm_match(S, D, m, D.body_base, sub_steps);
    }
}

__global__ void k_warm_sums(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    for (uint32_t x = grid_tid(); x < S.nb; x += grid_stride()) {
        const uint32_t w = S.bworld[x];
        const WorldDev& D = S.worlds[w];
        if (!(D.warm > 0.0f) || S.w_status[w] != 0) continue;
        const uint32_t o = S.deg_off[x];
        warm_body_sum(S, D, S.lists + o, S.deg_off[x + 1] - o, x - D.body_base, S.w_item_base[w],
                      (uint32_t)D.njoints, S.w_man_begin[w]);
    }
}

// after the solve: clear the tables' counts, then store the manifolds
__global__ void k_warm_clear(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    for (uint32_t x = grid_tid(); x < S.nb; x += grid_stride()) {
        const uint32_t w = S.bworld[x];
        const WorldDev& D = S.worlds[w];
        if (D.warm > 0.0f && S.w_status[w] == 0) D.wcnt[x - D.body_base] = 0u;
    }
}

__global__ void k_warm_save(StepDev S)
{
    if (S.counters[C_OVERFLOW]) return;
    const uint32_t M = dev_count(&S.counters[C_MANIFOLDS], S.cap_m);
    for (uint32_t m = grid_tid(); m < M; m += grid_stride()) {
        const uint32_t w = S.bworld[S.m_ref[m]];
        const WorldDev& D = S.worlds[w];
        if (D.warm > 0.0f && S.w_status[w] == 0)
            warm_save(S, D, m, S.w_man_begin[w], S.w_man_begin[w + 1], D.body_base);
    }
}

// ------------------------------------------------------ fused world steps
// Worlds of at most FUSED_NMAX bodies in the reference order can take whole
// steps in one workgroup: broadphase, narrowphase, schedule and solve of the
// world with workgroup barriers between the phases instead of kernel
// boundaries, and all the steps of a call in one launch (worlds are
// independent, so nothing crosses workgroups).  Each phase computes for its
// world exactly what the grid-wide kernels above compute: the same
// per-element functions (prep_body, narrow_pair, man_build_one, the solve
// paths) over the world's own scratch slices (WorldScratch), with the
// per-body and per-bucket arrays in LDS.

// The stale AABBs (aabb.zig:6-8) and flags of a world's bodies in LDS,
// for the pair filters of the fused broadphase
struct PairCache {
    float *ax, *ay, *ahw, *ahh;
    uint32_t* flags;
};
constexpr uint32_t PAIR_CACHE_WORDS = 5;   // per body

__device__ __forceinline__ PairCache pair_cache(uint32_t* p, uint32_t n)
{
    return PairCache{(float*)p, (float*)p + n, (float*)p + 2 * n, (float*)p + 3 * n, p + 4 * n};
}

// updateManifolds' pair filters that need no more than the cache: both
// bodies static (lib.zig:273), padded AABB overlap (lib.zig:282)
__device__ __forceinline__ uint32_t pair_passes(const PairCache& P, uint32_t a, uint32_t b)
{
    if ((P.flags[a] & BF_STATIC) && (P.flags[b] & BF_STATIC)) return 0u;
    return aabb_hit(P, a, b) ? 1u : 0u;
}

// The raw candidates of one cell entry of body a: the distinct members of
// its bucket above a (s[0, c), members in descending order, a body's repeats
// adjacent) that pass pair_passes, as the serial walk
//   for (j = 0; j < c && s[j] > a; ++j)
//       if (j == 0 || s[j] != s[j - 1]) { ok = pair_passes(P, a, s[j]); ... }
// counts them: their number, and the passing positions below 32 as a mask.
// Four members at a time, so the filters' LDS loads of four bodies are in
// flight together instead of one body's at a time.
__device__ __forceinline__ void entry_candidates(const PairCache& P, uint32_t a, const uint32_t* s, uint32_t c,
                                                 uint32_t& q_out, uint32_t& mask_out)
{
    uint32_t q = 0, mask = 0, prev = 0;
    for (uint32_t j = 0; j < c; j += 4) {
        uint32_t m[4];
        bool live[4];
        bool stop = false;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) m[k] = j + k < c ? s[j + k] : 0u;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const bool above = j + k < c && m[k] > a;
            const uint32_t before = k ? m[k - 1] : prev;
            live[k] = !stop && above && (j + k == 0 || m[k] != before);
            stop = stop || !above;
        }
        uint32_t ok[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) ok[k] = pair_passes(P, a, m[k]);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const bool pass = live[k] && ok[k] != 0u;
            q += pass;
            if (pass && j + k < 32u) mask |= 1u << (j + k);
        }
        if (stop) break;
        prev = m[3];
    }
    q_out = q;
    mask_out = mask;
}

// LDS of the fused kernel for a world of n bodies and tb hash buckets
struct FusedLds {
    uint32_t* dcnt;    // [n] solver items per ordering body
    uint32_t* doff;    // [n+1] -> list offsets
    uint32_t* dfill;   // [n]
    uint32_t* coff;    // [n+1] cells per body -> entry offsets
    float *cc, *cs;    // [n] cos / sin of the angle at step start
    uint32_t* boff;    // [tb+1] bucket occupancy -> bucket offsets
    uint32_t* bfill;   // [tb]
    uint32_t* pairs;   // [5 n] pair cache, then the entries' buckets and bucket members when they fit
};

// front part of a world's fused LDS (before the pair cache), in words
__host__ __device__ constexpr uint32_t fused_front_words(uint32_t n, uint32_t tb) { return 6u * n + 2u * tb + 3u; }
// the part of it that the solve still reads (dcnt, doff), 16-byte aligned
__host__ __device__ constexpr uint32_t fused_keep_words(uint32_t n) { return (2u * n + 4u) & ~3u; }

__device__ __forceinline__ FusedLds fused_carve(uint32_t* lds, uint32_t n, uint32_t tb)
{
    FusedLds L;
    uint32_t* p = lds;
    L.dcnt = p; p += n;
    L.doff = p; p += n + 1;
    L.dfill = p; p += n;
    L.coff = p; p += n + 1;
    L.cc = (float*)p; p += n;
    L.cs = (float*)p; p += n;
    L.boff = p; p += tb + 1;
    L.bfill = p; p += tb;
    L.pairs = p;
    return L;
}

// Words per body after the front part: the pair cache and room for the
// bucket arrays.  The solve then has the whole of LDS but dcnt and doff: 16
// words a body with 2 n buckets, 7 of them momenta and poses, and in the rest
// the plan (5 words an item), then 3 words a body and the impulses (2 a
// point).  A world of 500 bodies takes 36 KB: four to a CU.
constexpr uint32_t FUSED_TAIL_WORDS = 8;
// Least dynamic LDS of a launch: room for the plan of a small world with many
// joints, and no cost: the registers allow four workgroups a CU at most.
constexpr size_t FUSED_LDS_MIN = 24 * 1024;

size_t fused_lds_bytes(uint32_t n, uint32_t tb)
{
    return std::max<size_t>(FUSED_LDS_MIN, (fused_front_words(n, tb) + (size_t)FUSED_TAIL_WORDS * n) * 4u);
}

// The fused kernel's narrowphase test of one candidate, as a call: out of
// line, its registers are allocated apart from the step kernel's, which
// spills less.  It takes only pointers and values (no reference to the
// kernel's argument block, which would be copied to scratch).
__device__ __attribute__((noinline)) bool narrow_pair_call(const WorldDev& D, uint32_t sa, uint32_t sb, uint32_t k,
                                                         const uint32_t* ba, const uint32_t* bb, uint32_t nb,
                                                         float ca, float sa_sin, float cb, float sb_sin,
                                                         uint32_t& info, float& nx, float& ny)
{
    return narrow_pair<true>(D, D, sa, sb, k, ba, bb, nb, ca, sa_sin, cb, sb_sin, info, nx, ny);
}

// exclusive scan of a[0, len) in place (LDS or global), a[len] = the total,
// which is returned; called by the whole workgroup after a barrier, ends
// with one
__device__ __forceinline__ uint32_t group_scan(uint32_t* a, uint32_t len, uint32_t* sm)
{
    const uint32_t T = blockDim.x, t = threadIdx.x;
    const uint32_t chunk = (len + T - 1) / T;
    const uint32_t lo = umin(t * chunk, len), hi = umin(lo + chunk, len);
    uint32_t sum = 0;
    for (uint32_t i = lo; i < hi; ++i) sum += a[i];
    uint32_t total;
    uint32_t run = block_excl_scan(sum, sm, &total);
    for (uint32_t i = lo; i < hi; ++i) {
        uint32_t x = a[i];
        a[i] = run;
        run += x;
    }
    if (t == 0) a[len] = total;
    __syncthreads();
    return total;
}

// A world's slice of family k (0 cell entries, 1 raw candidates, 2
// manifolds, 3 solver items) is too small for `need` elements: the world
// moves to a larger slice taken from the free end of the arrays (S.fpool).
// False when the arrays are full; the world then stops (fused_overflow).
// Called by the whole workgroup; the slice table entry is updated for the host.
// Inlined: as a call it takes the kernel's StepDev by reference, and the
// kernel then copies its whole argument block to scratch at entry.
__device__ __forceinline__ bool fused_grow(const StepDev& S, uint32_t w, WorldScratch& X, int k, uint32_t need,
                                           uint32_t& s_slot)
{
    const uint32_t cap = need + need / 2 + 64;
    const uint32_t take = k != 2 ? cap + 1 : cap;   // entry and candidate slices end with a scan total, item slices with
                                                    // the chain's idle point
    if (threadIdx.x == 0) {
        // claim [base, base + take) only if it fits: a refused request leaves
        // the free end for smaller ones
        const uint32_t lim = S.fpool[4 + k];
        uint32_t base = __hip_atomic_load(&S.fpool[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (;;) {
            if (base > lim || take > lim - base) { base = 0xffffffffu; break; }
            const uint32_t seen = atomicCAS(&S.fpool[k], base, base + take);
            if (seen == base) break;
            base = seen;
        }
        s_slot = base;
    }
    __syncthreads();
    const uint32_t base = s_slot;
    __syncthreads();
    if (base == 0xffffffffu) return false;
    if (k == 0) { X.e0 = base; X.ecap = cap; }
    else if (k == 1) { X.r0 = base; X.rcap = cap; }
    else if (k == 2) { X.m0 = base; X.mcap = cap; }
    else { X.i0 = base; X.icap = cap; }
    if (threadIdx.x == 0) S.wscr[w] = X;
    return true;
}

// A world's scratch slice is too small for this step and the arrays are
// full: record what it needs and stop the world before its state changes
// (the host grows the arrays and runs the remaining steps)
__device__ __forceinline__ void fused_overflow(const StepDev& S, uint32_t w, uint32_t e, uint32_t r, uint32_t m,
                                               uint32_t it)
{
    if (threadIdx.x == 0) {
        uint32_t* c = S.w_cnt + 8 * (size_t)w;
        c[4] = e; c[5] = r; c[6] = m; c[7] = it;
        S.w_status[w] = WS_OVERFLOW;
    }
}

// ------------------------------------------------- the solve of a fused step
// what the gap between two chains reads of a world's bodies, in LDS or global
template <class F, class U>
struct BodyPoses {
    F px, py, ang, mass, inertia;
    U flags;
};
// a world's bodies in LDS during its sub-steps: momenta (16 bytes a body and a
// spare one), position and angle, then mass, inertia and flags
struct ChainBodies : BodyPoses<LF, LU32> {
    LF3 m;
};

// contact point record (words as in r2d_chain.h); the bodies' inverse masses
// and inertias are 0 for static ones
struct PointBodies {
    uint32_t a, b, flag_a, flag_b;
    float im1, im2, ii1, ii2;
};

// effective masses of a point (CollisionManifold.preStep, collision.zig:117-132)
__device__ __forceinline__ void point_masses(const PointBodies& B, v2 n, v2 r1, v2 r2, float& mn, float& mt)
{
    const v2 t = rot90cw(n);
    const float inv_mass = B.im1 + B.im2;
    const float r1n = cross2(r1, n), r2n = cross2(r2, n);
    const float kn = inv_mass + B.ii1 * (r1n * r1n) + B.ii2 * (r2n * r2n);
    const float r1t = cross2(r1, t), r2t = cross2(r2, t);
    const float kt = inv_mass + B.ii1 * (r1t * r1t) + B.ii2 * (r2t * r2t);
    mn = kn > 0.0f ? 1.0f / kn : 0.0f;
    mt = kt > 0.0f ? 1.0f / kt : 0.0f;
}

// Baumgarte bias of a sub-step of length dt (collision.zig:172), -1 for a
// point whose depth is >= 0 (calculateImpulses resets and skips it)
__device__ __forceinline__ float point_bias(float depth, float dt)
{
    return depth >= 0.f ? -1.0f : BAUMGARTE * maxn(0.0f, (-depth) - BAUMGARTE_SLOP) / dt;
}

__device__ __forceinline__ void point_store(u4v* recs, uint32_t at, const PointBodies& B, bool second, v2 n, float fric,
                                            float bias, v2 r1, v2 r2, float mn, float mt)
{
    u4v* q = recs + (size_t)at * 4u;
    const uint32_t drop = second ? ~(uint32_t)PR_WRITE : ~0u;   // the first point writes the bodies
    q[0] = u4v{B.a | (B.flag_a & drop), B.b | (B.flag_b & drop), asu(n.x), asu(n.y)};
    q[1] = u4v{asu(fric), asu(bias), asu(r1.x), asu(r1.y)};
    q[2] = u4v{asu(r2.x), asu(r2.y), asu(mn), asu(mt)};
    q[3] = u4v{asu(B.im1), asu(B.im2), asu(B.ii1), asu(B.ii2)};
}

// the ordering bodies' flags and inverse masses of manifold m's bodies
// (world slots a, b)
__device__ __forceinline__ PointBodies point_bodies(const StepDev& S, const WorldDev& D, uint32_t base, uint32_t a, uint32_t b)
{
    PointBodies B;
    B.a = a;
    B.b = b;
    const bool sa = (D.flags[a] & BF_STATIC) != 0, sb = (D.flags[b] & BF_STATIC) != 0;
    const bool wa = (S.sflag[base + a] & SF_RESOURCE) != 0, wb = (S.sflag[base + b] & SF_RESOURCE) != 0;
    const float m1 = D.mass[a], m2 = D.mass[b], i1 = D.inertia[a], i2 = D.inertia[b];
    B.flag_a = (wa ? PR_WRITE : 0u) | (sa ? PR_STATIC : 0u);
    B.flag_b = (wb ? PR_WRITE : 0u) | (sb ? PR_STATIC : 0u);
    B.im1 = sa ? 0.0f : 1.0f / m1;
    B.im2 = sb ? 0.0f : 1.0f / m2;
    B.ii1 = sa ? 0.0f : 1.0f / i1;
    B.ii2 = sb ? 0.0f : 1.0f / i2;
    return B;
}

// The records of manifold m (item j of its world; a second point at p1), and
// what preStep leaves in the manifold: friction and effective masses.
// Returns whether updateTGSDepth is live for it: a point whose depth is not
// within 1e-4 of its original depth, which at the step's start is the same
// number, so NaN or so deep that 1e-4 vanishes in it (1), and whether the
// chain needs the reference's sums to the letter (2): one of its bodies is
// static and an ordering body, or a normal or an arm is not finite.
// place(slot): where the
// chain keeps a body's momentum.
template <bool WARM, class PLACE>
__device__ __forceinline__ uint32_t point_build(const StepDev& S, const WorldDev& D, u4v* recs, uint32_t m, uint32_t base,
                                            uint32_t j, uint32_t p1, float sub_dt, PLACE place)
{
    const size_t cm = S.cap_m;
    float* P = S.m_pt;
    const uint32_t a = S.m_ref[m] - base, b = S.m_inc[m] - base, valid = S.m_valid[m];
    const v2 n = mk(S.m_nx[m], S.m_ny[m]);
    v2 r1[2], r2[2];
    float depth[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {   // in bounds whether or not the point exists
        r1[p] = mk(P[(MP_R1X * 2 + p) * cm + m], P[(MP_R1Y * 2 + p) * cm + m]);
        r2[p] = mk(P[(MP_R2X * 2 + p) * cm + m], P[(MP_R2Y * 2 + p) * cm + m]);
        depth[p] = P[(MP_DEPTH * 2 + p) * cm + m];
    }
    const float mua = D.mu[a], mub = D.mu[b];
    PointBodies B = point_bodies(S, D, base, a, b);
    B.a = place(a);
    B.b = place(b);
    if (WARM && (valid & MV_WARM)) B.flag_b |= PR_WARM;
    const float fric = sqrt_rn(mua * mub);   // preStep (collision.zig:114)
    S.m_fric[m] = fric;
    bool live = false, finite = true;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const bool on = (valid & (1u << p)) != 0u;
        if (!on && p == 1) continue;
        if (on) finite = finite && 0.f * n.x + 0.f * n.y + 0.f * r1[p].x + 0.f * r1[p].y + 0.f * r2[p].x + 0.f * r2[p].y == 0.f;
        float mn = 0.f, mt = 0.f;
        if (on) {
            point_masses(B, n, r1[p], r2[p], mn, mt);
            P[(MP_MASS_N * 2 + p) * cm + m] = mn;
            P[(MP_MASS_T * 2 + p) * cm + m] = mt;
            live = live || !approx(depth[p], depth[p], 1e-4f);
        }
        // a manifold without points keeps one record that adds 0 to its bodies
        const v2 z = mk(0.f, 0.f);
        point_store(recs, p ? p1 : j, B, p != 0, n, fric, on ? point_bias(depth[p], sub_dt) : -1.0f, on ? r1[p] : z,
                    on ? r2[p] : z, mn, mt);
    }
    const uint32_t both = PR_WRITE | PR_STATIC;
    return (live ? 1u : 0u) | ((B.flag_a & both) == both || (B.flag_b & both) == both || !finite ? 2u : 0u);
}

// updateTGSDepth (collision.zig:73-100) for manifold m where it is live:
// rotate lever arms by the bodies' rotation since the previous sub-step,
// recompute depth and (preStep) the effective masses, in the step's arrays
// and the records; reset(p): point p is separated now, its impulses are reset
// (calculateImpulses does so in the sub-step's first iteration)
template <class POSES, class RESET>
__device__ __forceinline__ void point_tgs(const StepDev& S, const WorldDev& D, u4v* recs, const POSES& C, uint32_t m,
                                          uint32_t base, uint32_t j, uint32_t p1, float sub_dt, RESET reset)
{
    const size_t cm = S.cap_m;
    float* P = S.m_pt;
    const uint32_t valid = S.m_valid[m];
    bool live = false;
    for (int p = 0; p < 2; ++p) {
        const float od = P[(MP_ODEPTH * 2 + p) * cm + m];
        live = live || ((valid & (1u << p)) && !approx(od, od, 1e-4f));
    }
    if (!live) return;
    const uint32_t a = S.m_ref[m] - base, b = S.m_inc[m] - base;
    const v2 n = mk(S.m_nx[m], S.m_ny[m]);
    const float a1 = C.ang[a], a2 = C.ang[b], prev1 = S.m_prev1[m], prev2 = S.m_prev2[m];
    const PointBodies B = point_bodies(S, D, base, a, b);
    for (int p = 0; p < 2; ++p) {
        if (!(valid & (1u << p))) continue;
        const float od = P[(MP_ODEPTH * 2 + p) * cm + m];
        if (approx(P[(MP_DEPTH * 2 + p) * cm + m], od, 1e-4f)) continue;
        const v2 r1 = rotate2(mk(P[(MP_R1X * 2 + p) * cm + m], P[(MP_R1Y * 2 + p) * cm + m]), a1 - prev1);
        const v2 r2 = rotate2(mk(P[(MP_R2X * 2 + p) * cm + m], P[(MP_R2Y * 2 + p) * cm + m]), a2 - prev2);
        const v2 q1 = add2(r1, mk(C.px[a], C.py[a])), q2 = add2(r2, mk(C.px[b], C.py[b]));
        const float depth = dot2(n, sub2(q2, q1)) + od;
        float mn, mt;
        point_masses(B, n, r1, r2, mn, mt);
        P[(MP_R1X * 2 + p) * cm + m] = r1.x; P[(MP_R1Y * 2 + p) * cm + m] = r1.y;
        P[(MP_R2X * 2 + p) * cm + m] = r2.x; P[(MP_R2Y * 2 + p) * cm + m] = r2.y;
        P[(MP_DEPTH * 2 + p) * cm + m] = depth;
        P[(MP_MASS_N * 2 + p) * cm + m] = mn;
        P[(MP_MASS_T * 2 + p) * cm + m] = mt;
        if (depth >= 0.f) reset(p);
        u4v* q = recs + (size_t)(p ? p1 : j) * 4u;
        q[1] = u4v{q[1].x, asu(point_bias(depth, sub_dt)), asu(r1.x), asu(r1.y)};
        q[2] = u4v{asu(r2.x), asu(r2.y), asu(mn), asu(mt)};
    }
    S.m_prev1[m] = a1;
    S.m_prev2[m] = a2;
}

// The record of joint J for a sub-step: everything its solve reads besides
// momenta is fixed within a sub-step (poses after the previous sub-step's
// position integration; torque as set for this one), so the terms that
// Constraints/*.zig derive from it are computed here, once, in their order.
template <class POSES, class PLACE>
__device__ __forceinline__ void joint_record(u4v* q, const Joint& J, const WorldDev& D, const POSES& C, bool first,
                                             PLACE place)
{
    const uint32_t type = (uint32_t)J.type, a = (uint32_t)J.s1, b = type <= 1u ? (uint32_t)J.s2 : a;
    u4v q0{PR_JOINT, type << PR_TYPE_SHIFT, 0u, 0u}, q1{}, q2{}, q3{};
    if (J.s1 < 0 || (type <= 1u && J.s2 < 0)) {   // a removed body: refused before any solve
        q0.x |= PR_SKIP;
        q[0] = q0;
        return;
    }
    const bool sa = (C.flags[a] & BF_STATIC) != 0, sb = (C.flags[b] & BF_STATIC) != 0;
    q0.x |= place(a) | (type <= 1u && a == b ? PR_SELF : 0u);
    q0.y |= place(b);
    q1.y = asu(J.pmin);
    q1.z = asu(J.pmax);
    const float im1 = sa ? 0.0f : 1.0f / C.mass[a], im2 = sb ? 0.0f : 1.0f / C.mass[b];
    const v2 pa = mk(C.px[a], C.py[a]), pb = mk(C.px[b], C.py[b]);
    q3.x = asu(im1);
    q3.y = asu(im2);
    if (type == 0u) {
        const v2 n = normalize2(sub2(pb, pa));
        const float dist_err = length2(sub2(pb, pa)) - J.target;
        q0.z = asu(n.x);
        q0.w = asu(n.y);
        q1.x = asu(J.beta * dist_err / maxn(J.target, 0.001f));
    } else if (type == 1u) {
        const float ta = C.ang[a], tb = C.ang[b];
        const v2 rr1 = rotcs(mk(J.r1x, J.r1y), cosf_r(ta), sinf_r(ta));
        const v2 rr2 = rotcs(mk(J.r2x, J.r2y), cosf_r(tb), sinf_r(tb));
        const v2 a1 = add2(rr1, pa), a2 = add2(rr2, pb);
        const v2 n = normalize2(sub2(a2, a1));
        const float ii1 = sa ? 0.0f : 1.0f / C.inertia[a], ii2 = sb ? 0.0f : 1.0f / C.inertia[b];
        const float dist_err = length2(sub2(a2, a1)) - J.target;
        const float r1xn = cross2(rr1, n), r2xn = cross2(rr2, n);
        q0.z = asu(n.x);
        q0.w = asu(n.y);
        q1.x = asu(J.beta * dist_err / maxn(J.target, GRAD_DIV_LIMIT));
        q1.w = asu(rr1.x);
        q2 = u4v{asu(rr1.y), asu(rr2.x), asu(rr2.y), asu(im1 + im2 + r1xn * r1xn * ii1 + r2xn * r2xn * ii2)};
        q3.z = asu(ii1);
        q3.w = asu(ii2);
    } else if (type == 2u) {
        const v2 delta = sub2(mk(J.tx, J.ty), pa);
        const float dist = length2(delta);
        if (sa || dist < ALLOWED_CONSTRAINT_VALUE) q0.x |= PR_SKIP;
        const v2 n = scale2(delta, 1.0f / dist);
        q0.z = asu(n.x);
        q0.w = asu(n.y);
        q1.x = asu(J.beta * dist);
    } else {
        if (sa) q0.x |= PR_SKIP;
        q0.z = asu(C.inertia[a]);
        q0.w = asu(J.target);
        q1.x = asu(J.beta);
        q1.w = asu(first ? D.tq[a] : 0.0f);
    }
    q[0] = q0; q[1] = q1; q[2] = q2; q[3] = q3;
}

// what a body's first pass reads of it beyond LDS
struct BodyIn {
    uint32_t f;
    float mass, inertia, fx, fy, tq;
};

// Body i's part of the gap between two chains: the position integration of
// sub-step s - 1 (lib.zig:238-249; body_move), then the forces, AABB refresh
// and velocity integration of sub-step s (lib.zig:200-216; body_push).  In
// between a dynamic body's force and torque are zero, so they need no memory;
// only the last sub-step's AABB is observable.  After the last chain: the
// positions, and the state back to global memory (body_done).
struct BodyState {
    f3v m;
    float px, py, ang;
};
__device__ __forceinline__ void body_move(BodyState& b, float mass, float inertia, float sub_dt)
{
    const float qd = sub_dt / mass;
    b.px = b.px + b.m.x * qd;
    b.py = b.py + b.m.y * qd;
    b.ang = b.ang + b.m.z * sub_dt / inertia;
}

__device__ __forceinline__ void body_done(const WorldDev& D, const BodyArrays& A, int i, bool stat, const BodyState& b)
{
    D.mx[i] = b.m.x; D.my[i] = b.m.y; D.L[i] = b.m.z;
    if (!stat) {
        A.px[i] = b.px; A.py[i] = b.py; A.ang[i] = b.ang;
        A.fx[i] = 0.0f; A.fy[i] = 0.0f; A.tq[i] = 0.0f;
    }
}

// a momentum component of -0: the chain then needs the reference's sums to the letter
__device__ __forceinline__ bool minus_zero(f3v m)
{
    return asu(m.x) == 0x80000000u || asu(m.y) == 0x80000000u || asu(m.z) == 0x80000000u;
}

template <bool WARM>
__device__ __forceinline__ f3v body_push(const BodyArrays& A, int i, bool last, const BodyState& b, BodyIn in, float sub_dt)
{
    const bool stat = (in.f & BF_STATIC) != 0;
    if (last) {
        // Disc.updateAABB / Rectangle.updateAABB
        float hw, hh;
        if (in.f & BF_RECT) {
            const float c = cosf_r(b.ang), sn = sinf_r(b.ang);
            const float x = A.hw[i], y = A.hh[i];
            v2 lv[4] = {mk(-x, -y), mk(-x, y), mk(x, y), mk(x, -y)};
            hw = 0.f; hh = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v2 r = rotcs(lv[k], c, sn);
                if (r.x > hw) hw = r.x;
                if (r.y > hh) hh = r.y;
            }
        } else {
            hw = hh = A.rad[i];
        }
        A.ax[i] = b.px; A.ay[i] = b.py; A.ahw[i] = hw; A.ahh[i] = hh;
    }
    if (stat) return b.m;
    for (int g = 0; g < A.ngens; ++g) {
        const auto& G = A.gens[g];   // fields read one by one (keeps G's address space)
        if (G.type == 0) {
            in.fx += G.gx * in.mass;
            in.fy += G.gy * in.mass;
        } else if (G.slot == i) {
            const float inv_m = 1.0f / in.mass;
            const v2 v = scale2(mk(b.m.x, b.m.y), inv_m);
            const v2 d = sub2(mk(b.px, b.py), mk(G.ax, G.ay));
            in.fx += (-G.k) * d.x - G.c * v.x;
            in.fy += (-G.k) * d.y - G.c * v.y;
        }
    }
    f3v m = b.m;
    m.x += in.fx * sub_dt;
    m.y += in.fy * sub_dt;
    m.z += in.tq * sub_dt;
    if constexpr (WARM) {
        if (A.warm > 0.0f) {
            // warm starting: the body's share of the matched manifolds' carried impulses
            const GlbCF ws = warm_sum(A, i);
            m.x += ws[0];
            m.y += ws[1];
            m.z += ws[2];
        }
    }
    return m;
}

// The kernel's argument block and the worlds' descriptors as the out-of-line
// parts of the solve read them: through the constant address space, so each
// field is a scalar load where it is used instead of a scalar register held
// (or spilled) through the whole step, and the pointers in them are known to
// be global memory.
typedef const __attribute__((address_space(4))) StepDev* StepArgs;
typedef const __attribute__((address_space(4))) WorldDev* WorldArgs;

// LDS of a world's solve from ChainShared::free_at on: the bodies, then the
// plan, and where the plan was the bodies' constants and the impulses.  In
// front of it: the items per ordering body and their offsets (n and n + 1).
struct ChainLds {
    ChainBodies C;
    LU32 rest, dcnt, doff;
    uint32_t n, rest_words, consts;
    LF2 acc;
    // the impulses of n contact points, and a spare one, beside the constants
    __device__ __forceinline__ bool holds(uint32_t n) const { return consts + 2u * (n + 1u) <= rest_words; }
    // beside: words that the plan keeps in front of the constants
    __device__ __forceinline__ ChainLds(LU32 smem, uint32_t free_at, uint32_t free_words, uint32_t n_, uint32_t beside) : n(n_)
    {
        dcnt = smem;
        doff = smem + n;
        LU32 lds = smem + free_at;
        C.m = (LF3)lds;
        C.px = (LF)(lds + 4u * (n + SPARE)); C.py = C.px + n; C.ang = C.py + n;
        const uint32_t fixed = (4u * (n + SPARE) + 3u * n + 1u) & ~1u;
        rest = lds + fixed + beside;
        rest_words = free_words - fixed - beside;
        C.mass = (LF)rest; C.inertia = C.mass + n; C.flags = (LU32)(C.inertia + n);
        consts = (3u * n + 1u) & ~1u;
        acc = (LF2)(rest + consts);
    }
};

// the gap before sub-step s's chain (s == sub_steps: after the last one), bodies
template <int T, bool WARM>
__device__ __attribute__((noinline)) void chain_bodies(StepArgs KS, LU32 smem, R2D_LDS ChainShared* shl, uint32_t s, uint32_t off)
{
    const StepDev& S = *(const StepDev*)uniform_ptr(KS);
    ChainShared& sh = *(ChainShared*)uniform_lds(shl);
    const WorldDev& D = *(const WorldDev*)(WorldArgs)(S.worlds + uniform(sh.w));
    const uint32_t sub_steps = uniform(sh.sub_steps);
    const float sub_dt = sh.dt / (float)sub_steps;
    const int n = D.nbodies;
    const ChainLds L(uniform_lds(smem), uniform(sh.free_at), uniform(sh.free_words), (uint32_t)n, uniform(sh.beside));
    const ChainBodies& C = L.C;
    const BodyArrays A = body_arrays(D);
    s = uniform(s);
    off = uniform(off);
    for (int i = (int)(threadIdx.x - off); i < n; i += (int)(T - off)) {
        BodyIn in{0u, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (s == 0u) {
            in = BodyIn{A.flags[i], A.mass[i], A.inertia[i], A.fx[i], A.fy[i], A.tq[i]};
            C.mass[i] = in.mass; C.inertia[i] = in.inertia; C.flags[i] = in.f;
        } else {
            in.f = C.flags[i]; in.mass = C.mass[i]; in.inertia = C.inertia[i];
        }
        const bool stat = (in.f & BF_STATIC) != 0;
        BodyState b{C.m[i], C.px[i], C.py[i], C.ang[i]};
        if (s > 0u && !stat) {
            body_move(b, in.mass, in.inertia, sub_dt);
            C.px[i] = b.px; C.py[i] = b.py; C.ang[i] = b.ang;
        }
        if (s == sub_steps) {
            body_done(D, A, i, stat, b);
        } else {
            const f3v m = body_push<WARM>(A, i, s + 1u == sub_steps, b, in, sub_dt);
            C.m[i] = m;
            if (minus_zero(m)) sh.fix = 1u;
        }
    }
}

// the gap, items: the joints' records, moved contact points, carried impulses
template <int T, bool WARM>
__device__ __attribute__((noinline)) void chain_items(StepArgs KS, LU32 smem, R2D_LDS ChainShared* shl, uint32_t s, uint32_t off)
{
    const StepDev& S = *(const StepDev*)uniform_ptr(KS);
    ChainShared& sh = *(ChainShared*)uniform_lds(shl);
    const uint32_t ibase = uniform(sh.ibase), mbeg = uniform(sh.mbeg), nj = uniform(sh.nj), M = uniform(sh.M),
                   base = uniform(sh.base), t = threadIdx.x - uniform(off), stride = (uint32_t)T - uniform(off);
    const WorldDev& D = *(const WorldDev*)(WorldArgs)(S.worlds + uniform(sh.w));
    const float sub_dt = sh.dt / (float)uniform(sh.sub_steps);
    const ChainLds L(uniform_lds(smem), uniform(sh.free_at), uniform(sh.free_words), (uint32_t)D.nbodies, uniform(sh.beside));
    u4v* recs = reinterpret_cast<u4v*>(S.recs + (size_t)ibase * 8);
    s = uniform(s);
    for (uint32_t j = t; j < nj; j += stride) joint_record(recs + (size_t)j * 4u, D.joints[j], D, L.C, s == 0u, [](uint32_t x) { return x; });
    const bool in_lds = L.holds(M + uniform(sh.pairs));
    GF2 accg = (GF2)(S.plan_ring + 2 * (size_t)ibase);
    if (sh.live)
        for (uint32_t q = t; q < M; q += stride) {
            const uint32_t p1 = S.it_k0[ibase + nj + q];
            point_tgs(S, D, recs, L.C, mbeg + q, base, nj + q, p1, sub_dt, [&](int p) {
                const uint32_t at = p ? p1 - nj : q;
                if (in_lds) L.acc[at] = f2v{0.f, 0.f};
                else accg[at] = f2v{0.f, 0.f};
            });
        }
    if constexpr (WARM) {
        if (!(D.warm > 0.0f)) return;
        const size_t cm = S.cap_m;
        for (uint32_t q = t; q < M; q += stride) {
            // warm starting: the carried impulse per sub-step joins the accumulators
            const uint32_t m = mbeg + q, valid = S.m_valid[m];
            if (!(valid & MV_WARM)) continue;
            for (uint32_t p = 0; p < 2u; ++p) {
                if (!(valid & (1u << p))) continue;
                const f2v add{S.m_pt[(MP_WARM_N * 2 + p) * cm + m], S.m_pt[(MP_WARM_T * 2 + p) * cm + m]};
                const uint32_t at = p ? S.it_k0[ibase + nj + q] - nj : q;
                if (in_lds) L.acc[at] = L.acc[at] + add;
                else accg[at] = accg[at] + add;
            }
        }
    }
}

// a world's program in memory
__device__ __forceinline__ ChainProgram chain_program(const StepDev& S, uint32_t ibase, uint32_t room, uint32_t nslots,
                                                      uint32_t reps, uint32_t nj, uint32_t M, uint32_t pairs)
{
    return ChainProgram{(GCU2)(S.prog_rows + (size_t)ibase * room), (GCU32)(S.prog_entries + (size_t)ibase * 2u * room),
                        (GCU2)(S.prog_slots + (size_t)ibase * room), (GCU4)(S.recs + (size_t)ibase * 8),
                        nslots, reps, nj, M + pairs, 2u * room * (nj + M), 0u};
}

// The plan, and meanwhile the bodies into LDS and the point records: wave 0
// plans a world run by one wave while the other waves build; a wider world is
// planned by all waves, then built by all.
//
// Where the plan, the constants and the impulses fit LDS side by side, the
// other waves also do the first sub-step's bodies and items, and wave 1 then
// runs its chain behind the planner, FOLLOW_ROWS rows at a time (a row takes
// the planner 0.46 us and the chain 0.28, so the first chain costs little more
// than the rows of its last part): returns whether it did.
constexpr uint32_t FOLLOW_ROWS = 24;
template <int T, bool WARM>
__device__ __attribute__((noinline)) bool chain_prepare(StepArgs KS, LU32 smem, R2D_LDS ChainShared* shl)
{
    const StepDev& S = *(const StepDev*)uniform_ptr(KS);
    ChainShared& sh = *(ChainShared*)uniform_lds(shl);
    const uint32_t w = uniform(sh.w), ibase = uniform(sh.ibase), mbeg = uniform(sh.mbeg), nj = uniform(sh.nj),
                   M = uniform(sh.M), base = uniform(sh.base);
    const WorldDev& D = *(const WorldDev*)(WorldArgs)(S.worlds + w);
    const uint32_t t = threadIdx.x, n = (uint32_t)D.nbodies, nit = nj + M, room = S.chain_room();
    const float sub_dt = sh.dt / (float)uniform(sh.sub_steps);
    const ChainLds L(uniform_lds(smem), uniform(sh.free_at), uniform(sh.free_words), n, 0u);
    const ChainBodies& C = L.C;
    u4v* recs = reinterpret_cast<u4v*>(S.recs + (size_t)ibase * 8);
    const uint32_t waves = fused_waves(nit, S.chain_iters, (uint32_t)T / 64u);
    const bool chain = nit > 0u && sh.iters > 0u;
    const bool plan_in_lds = nit <= PLAN_MAX_ITEMS && plan_lds_words(nit, waves) <= L.rest_words;
    const bool slow = S.chain_less != 0u && (waves > 1u || !plan_in_lds);
    const uint32_t kc = slow ? S.chain_less : S.chain_iters;
    Program G;
    G.rows = (GU2)(S.prog_rows + (size_t)ibase * room);
    G.entries = (GU32)(S.prog_entries + (size_t)ibase * 2u * room);
    G.slots = (GU2)(S.prog_slots + (size_t)ibase * room);
    PlanLds PL(L.rest, nit, waves);
    PlanGlb PG((GU4)(S.plan_items + 2 * (size_t)ibase), (GU4)(S.plan_ring + 2 * (size_t)ibase), nit, waves);
    const uint32_t* lists = S.lists + 2 * (size_t)ibase;
    // successors, and the items that wait for nothing in the first iteration
    auto fill = [&](auto& P) {
        for (uint32_t j = t; j < nit; j += T) {
            const int32_t r0 = S.it_r0[ibase + j], r1 = S.it_r1[ibase + j];
            const uint32_t k0 = S.it_k0[ibase + j], k1 = S.it_k1[ibase + j];
            const bool pair = j >= nj && (S.m_valid[mbeg + (j - nj)] & 3u) == 3u;
            auto next = [&](int32_t r, uint32_t k) {
                const uint32_t x = (uint32_t)r - base;
                return lists[L.doff[x] + (k + 1u == L.dcnt[x] ? 0u : k + 1u)] >> 1;
            };
            // one ordering body (or none: the item then only follows itself)
            const bool two = r0 >= 0 && r1 >= 0;
            const uint32_t s0 = r0 >= 0 ? next(r0, k0) : r1 >= 0 ? next(r1, k1) : j;
            const uint32_t s1 = two ? next(r1, k1) : nit | SINGLE;
            const uint32_t need = (r0 >= 0 && k0 > 0u ? 1u : 0u) + (r1 >= 0 && k1 > 0u ? 1u : 0u);
            const uint32_t sec = pair ? 1u + __hip_atomic_fetch_add(&sh.pairs, 1u, __ATOMIC_RELAXED,
                                                                    __HIP_MEMORY_SCOPE_WORKGROUP)
                                      : 0u;
            S.it_k0[ibase + j] = nit + sec - 1u;          // the second point's index; the ranks are not read again
            P.init(j, s0, s1, need * STATE_BODY + kc, sec);
            if (need == 0u)
                P.push(__hip_atomic_fetch_add(&sh.ready, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP),
                       P.pack(PlanEntry{j, sec, s0, s1}));
        }
        if (t == 0u) P.init(nit, nit, nit | SINGLE, 0u, 0u);   // the spare item: no iterations, never ready
    };
    if (plan_in_lds) fill(PL); else fill(PG);
    __syncthreads();
    const uint32_t ready = uniform(sh.ready);
    // the point that does nothing, after the others (an item slice has an item
    // to spare); by wave 1, whose chain may start without a barrier
    if (t - 64u < 4u) recs[(size_t)(nit + uniform(sh.pairs)) * 4u + (t - 64u)] = idle_word((int)(t - 64u));
    if (t == 64u) G.entries[2u * room * nit] = nit + uniform(sh.pairs);
    auto build = [&](uint32_t t0, uint32_t stride) {
        for (uint32_t i = t0; i < n; i += stride) {
            C.m[i] = f3v{D.mx[i], D.my[i], D.L[i]};
            C.px[i] = D.px[i]; C.py[i] = D.py[i]; C.ang[i] = D.ang[i];
        }
        for (uint32_t q = t0; q < M; q += stride) {
            const uint32_t f = point_build<WARM>(S, D, recs, mbeg + q, base, nj + q, S.it_k0[ibase + nj + q], sub_dt,
                                                 [](uint32_t x) { return x; });
            if (f & 1u) sh.live = 1u;
            if (f & 2u) sh.fix = 1u;
        }
    };
    const uint32_t nacc = M + uniform(sh.pairs);
    const uint32_t plan_words = (plan_lds_words(nit, 1u) + 1u) & ~1u;
    const bool follow = chain && waves == 1u && plan_in_lds && sh.iters == kc && plan_words < L.rest_words &&
                        L.consts + 2u * (nacc + 1u) <= L.rest_words - plan_words;
    uint32_t ns = 1u, entries = 0u;
    if (follow) {
        sh.beside = plan_words;   // the same from every thread
        if (t < 64u) {
            ns = plan_single<true>(PL, G, nit, nj, kc, ready, entries, &sh.progress);
        } else {
            constexpr uint32_t OTHERS = (uint32_t)T / 64u - 1u;
            LF2 acc = L.acc + plan_words / 2u;
            build(t - 64u, T - 64u);
            for (uint32_t q = t - 64u; q < nacc; q += T - 64u) acc[q] = f2v{0.f, 0.f};
            chain_bodies<T, WARM>(KS, smem, shl, 0u, 64u);
            waves_meet(&sh.met, OTHERS, 1u);
            if (nj || sh.live || (WARM && D.warm > 0.0f)) {
                chain_items<T, WARM>(KS, smem, shl, 0u, 64u);
                waves_meet(&sh.met, OTHERS, 2u);
            }
            if (t < 128u) {
                ChainProgram P = chain_program(S, ibase, room, 0u, 1u, nj, M, uniform(sh.pairs));
                const bool fix = (uniform(sh.fix) | uniform(sh.live)) != 0u;
                for (uint32_t run = 0u;;) {
                    const uint32_t p = uniform(__hip_atomic_load(&sh.progress, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                    const uint32_t have = p & ~PLANNED, rows = have > run ? have - run : 0u;   // (none of a failed plan)
                    asm volatile("" ::: "memory");   // the rows are read after their count
                    if (rows >= FOLLOW_ROWS || ((p & PLANNED) && rows != 0u)) {
                        P.nslots = rows;
                        chain_lds<false, WARM, false>(P, C.m, n, acc, fix, sub_dt);
                        P.rows += rows;
                        run += rows;
                    } else if (p & PLANNED) {
                        break;
                    } else {
                        __builtin_amdgcn_s_sleep(4);
                    }
                }
            }
        }
    } else if (chain && waves > 1u) {
        ns = plan_in_lds ? plan_multi(PL, G, nit, nj, kc, ready, waves, sh)
                         : plan_multi(PG, G, nit, nj, kc, ready, waves, sh);
        build(t, T);
    } else if (t < 64u) {
        if (chain)
            ns = plan_in_lds ? plan_single(PL, G, nit, nj, kc, ready, entries) : plan_single(PG, G, nit, nj, kc, ready, entries);
    } else {
        build(t - 64u, T - 64u);
    }
    if (t == 0) {
        sh.nslots = ns;
        sh.reps = sh.iters / kc;
        sh.slow = slow;
        if (waves == 1u) sh.entries = entries;
        sh.failed = ns == 0u;
        if (ns == 0u) S.w_status[w] = WS_STALL;   // corrupt ordering data: the world stops
    }
    __syncthreads();
    return follow;
}

// Between plan and first chain, where that has not run behind the planner: the
// program for the rest of the iterations, and the impulses at zero.
// A function of its own: in the planner's it costs every step 1.5 %.
template <int T>
__device__ __attribute__((noinline)) void chain_ready(StepArgs KS, LU32 smem, R2D_LDS ChainShared* shl)
{
    const StepDev& S = *(const StepDev*)uniform_ptr(KS);
    ChainShared& sh = *(ChainShared*)uniform_lds(shl);
    const uint32_t w = uniform(sh.w), ibase = uniform(sh.ibase), nj = uniform(sh.nj), M = uniform(sh.M), nit = nj + M,
                   t = threadIdx.x, nacc = M + uniform(sh.pairs);
    const WorldDev& D = *(const WorldDev*)(WorldArgs)(S.worlds + w);
    const ChainLds L(uniform_lds(smem), uniform(sh.free_at), uniform(sh.free_words), (uint32_t)D.nbodies, 0u);
    const GU4 ring = (GU4)(S.plan_ring + 2 * (size_t)ibase);
    if (S.chain_rest && !uniform(sh.slow) && nit > 0u && sh.iters > 0u) {
        const uint32_t room = S.chain_room(), waves = fused_waves(nit, S.chain_iters, (uint32_t)T / 64u);
        const Program G{(GU2)(S.prog_rows + (size_t)ibase * room), (GU32)(S.prog_entries + (size_t)ibase * 2u * room),
                        (GU2)(S.prog_slots + (size_t)ibase * room)};
        plan_rest(PlanMemory{L.rest, (GU4)(S.plan_items + 2 * (size_t)ibase), ring, G},
                  nit <= PLAN_MAX_ITEMS && plan_lds_words(nit, waves) <= L.rest_words, nit, nj, S.chain_iters, S.chain_rest,
                  waves, shl);
        if (t == 0 && sh.rest_slots == 0u) {
            sh.failed = 1u;
            S.w_status[w] = WS_STALL;   // corrupt ordering data: the world stops
        }
    }
    // accumulated impulses (normal, tangential) of the contact points, by
    // point index less the joints: in LDS after the constants when they fit
    if (L.holds(nacc)) {
        for (uint32_t q = t; q < nacc; q += T) L.acc[q] = f2v{0.f, 0.f};
    } else {
        GF2 accg = (GF2)ring;
        for (uint32_t q = t; q < nacc; q += T) accg[q] = f2v{0.f, 0.f};
    }
    __syncthreads();
}

// the impulses -> the step's manifold arrays (what r2d_get_manifolds reports)
template <int T>
__device__ __attribute__((noinline)) void chain_finish(StepArgs KS, LU32 smem, R2D_LDS ChainShared* shl)
{
    const StepDev& S = *(const StepDev*)uniform_ptr(KS);
    ChainShared& sh = *(ChainShared*)uniform_lds(shl);
    const uint32_t ibase = uniform(sh.ibase), mbeg = uniform(sh.mbeg), nj = uniform(sh.nj), M = uniform(sh.M);
    const WorldDev& D = *(const WorldDev*)(WorldArgs)(S.worlds + uniform(sh.w));
    const ChainLds L(uniform_lds(smem), uniform(sh.free_at), uniform(sh.free_words), (uint32_t)D.nbodies, uniform(sh.beside));
    const bool in_lds = L.holds(M + uniform(sh.pairs));
    GF2 accg = (GF2)(S.plan_ring + 2 * (size_t)ibase);
    const size_t cm = S.cap_m;
    for (uint32_t q = threadIdx.x; q < M; q += T) {
        const uint32_t m = mbeg + q, valid = S.m_valid[m];
        for (uint32_t p = 0; p < 2u; ++p) {
            if (!(valid & (1u << p))) continue;
            const uint32_t at = p ? S.it_k0[ibase + nj + q] - nj : q;
            const f2v v = in_lds ? (f2v)L.acc[at] : (f2v)accg[at];
            S.m_pt[(MP_ACC_PN * 2 + p) * cm + m] = v.x;
            S.m_pt[(MP_ACC_PT * 2 + p) * cm + m] = v.y;
        }
    }
}

// The solve of one world's step (described by sh; sub_steps > 0): S sub-steps
// of forces, integration, pre-step and K solver iterations (lib.zig:199-250),
// by a workgroup of T threads.  The K iterations run as a program of rows
// (r2d_chain.h); between the chains the bodies live in LDS.  Each part is a
// function of its own: inlined into the step kernel they pushed it over its
// register budget (80 spilled VGPRs, 490 spilled SGPRs, and machine code that
// the compiler's own verifier refused).
template <int T, bool WARM>
__device__ __forceinline__ void chain_world(StepArgs KS, LU32 smem, R2D_LDS ChainShared* shl)
{
    ChainShared& sh = *(ChainShared*)shl;
    const bool first = uniform(chain_prepare<T, WARM>(KS, smem, shl)) != 0u;
    if (sh.failed) return;
    if (!first) {   // else the first chain has run behind the planner
        chain_ready<T>(KS, smem, shl);
        if (sh.failed) return;
    }
    const StepDev& S = *(const StepDev*)KS;
    const WorldDev& D = *(const WorldDev*)(WorldArgs)(S.worlds + uniform(sh.w));
    const uint32_t sub_steps = uniform(sh.sub_steps), iters = uniform(sh.iters), nj = uniform(sh.nj);
    const bool any = nj + sh.M > 0u, items = nj || sh.live || (WARM && D.warm > 0.0f);
    for (uint32_t s = first ? 1u : 0u;; ++s) {
        chain_bodies<T, WARM>(KS, smem, shl, s, 0u);
        if (s == sub_steps) break;
        __syncthreads();
        if (!any) continue;
        if (items) {
            chain_items<T, WARM>(KS, smem, shl, s, 0u);
            __syncthreads();
        }
        if (iters == 0u) continue;
        const uint32_t M = uniform(sh.M), ibase = uniform(sh.ibase);
        const ChainLds L(smem, uniform(sh.free_at), uniform(sh.free_words), (uint32_t)D.nbodies, uniform(sh.beside));
        const bool in_lds = L.holds(M + uniform(sh.pairs));
        ChainProgram G = chain_program(S, ibase, S.chain_room(), uniform(sh.nslots), uniform(sh.reps), nj, M, uniform(sh.pairs));
        GF2 accg = (GF2)(S.plan_ring + 2 * (size_t)ibase);
        const float sub_dt = sh.dt / (float)sub_steps;
        const bool fix = (uniform(sh.fix) | uniform(sh.live)) != 0u;
        const bool several = fused_waves(nj + M, S.chain_iters, (uint32_t)T / 64u) > 1u;
#pragma clang loop unroll(disable)
        for (uint32_t left = S.chain_rest ? uniform(sh.rest_slots) : 0u;;) {
            if (several) {
                if (in_lds) chain_lds<true, WARM, false>(G, L.C.m, L.n, L.acc, fix, sub_dt);
                else chain_lds_accg<true, WARM, false>(G, L.C.m, L.n, accg, fix, sub_dt);
            } else if (threadIdx.x < 64u) {
                if (in_lds) chain_lds<false, WARM, false>(G, L.C.m, L.n, L.acc, fix, sub_dt);
                else chain_lds_accg<false, WARM, false>(G, L.C.m, L.n, accg, fix, sub_dt);
            }
            if (left == 0u) break;
            G = rest_program(G, S.chain_iters * (nj + M), left);
            left = 0u;
        }
        __syncthreads();
    }
    chain_finish<T>(KS, smem, shl);
}

// ------------------------------------------- the solve in separate launches
// For the worlds whose step is not one kernel: grid-wide kernels over all
// worlds' bodies and items around a workgroup per world that plans, then (once
// per sub-step) runs its program.  The momenta of the bodies that take part in
// items live under chain places (cmap) in g_mom between the launches, 16 bytes
// each, so that a chain takes them into LDS with plain wide copies; poses stay
// in the world's arrays.
typedef BodyPoses<GlbCF, GlbCU> GlobalPoses;
__device__ __forceinline__ GlobalPoses global_poses(const WorldDev& D)
{
    GlobalPoses P;
    P.px = (GlbCF)D.px; P.py = (GlbCF)D.py; P.ang = (GlbCF)D.ang; P.mass = (GlbCF)D.mass; P.inertia = (GlbCF)D.inertia;
    P.flags = (GlbCU)D.flags;
    return P;
}
// a world's momenta: one place more than its bodies
__device__ __forceinline__ GF3 world_momenta(const StepDev& S, const WorldDev& D, uint32_t w)
{
    return (GF3)(S.g_mom + D.body_base + w);
}

// a world's records in program order: entries, then joints, in blocks of four, each last one
// perhaps not full, then the idle point's (up to 8 places beyond 2 chain_room an item)
__device__ __forceinline__ GU4 world_records(const StepDev& S, uint32_t w, uint32_t ibase)
{
    return (GU4)(S.prog_recs + (size_t)ibase * 8u * S.chain_room() + (size_t)w * 32u);
}

__device__ __forceinline__ GU32 world_entries(const StepDev& S, uint32_t w, uint32_t ibase)
{
    return (GU32)(S.prog_entries + (size_t)ibase * 2u * S.chain_room() + (size_t)w * 8u);
}
// where the joints' records start
__device__ __forceinline__ uint32_t joint_entries(uint32_t entries) { return (entries + 3u) & ~3u; }

// the planning state of item j of a world, and where its second point is
__device__ __forceinline__ void plan_item(const StepDev& S, uint32_t ibase, uint32_t j, uint32_t nit, uint32_t second)
{
    const uint32_t it = ibase + j;
    const int32_t r0 = S.it_r0[it], r1 = S.it_r1[it];
    auto next = [&](int32_t r, uint32_t k, uint32_t& need) {
        const uint32_t o = S.deg_off[r], c = S.deg_off[r + 1] - o;
        need += k > 0u ? 1u : 0u;
        return (S.lists[o + (k + 1u == c ? 0u : k + 1u)] >> 1) - ibase;
    };
    uint32_t need = 0u, s0 = j, s1 = nit | SINGLE;   // no ordering body: the item only follows itself
    if (r0 >= 0) s0 = next(r0, S.it_k0[it], need);
    if (r1 >= 0) {
        const uint32_t q = next(r1, S.it_k1[it], need);
        if (r0 >= 0) s1 = q; else s0 = q;
    }
    S.it_k0[it] = nit + second - 1u;                 // the ranks are not read again
    S.plan_items[2 * (size_t)ibase + j] = make_uint4(s0, s1, need * STATE_BODY + S.chain_iters, second);
}

// per item: planning state, and the records of a manifold's points
template <bool WARM>
__global__ __launch_bounds__(256) void k_chain_build(StepDev S, float sub_dt)
{
    if (S.counters[C_OVERFLOW]) return;
    for (uint32_t q = grid_tid(); q < S.njoints; q += grid_stride()) {
        const uint32_t lo = joint_world(S, q), ibase = S.w_item_base[lo];
        plan_item(S, ibase, q - S.worlds[lo].joint_base, S.w_item_base[lo + 1] - ibase, 0u);
    }
    const uint32_t M = dev_count(&S.counters[C_MANIFOLDS], S.cap_m);
    for (uint32_t m = grid_tid(); m < M; m += grid_stride()) {
        const uint32_t w = S.bworld[S.m_ref[m]];
        const WorldDev& D = S.worlds[w];
        const uint32_t ibase = S.w_item_base[w], nit = S.w_item_base[w + 1] - ibase, base = D.body_base;
        const uint32_t j = (uint32_t)D.njoints + (m - S.w_man_begin[w]);
        const bool pair = (S.m_valid[m] & 3u) == 3u;
        const uint32_t rank = world_rank(S, pair, w, &WorldChain::pairs), second = pair ? 1u + rank : 0u;
        plan_item(S, ibase, j, nit, second);
        const uint32_t f = point_build<WARM>(S, D, reinterpret_cast<u4v*>(S.recs + (size_t)ibase * 8), m, base, j,
                                             nit + second - 1u, sub_dt, [&](uint32_t x) { return S.cmap[base + x]; });
        if (f) atomicOr(&S.w_chain[w].flags, f);
    }
}

// The program of each world, one workgroup each; with `rest`, in a launch after
// it, the one for the rest of the iterations: its rows and slots from
// chain_iters * nit on, its entries after the others.  (Planned through, every
// item waits for what it waited for at first.)
template <int T>
__global__ __launch_bounds__(T) void k_chain_plan(StepDev S, uint32_t iters, uint32_t lds_words, uint32_t rest)
{
    extern __shared__ __align__(16) uint32_t smem[];
    __shared__ ChainShared sh;
    if (S.counters[C_OVERFLOW]) return;
    const uint32_t w = S.w_order[blockIdx.x];
    const uint32_t ibase = S.w_item_base[w], nit = S.w_item_base[w + 1] - ibase, nj = (uint32_t)S.worlds[w].njoints;
    if (S.w_status[w] != 0 || nit == 0u) return;
    const uint32_t t = threadIdx.x, waves = chain_waves(nit, S.chain_iters, (uint32_t)T / 64u, CHAIN_WAVE_ROWS);
    const size_t rows = (size_t)ibase * S.chain_room() + (rest ? (size_t)S.chain_iters * nit : 0u);
    const uint32_t before = rest ? S.w_chain[w].entries : 0u;
    const bool in_lds = nit <= PLAN_MAX_ITEMS && plan_lds_words(nit, waves) <= lds_words;
    const bool slow = S.chain_less != 0u && !in_lds;
    if (rest && slow) return;   // its programs have no rest
    const uint32_t kc = rest ? rest : slow ? S.chain_less : S.chain_iters;
    if (t == 0) {
        sh.ready = sh.taken = 0u;
        sh.entries = before;
        sh.queued[0] = sh.queued[1] = sh.queued[2] = 0u;
    }
    __syncthreads();
    Program G;
    G.rows = (GU2)(S.prog_rows + rows);
    G.entries = world_entries(S, w, ibase);
    G.slots = (GU2)(S.prog_slots + rows);
    const GU4 items = (GU4)(S.plan_items + 2 * (size_t)ibase);
    PlanLds PL((LU32)smem, nit, waves);
    PlanGlb PG(items, (GU4)(S.plan_ring + 2 * (size_t)ibase), nit, waves);
    auto start = [&](auto& P, bool init) {
        for (uint32_t j = t; j < nit; j += T) {
            u4v v = items[j];
            v.z = (v.z & ~(STATE_BODY - 1u)) + kc;
            if (init || rest || slow) P.init(j, v.x, v.y, v.z, v.w);
            if (v.z < STATE_BODY)
                P.push(__hip_atomic_fetch_add(&sh.ready, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP),
                       P.pack(PlanEntry{j, v.w, v.x, v.y}));
        }
        if (t == 0u) P.init(nit, nit, nit | SINGLE, 0u, 0u);   // the spare item: no iterations, never ready
    };
    if (in_lds) start(PL, true); else start(PG, false);
    __syncthreads();
    const uint32_t ready = uniform(sh.ready);
    uint32_t ns = 0u, entries = before;
    if (waves > 1u)
        ns = in_lds ? plan_multi(PL, G, nit, nj, kc, ready, waves, sh) : plan_multi(PG, G, nit, nj, kc, ready, waves, sh);
    else if (t < 64u)
        ns = in_lds ? plan_single(PL, G, nit, nj, kc, ready, entries) : plan_single(PG, G, nit, nj, kc, ready, entries);
    if (t == 0) {
        if (rest) S.w_chain[w].rest_slots = ns; else S.w_chain[w].slots = ns;
        if (!rest) S.w_chain[w].reps = iters / kc;
        S.w_chain[w].entries = waves > 1u ? sh.entries : entries;
        if (ns == 0u) S.w_status[w] = WS_STALL;   // corrupt ordering data: the world stops
    }
}

// The gap before sub-step s's chain (s == sub_steps: after the last one):
// bodies; before the first one the points' records into program order, after
// the last one the impulses into the step's manifold arrays (what
// r2d_get_manifolds reports)
template <bool WARM>
__global__ __launch_bounds__(256) void k_chain_bodies(StepDev S, uint32_t s, uint32_t sub_steps, float sub_dt)
{
    if (S.counters[C_OVERFLOW]) return;
    for (uint32_t x = grid_tid(); x < S.nb; x += grid_stride()) {
        const uint32_t w = S.bworld[x];
        if (S.w_status[w] != 0) continue;
        const WorldDev& D = S.worlds[w];
        const BodyArrays A = body_arrays(D);
        const int i = (int)(x - D.body_base);
        const uint32_t c = S.cmap[x];
        const bool touched = c != UNTOUCHED;
        const GF3 mom = world_momenta(S, D, w) + (touched ? c : 0u);
        BodyIn in{A.flags[i], A.mass[i], A.inertia[i], 0.f, 0.f, 0.f};
        BodyState b;
        if (s > 0u && touched) b.m = *mom; else b.m = f3v{D.mx[i], D.my[i], D.L[i]};
        b.px = A.px[i]; b.py = A.py[i]; b.ang = A.ang[i];
        const bool stat = (in.f & BF_STATIC) != 0;
        if (s == 0u) { in.fx = A.fx[i]; in.fy = A.fy[i]; in.tq = A.tq[i]; }
        else if (!stat) {
            body_move(b, in.mass, in.inertia, sub_dt);
            if (s < sub_steps) { A.px[i] = b.px; A.py[i] = b.py; A.ang[i] = b.ang; }
        }
        if (s == sub_steps) { body_done(D, A, i, stat, b); continue; }
        const f3v m = body_push<WARM>(A, i, s + 1u == sub_steps, b, in, sub_dt);
        if (touched) {
            *mom = m;
            if (minus_zero(m)) atomicOr(&S.w_chain[w].flags, 2u);
        }
        else { D.mx[i] = m.x; D.my[i] = m.y; D.L[i] = m.z; }
    }
    if (s == 0u) {
        // each world's entries over gridDim / worlds workgroups
        const uint32_t parts = gridDim.x > S.nworlds ? gridDim.x / S.nworlds : 1u;
        for (uint32_t b = blockIdx.x; b < parts * S.nworlds; b += gridDim.x) {
            const uint32_t w = b % S.nworlds, ibase = S.w_item_base[w], nj = (uint32_t)S.worlds[w].njoints;
            if (S.w_status[w] != 0 || S.w_item_base[w + 1] == ibase) continue;
            const GU32 entries = world_entries(S, w, ibase);
            const GU4 to = world_records(S, w, ibase);
            const uint32_t n = S.w_chain[w].entries;
            if (b < S.nworlds && threadIdx.x < 4u) {
                const uint32_t idle = joint_entries(n) + nj;
                to[entry_at(idle) + threadIdx.x * ENTRY_WORD] = idle_word((int)threadIdx.x);
                if (threadIdx.x == 0u) entries[idle] = S.w_item_base[w + 1] - ibase + S.w_chain[w].pairs;
            }
            for (uint32_t e = (b / S.nworlds) * blockDim.x + threadIdx.x; e < n; e += parts * blockDim.x) {
                const uint32_t p = entries[e];
                if (p >= nj) entry_copy(to, e, (GCU4)(S.recs + (size_t)ibase * 8), p);
            }
        }
    }
    if (s != sub_steps) return;
    if (grid_tid() == 0u) S.counters[C_STEPS] += 1u;   // the step is done
    const size_t cm = S.cap_m;
    const uint32_t M = dev_count(&S.counters[C_MANIFOLDS], S.cap_m);
    for (uint32_t m = grid_tid(); m < M; m += grid_stride()) {
        const uint32_t w = S.bworld[S.m_ref[m]];
        if (S.w_status[w] != 0) continue;
        const uint32_t ibase = S.w_item_base[w], q = m - S.w_man_begin[w], nj = (uint32_t)S.worlds[w].njoints;
        const GF2 acc = (GF2)(S.plan_ring + 2 * (size_t)ibase);
        const uint32_t valid = S.m_valid[m];
        for (uint32_t p = 0; p < 2u; ++p) {
            if (!(valid & (1u << p))) continue;
            const f2v v = acc[p ? S.it_k0[ibase + nj + q] - nj : q];
            S.m_pt[(MP_ACC_PN * 2 + p) * cm + m] = v.x;
            S.m_pt[(MP_ACC_PT * 2 + p) * cm + m] = v.y;
        }
    }
}

// Sub-step s's joint records, moved contact points and carried impulses, and
// its iterations, one workgroup per world; REST, in a launch after it, only
// the iterations that end the sub-step (told apart at run time they cost those
// without a rest 0.5 us of 30.6 a launch, coloured pile of 4,096 bodies).  Momenta in LDS for worlds of
// at most lds_nmax bodies whose places fit it, and beside them the impulses
// when they fit too; otherwise they stay in global memory.
template <int T, bool WARM, bool REST>
__global__ __launch_bounds__(T) void k_chain_run(StepDev S, uint32_t s, uint32_t iters, float sub_dt, uint32_t lds_words,
                                                 uint32_t lds_nmax)
{
    extern __shared__ __align__(16) uint32_t smem[];
    if (S.counters[C_OVERFLOW]) return;
    const uint32_t w = S.w_order[blockIdx.x];
    const uint32_t ibase = S.w_item_base[w], nit = S.w_item_base[w + 1] - ibase;
    if (S.w_status[w] != 0 || nit == 0u) return;
    const WorldDev& D = S.worlds[w];
    const WorldChain W = S.w_chain[w];
    if (REST && W.rest_slots == 0u) return;
    const uint32_t t = threadIdx.x, nj = (uint32_t)D.njoints, M = nit - nj, mbeg = S.w_man_begin[w], base = D.body_base;
    const uint32_t nc = W.bodies, nacc = M + W.pairs, mwords = 4u * (nc + SPARE);
    const bool m_lds = (uint32_t)D.nbodies <= lds_nmax && mwords <= lds_words;
    const bool a_lds = m_lds && mwords + 2u * (nacc + 1u) <= lds_words;
    const LF3 m = (LF3)(LU32)smem;
    const LF2 acc = (LF2)((LU32)smem + mwords);
    const GF3 mom = world_momenta(S, D, w);
    const GF2 accg = (GF2)(S.plan_ring + 2 * (size_t)ibase);
    u4v* recs = reinterpret_cast<u4v*>(S.recs + (size_t)ibase * 8);
    if (m_lds)
        for (uint32_t c = t; c < nc; c += T) m[c] = mom[c];
    if (s == 0u && !REST)
        for (uint32_t q = t; q < nacc; q += T) {
            if (a_lds) acc[q] = f2v{0.f, 0.f}; else accg[q] = f2v{0.f, 0.f};
        }
    else if (a_lds)
        for (uint32_t q = t; q < nacc; q += T) acc[q] = accg[q];
    const GU4 prog = world_records(S, w, ibase);
    const GCU32 entries = (GCU32)world_entries(S, w, ibase);
    const uint32_t jbase = joint_entries(W.entries);
    const GlobalPoses C = global_poses(D);
    for (uint32_t j = t; j < nj && iters > 0u && !REST; j += T) {
        u4v q[4];
        joint_record(q, D.joints[j], D, C, s == 0u, [&](uint32_t x) { return S.cmap[base + x]; });
        const GU4 to = prog + entry_at(jbase + j);
        for (int p = 0; p < 4; ++p) to[p * ENTRY_WORD] = q[p];
    }
    __syncthreads();
    if ((W.flags & 1u) && !REST) {
        for (uint32_t q = t; q < M; q += T) {
            const uint32_t p1 = S.it_k0[ibase + nj + q];
            point_tgs(S, D, recs, C, mbeg + q, base, nj + q, p1, sub_dt, [&](int p) {
                const uint32_t at = p ? p1 - nj : q;
                if (a_lds) acc[at] = f2v{0.f, 0.f}; else accg[at] = f2v{0.f, 0.f};
            });
        }
        __syncthreads();
        for (uint32_t e = t; e < W.entries && iters > 0u; e += T) {
            const uint32_t p = entries[e];
            if (p >= nj) entry_copy(prog, e, (GCU4)(S.recs + (size_t)ibase * 8), p);
        }
    }
    if constexpr (WARM) {
        if (D.warm > 0.0f && !REST) {
            const size_t cm = S.cap_m;
            for (uint32_t q = t; q < M; q += T) {
                // warm starting: the carried impulse per sub-step joins the accumulators
                const uint32_t mi = mbeg + q, valid = S.m_valid[mi];
                if (!(valid & MV_WARM)) continue;
                for (uint32_t p = 0; p < 2u; ++p) {
                    if (!(valid & (1u << p))) continue;
                    const f2v add{S.m_pt[(MP_WARM_N * 2 + p) * cm + mi], S.m_pt[(MP_WARM_T * 2 + p) * cm + mi]};
                    const uint32_t at = p ? S.it_k0[ibase + nj + q] - nj : q;
                    if (a_lds) acc[at] = acc[at] + add; else accg[at] = accg[at] + add;
                }
            }
        }
    }
    __syncthreads();
    if (iters > 0u) {
        const size_t rows = (size_t)ibase * S.chain_room() + (REST ? (size_t)S.chain_iters * nit : 0u);
        const ChainProgram G{(GCU2)(S.prog_rows + rows), entries, (GCU2)(S.prog_slots + rows), (GCU4)prog,
                             REST ? W.rest_slots : W.slots, REST ? 1u : W.reps, nj, nacc, jbase + nj, jbase};
        const bool fix = W.flags != 0u;
        if (chain_waves(nit, S.chain_iters, (uint32_t)T / 64u, CHAIN_WAVE_ROWS) > 1u) {
            if (a_lds) chain_lds<true, WARM, true>(G, m, nc, acc, fix, sub_dt);
            else if (m_lds) chain_lds_accg<true, WARM, true>(G, m, nc, accg, fix, sub_dt);
            else chain_glb<true, WARM, true>(G, mom, nc, accg, fix, sub_dt);
        } else if (t < 64u) {
            if (a_lds) chain_lds<false, WARM, true>(G, m, nc, acc, fix, sub_dt);
            else if (m_lds) chain_lds_accg<false, WARM, true>(G, m, nc, accg, fix, sub_dt);
            else chain_glb<false, WARM, true>(G, mom, nc, accg, fix, sub_dt);
        }
        __syncthreads();
    }
    if (m_lds)
        for (uint32_t c = t; c < nc; c += T) mom[c] = m[c];
    if (a_lds)
        for (uint32_t q = t; q < nacc; q += T) accg[q] = acc[q];
}

// ------------------------------------------- the other parts of a fused step
// Like the solve, each a function of its own that reads the argument block and
// the world's descriptor through the constant address space: inlined together
// they held 269 scalar registers' worth in spills and, at four workgroups a CU,
// 80 vector registers.
struct FusedShared {
    uint32_t w, lds_words, err, slot;
    uint32_t E, R, M;
    WorldScratch X;
    uint32_t sm[16];
};

template <int T>
struct FusedView {
    const StepDev& S;
    const WorldDev& D;
    uint32_t &err, *s_sm;
    uint32_t w, n, tb, base, nj, t, lds_words, E, R, M;
    WorldScratch X;
    FusedLds L;
    PairCache P;
    // the entries' buckets and the bucket members are read in serial loops: in
    // LDS after the pair cache when they fit (E is about 1.5 n for bodies up to
    // a cell wide)
    uint32_t *ent_body, *ecnt, *ent_bkt, *items, *sorted;   // ecnt: raw candidates per entry -> offsets
    uint4* cand;
    uint32_t* cflag;   // collides per candidate -> manifold offsets
    __device__ __forceinline__ FusedView(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl)
        : S(*(const StepDev*)uniform_ptr(KS)),
          D(*(const WorldDev*)(WorldArgs)(((const StepDev*)uniform_ptr(KS))->worlds + uniform(((FusedShared*)fsl)->w))),
          err(((FusedShared*)uniform_lds(fsl))->err), s_sm(((FusedShared*)uniform_lds(fsl))->sm)
    {
        const FusedShared& fs = *(FusedShared*)uniform_lds(fsl);
        w = uniform(fs.w);
        lds_words = uniform(fs.lds_words);
        E = uniform(fs.E); R = uniform(fs.R); M = uniform(fs.M);
        X.e0 = uniform(fs.X.e0); X.r0 = uniform(fs.X.r0); X.m0 = uniform(fs.X.m0); X.i0 = uniform(fs.X.i0);
        n = (uint32_t)D.nbodies; tb = D.table; base = D.body_base; nj = (uint32_t)D.njoints;
        t = threadIdx.x;
        L = fused_carve((uint32_t*)uniform_lds(smem), n, tb);
        P = pair_cache(L.pairs, n);
        ent_body = S.ent_body + X.e0;
        ecnt = S.ent_cnt + X.e0;
        const bool e_lds = 3 * (size_t)E <= (size_t)(lds_words - fused_front_words(n, tb) - PAIR_CACHE_WORDS * n);
        uint32_t* e_free = L.pairs + PAIR_CACHE_WORDS * n;
        ent_bkt = e_lds ? e_free : S.ent_bkt + X.e0;
        items = e_lds ? e_free + E : S.bkt_items + X.e0;
        sorted = e_lds ? e_free + 2 * E : S.bkt_sorted + X.e0;
        cand = S.cand + X.r0;
        cflag = S.cand_flag + X.r0;
    }
};

// broadphase, per body (k_prep); returns the cell entries
template <int T>
__device__ __attribute__((noinline)) uint32_t fused_cells(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl)
{
    const FusedView<T> V(KS, smem, fsl);
    const StepDev& S = V.S;
    const WorldDev& D = V.D;
    const uint32_t n = V.n, base = V.base, t = V.t;
    const FusedLds& L = V.L;
    const PairCache& P = V.P;
    uint32_t* const s_sm = V.s_sm;
    // stale AABBs and flags in LDS for the pair filters below
    for (uint32_t i = t; i < n; i += T) {
        const Prep o = prep_body(D, i);
        P.ax[i] = D.ax[i]; P.ay[i] = D.ay[i]; P.ahw[i] = D.ahw[i]; P.ahh[i] = D.ahh[i];
        P.flags[i] = D.flags[i];
        L.cc[i] = o.c;
        L.cs[i] = o.s;
        S.sflag[base + i] = o.res;
        if (o.err) atomicOr(&V.err, o.err == WS_NONFINITE ? 2u : 1u);
        if (!o.err && o.ncell) { S.cx0[base + i] = o.x0; S.cy0[base + i] = o.y0; S.cnx[base + i] = o.nx; }
        L.coff[i] = o.ncell;
    }
    __syncthreads();
    return group_scan(L.coff, n, s_sm);
}

// cell entries and buckets (k_entries .. k_bucket_rank)
template <int T>
__device__ __attribute__((noinline)) void fused_buckets(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl)
{
    const FusedView<T> V(KS, smem, fsl);
    const StepDev& S = V.S;
    const uint32_t n = V.n, tb = V.tb, base = V.base, t = V.t, E = V.E;
    const FusedLds& L = V.L;
    uint32_t *const ent_body = V.ent_body, *const ent_bkt = V.ent_bkt, *const items = V.items, *const sorted = V.sorted, *const s_sm = V.s_sm;
    for (uint32_t b = t; b <= tb; b += T) {
        L.boff[b] = 0u;
        if (b < tb) L.bfill[b] = 0u;
    }
    __syncthreads();
    // cell entries and bucket occupancy (k_entries)
    for (uint32_t e = t; e < E; e += T) {
        uint32_t i = upper_idx(L.coff, n, e);
        uint32_t k = e - L.coff[i];
        uint32_t nx = S.cnx[base + i];
        int64_t yi = S.cy0[base + i] + (int64_t)(k / nx);
        int64_t xi = S.cx0[base + i] + (int64_t)(k % nx);
        uint32_t b = (uint32_t)cell_hash((uint64_t)tb, xi, yi);
        ent_body[e] = i;
        ent_bkt[e] = b;
        atomicAdd(&L.boff[b], 1u);
    }
    __syncthreads();
    group_scan(L.boff, tb, s_sm);
    // bucket members (k_bucket_fill), then in descending slot with a
    // body's repeats adjacent (k_bucket_rank)
    for (uint32_t e = t; e < E; e += T) {
        uint32_t b = ent_bkt[e];
        uint32_t pos = atomicAdd(&L.bfill[b], 1u);
        items[L.boff[b] + pos] = ent_body[e];
    }
    __syncthreads();
    for (uint32_t e = t; e < E; e += T) {
        uint32_t a = ent_body[e], b = ent_bkt[e];
        uint32_t o = L.boff[b], c = L.boff[b + 1] - o;
        uint32_t greater, same;
        bucket_rank_of(items + o, c, a, greater, same);
        uint32_t dup = 0;
        if (same > 1)
            for (uint32_t x = L.coff[a]; x < e; ++x) dup += ent_bkt[x] == b;
        sorted[o + greater + dup] = a;
    }
    __syncthreads();
}

template <int T>
__device__ __attribute__((noinline)) uint32_t fused_count(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl)
{
    const FusedView<T> V(KS, smem, fsl);
    const uint32_t t = V.t, E = V.E;
    const FusedLds& L = V.L;
    const PairCache& P = V.P;
    uint32_t *const ent_body = V.ent_body, *const ecnt = V.ecnt, *const ent_bkt = V.ent_bkt, *const items = V.items, *const sorted = V.sorted, *const s_sm = V.s_sm;
    // raw candidates per entry: distinct bucket members above the entry's
    // body (k_ent_cnt) that pass the both-static and AABB filters; the
    // passing members among the first 32 as a mask (in `items`, whose
    // bucket lists are no longer read)
    for (uint32_t e = t; e < E; e += T) {
        const uint32_t a = ent_body[e], b = ent_bkt[e];
        const uint32_t o = L.boff[b], c = L.boff[b + 1] - o;
        uint32_t q, mask;
        entry_candidates(P, a, sorted + o, c, q, mask);
        ecnt[e] = q;
        items[e] = mask;
    }
    __syncthreads();
    return group_scan(ecnt, E, s_sm);
}

template <int T>
__device__ __attribute__((noinline)) void fused_emit(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl)
{
    const FusedView<T> V(KS, smem, fsl);
    const uint32_t t = V.t, E = V.E;
    const FusedLds& L = V.L;
    const PairCache& P = V.P;
    uint32_t *const ent_body = V.ent_body, *const ecnt = V.ecnt, *const ent_bkt = V.ent_bkt, *const items = V.items, *const sorted = V.sorted;
    uint4* const cand = V.cand;
    // raw candidates in query order (k_cand_emit)
    for (uint32_t e = t; e < E; e += T) {
        uint32_t a = ent_body[e], b = ent_bkt[e];
        uint32_t o = L.boff[b];
        uint32_t ro = ecnt[e], c = ecnt[e + 1] - ro;
        uint32_t k = e - L.coff[a];
        uint32_t q = 0;
        for (uint32_t mask = items[e]; mask; mask &= mask - 1u, ++q)
            cand[ro + q] = make_uint4(a, sorted[o + (uint32_t)__builtin_ctz(mask)], k, 0u);
        for (uint32_t j = 32; q < c; ++j) {
            const uint32_t bj = sorted[o + j];
            if (bj == sorted[o + j - 1] || !pair_passes(P, a, bj)) continue;
            cand[ro + q] = make_uint4(a, bj, k, 0u);
            ++q;
        }
    }
    __syncthreads();
}

template <int T>
__device__ __attribute__((noinline)) uint32_t fused_narrow(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl)
{
    const FusedView<T> V(KS, smem, fsl);
    const WorldDev& D = V.D;
    const uint32_t t = V.t, R = V.R;
    const FusedLds& L = V.L;
    uint32_t *const ent_bkt = V.ent_bkt, *const cflag = V.cflag, *const s_sm = V.s_sm;
    uint4* const cand = V.cand;
    // ---- narrowphase (k_narrow): the collision overwrites its candidate
    // (partner, face id | ref-is-a, normal)
    for (uint32_t q = t; q < R; q += T) {
        const uint4 cq = cand[q];
        const uint32_t a = cq.x, b = cq.y;
        uint32_t info = 0;
        float nx = 0.f, ny = 0.f;
        bool hit = narrow_pair_call(D, a, b, cq.z, ent_bkt + L.coff[a], ent_bkt + L.coff[b],
                                     L.coff[b + 1] - L.coff[b], L.cc[a], L.cs[a], L.cc[b], L.cs[b], info, nx, ny);
        cflag[q] = hit ? 1u : 0u;
        if (hit) cand[q] = make_uint4(a | (b << 16), info, __float_as_uint(nx), __float_as_uint(ny));
    }
    __syncthreads();
    return group_scan(cflag, R, s_sm);
}

template <int T>
__device__ __attribute__((noinline)) void fused_contacts(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl)
{
    const FusedView<T> V(KS, smem, fsl);
    const StepDev& S = V.S;
    const WorldDev& D = V.D;
    const uint32_t n = V.n, base = V.base, nj = V.nj, t = V.t, R = V.R;
    const FusedLds& L = V.L;
    const WorldScratch& X = V.X;
    uint32_t* const cflag = V.cflag;
    uint4* const cand = V.cand;
    // contact points (k_man_build), manifolds in discovery order
    for (uint32_t q = t; q < R; q += T) {
        const uint32_t mi = cflag[q];
        if (cflag[q + 1] == mi) continue;
        const uint4 x = cand[q];
        const uint32_t a = x.x & 0xffffu, b = x.x >> 16;
        man_build_one(S, D, D, X.m0 + mi, base, a, b, x.y, mk(__uint_as_float(x.z), __uint_as_float(x.w)), L.cc[a],
                      L.cs[a], L.cc[b], L.cs[b]);
    }
    // ---- schedule: distance / offset joints make both bodies ordering (k_joint_mark)
    for (uint32_t j = t; j < nj; j += T) {
        const Joint& J = D.joints[j];
        if (J.type <= 1) {
            if (J.s1 >= 0) atomicOr(&S.sflag[base + J.s1], SF_RESOURCE);
            if (J.s2 >= 0) atomicOr(&S.sflag[base + J.s2], SF_RESOURCE);
        }
    }
    for (uint32_t i = t; i < n; i += T) { L.dcnt[i] = 0u; L.dfill[i] = 0u; }
    __syncthreads();
}

template <int T, bool WARM>
__device__ __attribute__((noinline)) void fused_schedule(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl, uint32_t sub_steps)
{
    const FusedView<T> V(KS, smem, fsl);
    const StepDev& S = V.S;
    const WorldDev& D = V.D;
    const uint32_t n = V.n, base = V.base, nj = V.nj, t = V.t, M = V.M;
    const FusedLds& L = V.L;
    const WorldScratch& X = V.X;
    uint32_t* const s_sm = V.s_sm;
    const uint32_t nit = nj + M;
    // items: joints, then manifolds, with their ordering bodies
    for (uint32_t j = t; j < nit; j += T) {
        int32_t r0 = -1, r1 = -1;
        if (j < nj) {
            const Joint& J = D.joints[j];
            r0 = J.s1 >= 0 ? (int32_t)(base + J.s1) : -1;
            if (J.type <= 1 && J.s2 >= 0 && J.s2 != J.s1) r1 = (int32_t)(base + J.s2);
        } else {
            const uint32_t m = X.m0 + (j - nj);
            const uint32_t ref = S.m_ref[m], inc = S.m_inc[m];
            r0 = (S.sflag[ref] & SF_RESOURCE) ? (int32_t)ref : -1;
            r1 = (S.sflag[inc] & SF_RESOURCE) ? (int32_t)inc : -1;
        }
        S.it_r0[X.i0 + j] = r0;
        S.it_r1[X.i0 + j] = r1;
        if (r0 >= 0) atomicAdd(&L.dcnt[r0 - (int32_t)base], 1u);
        if (r1 >= 0) atomicAdd(&L.dcnt[r1 - (int32_t)base], 1u);
    }
    __syncthreads();
    for (uint32_t i = t; i < n; i += T) L.doff[i] = L.dcnt[i];
    __syncthreads();
    group_scan(L.doff, n, s_sm);
    // per-body item lists (k_list_fill), ranks in item order (k_list_rank).
    // When the lists fit LDS behind the items per body (the cell, trig,
    // bucket and pair arrays are dead after the contacts), they are filled there in any
    // order and each entry then finds its rank by counting the smaller
    // entries of its body's list (independent LDS reads) and goes to that
    // place of the global lists; else they are filled in global memory and
    // sorted per body.
    const uint32_t lds_words = V.lds_words;
    uint32_t* const lists = S.lists + 2 * (size_t)X.i0;
    uint32_t* const ul = L.coff;
    const bool lds_lists = L.doff[n] <= lds_words - (3u * n + 1u);
    uint32_t* const fill = lds_lists ? ul : lists;
    for (uint32_t j = t; j < nit; j += T) {
        const int32_t r0 = S.it_r0[X.i0 + j], r1 = S.it_r1[X.i0 + j];
        if (r0 >= 0) {
            const uint32_t x = (uint32_t)r0 - base;
            fill[L.doff[x] + atomicAdd(&L.dfill[x], 1u)] = j * 2u;
        }
        if (r1 >= 0) {
            const uint32_t x = (uint32_t)r1 - base;
            fill[L.doff[x] + atomicAdd(&L.dfill[x], 1u)] = j * 2u + 1u;
        }
    }
    __syncthreads();
    if (lds_lists) {
        for (uint32_t j = t; j < nit; j += T) {
#pragma unroll
            for (uint32_t side = 0; side < 2; ++side) {
                const int32_t r = side ? S.it_r1[X.i0 + j] : S.it_r0[X.i0 + j];
                if (r < 0) continue;
                const uint32_t x = (uint32_t)r - base, o = L.doff[x];
                const uint32_t v = j * 2u + side;
                const uint32_t rank = count_below(ul + o, L.dcnt[x], v);
                lists[o + rank] = v;
                if (side) S.it_k1[X.i0 + j] = rank; else S.it_k0[X.i0 + j] = rank;
            }
        }
    } else {
        for (uint32_t x = t; x < n; x += T) {
            uint32_t* l = lists + L.doff[x];
            const uint32_t c = L.dcnt[x];
            for (uint32_t i = 1; i < c; ++i) {
                uint32_t v = l[i];
                uint32_t j = i;
                while (j > 0 && l[j - 1] > v) { l[j] = l[j - 1]; --j; }
                l[j] = v;
            }
            for (uint32_t p = 0; p < c; ++p) {
                uint32_t v = l[p];
                if (v & 1u) S.it_k1[X.i0 + (v >> 1)] = p; else S.it_k0[X.i0 + (v >> 1)] = p;
            }
        }
    }
    __syncthreads();
    if (WARM && D.warm > 0.0f) {
        // warm starting: match last step's manifolds, then each body's carried impulse
        for (uint32_t q = t; q < M; q += T) warm_match(S, D, X.m0 + q, base, sub_steps);
        __syncthreads();
        for (uint32_t x = t; x < n; x += T) warm_body_sum(S, D, lists + L.doff[x], L.dcnt[x], x, 0u, nj, X.m0);
        __syncthreads();
    }
}

// Room for the step's entries (stage 0), raw candidates (1) and manifolds and
// items (2; the counts not known yet are 0): a slice that is too small is replaced, or the world stops before its state changes.
// The counts are then what the parts read.
template <int T>
__device__ __attribute__((noinline)) bool fused_room(StepArgs KS, R2D_LDS FusedShared* fsl, uint32_t E, uint32_t R, uint32_t M,
                                                     uint32_t stage)
{
    const StepDev& S = *(const StepDev*)uniform_ptr(KS);
    FusedShared& fs = *(FusedShared*)uniform_lds(fsl);
    E = uniform(E); R = uniform(R); M = uniform(M); stage = uniform(stage);
    const uint32_t w = uniform(fs.w), nit = (uint32_t)S.worlds[w].njoints + M;
    WorldScratch X = fs.X;
    const bool fits = stage == 0u ? E <= X.ecap : stage == 1u ? R <= X.rcap : M <= X.mcap && nit <= X.icap;
    bool ok = true;
    if (!uniform(fits)) {
        if (stage == 0u) ok = fused_grow(S, w, X, 0, E, fs.slot);
        else if (stage == 1u) ok = fused_grow(S, w, X, 1, R, fs.slot);
        else ok = (M <= X.mcap || fused_grow(S, w, X, 2, M, fs.slot)) && (nit <= X.icap || fused_grow(S, w, X, 3, nit, fs.slot));
        if (!ok) fused_overflow(S, w, E, R, M, stage == 2u ? nit : 0u);
    }
    __syncthreads();   // every thread has read the slices
    if (threadIdx.x == 0) {
        fs.E = E; fs.R = R; fs.M = M;
        fs.X = X;
    }
    __syncthreads();
    return ok;
}

// the end of a step: warm-start tables, counts
template <int T, bool WARM>
__device__ __attribute__((noinline)) void fused_done(StepArgs KS, LU32 smem, R2D_LDS FusedShared* fsl, uint32_t step)
{
    const FusedView<T> V(KS, smem, fsl);
    const StepDev& S = V.S;
    const WorldDev& D = V.D;
    const uint32_t n = V.n, t = V.t, M = V.M, w = V.w, m0 = V.X.m0, nit = V.nj + M;
    step = uniform(step);
    if (WARM && D.warm > 0.0f) {
        // warm starting: this step's manifolds become the next step's tables
        for (uint32_t x = t; x < n; x += T) D.wcnt[x] = 0u;
        __syncthreads();
        for (uint32_t q = t; q < M; q += T) warm_save(S, D, m0 + q, m0, m0 + M, V.base);
        __syncthreads();
    }
    if (t == 0) {
        uint32_t* cnt = S.w_cnt + 8 * (size_t)w;
        cnt[0] = V.E; cnt[1] = V.R; cnt[2] = M; cnt[3] = nit;
        unsigned long long* sums = reinterpret_cast<unsigned long long*>(S.counters + C_SUMS);
        atomicAdd(&sums[0], (unsigned long long)n);
        atomicAdd(&sums[1], (unsigned long long)V.E);
        atomicAdd(&sums[2], (unsigned long long)V.R);
        atomicAdd(&sums[3], (unsigned long long)M);
        atomicAdd(&sums[4], (unsigned long long)nit);
        S.w_man_begin[w] = m0;
        S.w_man_end[w] = m0 + M;
        S.w_done[w] = step + 1;
        if (S.w_tstamp && step < S.tcap) S.w_tstamp[(size_t)w * (S.tcap + 1) + step + 1] = wall_clock64();
    }
}

// One workgroup per world (S.w_order), up to nsteps steps per world counted
// in S.w_done, so a relaunch after an overflow resumes each world where it
// stopped.  lds_words: the launch's dynamic LDS.
template <int MAXT, int WAVES, bool WARM = false>
__global__ __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(WAVES)))
void k_fused(StepDev /* read from the argument segment, which it starts */, float dt, uint32_t sub_steps, uint32_t iters, uint32_t nsteps, uint32_t lds_words)
{
    extern __shared__ __align__(16) uint32_t smem[];
    __shared__ FusedShared s_fs;
    __shared__ ChainShared s_chain;
    const uint32_t t = threadIdx.x;
    constexpr int T = MAXT;
    const StepArgs KS = (StepArgs)__builtin_amdgcn_kernarg_segment_ptr();
    const LU32 lds = (LU32)smem;
    R2D_LDS FusedShared* const fs = (R2D_LDS FusedShared*)&s_fs;
    // the argument block where it is read (nothing of it is held across a part)
    auto args = [&]() -> const StepDev& {
        StepArgs p = KS;
        asm volatile("" : "+s"(p));
        return *(const StepDev*)p;
    };
    const uint32_t w = args().w_order[blockIdx.x];
    // phase times (profiling): thread 0 adds the wall clock between marks
    uint64_t tmark = 0;
    auto mark = [&](int ph) {
        const StepDev& S = args();
        if (S.w_prof && t == 0) {
            const uint64_t now = wall_clock64();
            if (ph >= 0) S.w_prof[(size_t)w * FP_N + ph] += now - tmark;
            tmark = now;
        }
    };
    uint32_t step;
    {
        const StepDev& S = args();
        step = S.w_done[w];
        if (t == 0) {
            s_fs.w = w;
            s_fs.lds_words = lds_words;
            s_fs.E = s_fs.R = s_fs.M = 0u;
            s_fs.X = S.wscr[w];
            if (S.w_tstamp && step < nsteps && step <= S.tcap) S.w_tstamp[(size_t)w * (S.tcap + 1) + step] = wall_clock64();
        }
    }
    __syncthreads();
    mark(-1);
    for (; step < nsteps; ++step) {
        if (args().w_status[w] != WS_OK) break;      // uniform: read before the barrier below
        if (t == 0) s_fs.err = 0u;
        __syncthreads();
        const uint32_t E = uniform(fused_cells<T>(KS, lds, fs));
        if (s_fs.err) {   // (its scan's barriers lie between)
            if (t == 0) args().w_status[w] = (s_fs.err & 2u) ? WS_NONFINITE : WS_CELLS;
            break;
        }
        mark(FP_PREP);
        if (!uniform(fused_room<T>(KS, fs, E, 0u, 0u, 0u))) break;
        fused_buckets<T>(KS, lds, fs);
        mark(FP_BUCKETS);
        const uint32_t R = uniform(fused_count<T>(KS, lds, fs));
        if (!uniform(fused_room<T>(KS, fs, E, R, 0u, 1u))) break;
        fused_emit<T>(KS, lds, fs);
        mark(FP_CANDS);
        const uint32_t M = uniform(fused_narrow<T>(KS, lds, fs));
        mark(FP_NARROW);
        if (!uniform(fused_room<T>(KS, fs, E, R, M, 2u))) break;
        fused_contacts<T>(KS, lds, fs);
        mark(FP_CONTACTS);
        fused_schedule<T, WARM>(KS, lds, fs, sub_steps);
        mark(FP_SCHED);
        // ---- solve
        // (all of LDS but the items per body and their offsets is dead by now)
        if (sub_steps > 0u) {
            if (t == 0) {
                const WorldDev& D = args().worlds[w];
                const uint32_t keep = fused_keep_words((uint32_t)D.nbodies);
                s_chain = ChainShared{w, s_fs.X.i0, s_fs.X.m0, (uint32_t)D.njoints, M, D.body_base, sub_steps, iters, dt, keep,
                                      lds_words - keep, 0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u, {0u, 0u, 0u}, 0u, 0u, 0u};
            }
            __syncthreads();
            chain_world<MAXT, WARM>(KS, lds, (R2D_LDS ChainShared*)&s_chain);
        }
        __syncthreads();
        mark(FP_SOLVE);
        if (sub_steps > 0u && s_chain.failed) break;   // status set
        fused_done<T, WARM>(KS, lds, fs, step);
    }
    // the counts of the world's last step into the call's totals
    __syncthreads();
    if (t < 4) atomicAdd(&args().counters[t], args().w_cnt[8 * (size_t)w + t]);
}

// the end of a step without sub-steps
__global__ void k_commit_step(uint32_t* counters)
{
    if (threadIdx.x == 0 && counters[C_OVERFLOW] == 0u) counters[C_STEPS] += 1u;
}

// ------------------------------------------------------------ host side
static inline unsigned blocks_for(uint64_t n, unsigned bs, unsigned cap = 4096)
{
    uint64_t b = (n + bs - 1) / bs;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (unsigned)b;
}

typedef void (*FusedFn)(StepDev, float, uint32_t, uint32_t, uint32_t, uint32_t);
struct SolveVariant {
    unsigned threads;    // workgroup of the separate launches' chain (CHAIN_THREADS: wide, or CHAIN_NARROW)
    FusedFn fused_fn;    // whole steps per workgroup (nullptr: none)
    unsigned fused_t;    // its workgroup size
};
// Separate launches' workgroups.  The coloured order's slots hold about 700
// points of a 4,096-body pile, eleven waves' rows, and take twelve waves
// (solve 287 -> 257 us a step; sixteen, which spill, were slower); the reference
// order's about 200, and twelve waves cost it their barriers (24 piles 535 ->
// 547, a pile 413 -> 417).  So do coloured worlds whose slots eight waves
// hold, up to 3,000 bodies (solve by eight and twelve waves, 24 piles of 300 /
// 1,000 / 2,500 / 3,000 / 3,500 / 4,096 bodies: 145 / 193 / 261 / 295 / 324 /
// 361 and 148 / 196 / 269 / 293 / 306 / 334 us).
constexpr unsigned CHAIN_THREADS = 512, CHAIN_COLORED = 768, CHAIN_NARROW = 256;
constexpr uint32_t CHAIN_COLORED_BODIES = 3000;
// Solve variants: shapes of the kernels that run worlds' programs.  The fused
// kernels differ in threads and in waves per SIMD (registers); 0, 6 and 8
// have none and take the separate launches.  1, 3, 7 and 9 are alike, and 5
// and 12: the numbers are the interface's and stay.
static const SolveVariant kSolveVariants[SOLVE_TABLE] = {
    {CHAIN_THREADS, nullptr, 0},
    {CHAIN_NARROW, k_fused<256, 3>, 256},
    {CHAIN_NARROW, k_fused<512, 3>, 512},
    {CHAIN_NARROW, k_fused<256, 3>, 256},
    {CHAIN_NARROW, k_fused<256, 2>, 256},
    {CHAIN_NARROW, k_fused<128, 2>, 128},
    {CHAIN_NARROW, nullptr, 0},
    {CHAIN_NARROW, k_fused<256, 3>, 256},
    {CHAIN_NARROW, nullptr, 0},
    {CHAIN_NARROW, k_fused<256, 3>, 256},
    {CHAIN_NARROW, k_fused<256, 4>, 256},
    {CHAIN_NARROW, k_fused<192, 3>, 192},
    {CHAIN_NARROW, k_fused<128, 2>, 128},
    {CHAIN_THREADS, k_fused<512, 2>, 512},
    {CHAIN_THREADS, k_fused<768, 3>, 768},      // WIDE_VARIANT
    {CHAIN_NARROW, k_fused<256, 4, true>, 256}, // WARM_VARIANT (the kernels above carry no warm-start passes)
    {CHAIN_THREADS, k_fused<768, 3, true>, 768}, // WARM_WIDE_VARIANT
};

uint32_t fused_threads(int v)
{
    return kSolveVariants[v].fused_t;
}

// a fused kernel runs only at the workgroup size it was compiled for (its
// loops stride by MAXT): set_solve_smem_limit checks each against the width
// it would be launched with, and a mismatch leaves the variant without one
static bool g_fused_width_ok[SOLVE_TABLE];
static std::atomic<uint32_t> g_fused_groups[SOLVE_TABLE];   // asked once: the same for every context

uint32_t fused_groups(int v)
{
    return std::max(1u, g_fused_groups[v].load(std::memory_order_relaxed));
}

bool fused_available(int v)
{
    return v >= 0 && v < SOLVE_TABLE && kSolveVariants[v].fused_fn != nullptr && g_fused_width_ok[v];
}

hipError_t fused_attributes(int v, hipFuncAttributes* out)
{
    return hipFuncGetAttributes(out, (const void*)kSolveVariants[v].fused_fn);
}

void launch_fused(const StepDev& S, int v, uint32_t nworlds, float dt, uint32_t sub_steps, uint32_t iters,
                  uint32_t nsteps, size_t lds, hipStream_t st)
{
    const SolveVariant& sv = kSolveVariants[v];
    const unsigned threads = fused_threads(v);
    hipLaunchKernelGGL(sv.fused_fn, dim3(nworlds), dim3(threads), lds, st, S, dt, sub_steps, iters, nsteps,
                       (uint32_t)(lds / 4u));
}

void KernelTrace::mark(const char* name, hipStream_t st)
{
    if (marks.size() == pool.size()) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) return;
        pool.push_back(e);
    }
    hipEvent_t e = pool[marks.size()];
    if (hipEventRecord(e, st) != hipSuccess) return;
    marks.push_back({name, e});
}

void KernelTrace::flush()
{
    if (marks.empty()) return;
    (void)hipDeviceSynchronize();
    // a kernel's interval starts at the mark before it
    const Mark* before = nullptr;
    for (const Mark& m : marks) {
        if (before && m.name[0]) {
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, before->ev, m.ev) == hipSuccess) {
                auto& t = totals[m.name];
                t.first += ms;
                t.second += 1;
            }
        }
        before = &m;
    }
    marks.clear();
}

void KernelTrace::report(FILE* f)
{
    flush();
    std::vector<std::pair<double, std::string>> v;
    double all = 0;
    for (auto& kv : totals) { v.push_back({kv.second.first, kv.first}); all += kv.second.first; }
    std::sort(v.rbegin(), v.rend());
    std::fprintf(f, "[r2d] kernel times (eager launches, one event after each):\n");
    for (auto& e : v) {
        const auto& t = totals[e.second];
        std::fprintf(f, "[r2d] %-28s calls %8llu  total %10.3f ms  avg %9.2f us  %5.1f%%\n", e.second.c_str(),
                     (unsigned long long)t.second, t.first, 1e3 * t.first / (double)std::max<uint64_t>(t.second, 1),
                     100.0 * t.first / std::max(all, 1e-9));
    }
}

KernelTrace::~KernelTrace()
{
    for (hipEvent_t e : pool) (void)hipEventDestroy(e);
}

static inline void tmark(const Streams& ss, const char* name, hipStream_t st)
{
    if (ss.trace) ss.trace->mark(name, st);
}

SolvePlan plan_solve(int chosen, const uint32_t* nbodies, size_t nw, uint32_t lds_limit, bool any_colored,
                     bool any_warm, bool allow_wide)
{
    SolvePlan p;
    p.any_colored = any_colored ? 1u : 0u;
    p.any_warm = any_warm ? 1u : 0u;
    p.lds_nmax = lds_limit ? lds_limit : 0xffffffffu;
    const bool wide = (nw <= CHAIN_WIDE_WORLDS && allow_wide) ||
                      (chosen >= 0 && chosen < SOLVE_TABLE && kSolveVariants[chosen].threads == CHAIN_THREADS);
    // LDS: worlds that are alone on their CU take all of it; of larger batches
    // each world takes what its momenta (16 bytes a touched body), impulses (8
    // a point) and plan (20 an item) commonly need, so that CUs hold several
    uint32_t maxn = 0;
    for (size_t i = 0; i < nw; ++i) maxn = std::max(maxn, nbodies[i]);
    p.threads = !wide ? CHAIN_NARROW : any_colored && !any_warm && maxn >= CHAIN_COLORED_BODIES ? CHAIN_COLORED : CHAIN_THREADS;
    const size_t want = std::max<size_t>(CHAIN_LDS_MIN, (size_t)maxn * CHAIN_LDS_BODY);
    p.lds = (uint32_t)(nw <= CHAIN_WIDE_WORLDS ? CHAIN_LDS : std::min<size_t>(CHAIN_LDS, want));
    return p;
}

void launch_phase(const StepDev& S, const Streams& ss, int phase, float dt, uint32_t sub_steps, uint32_t iters,
                  const SolvePlan& sp)
{
    const unsigned BS = 256;
    const unsigned GRID = 1024;   // grid-stride kernels over device-sized ranges
    hipStream_t st = ss.main;
    switch (phase) {
    case PH_BROAD:
        hipLaunchKernelGGL(k_begin_step, dim3(blocks_for(std::max<uint64_t>(std::max(S.nb, S.nbuckets), SCANS * SCAN_TILES), BS, 1024)),
                           dim3(BS), 0, st, S);
        tmark(ss, "k_begin_step", st);
        hipLaunchKernelGGL(k_prep, dim3(blocks_for(S.nb, BS)), dim3(BS), 0, st, S);
        tmark(ss, "k_prep", st);
        scan_u32(S.ncell, S.cell_off, nullptr, S.nb, S.nb, &S.counters[C_ENTRIES], S, 0, st);
        tmark(ss, "scan ncell", st);
        hipLaunchKernelGGL(k_entries, dim3(GRID), dim3(BS), 0, st, S);
        tmark(ss, "k_entries", st);
        scan_u32(S.bkt_cnt, S.bkt_off, nullptr, S.nbuckets, S.nbuckets, nullptr, S, 1, st);
        tmark(ss, "scan bkt_cnt", st);
        hipLaunchKernelGGL(k_bucket_fill, dim3(GRID), dim3(BS), 0, st, S);
        tmark(ss, "k_bucket_fill", st);
        hipLaunchKernelGGL(k_bucket_rank, dim3(GRID), dim3(BS), 0, st, S);
        tmark(ss, "k_bucket_rank", st);
        hipLaunchKernelGGL(k_ent_cnt, dim3(GRID), dim3(BS), 0, st, S);
        tmark(ss, "k_ent_cnt", st);
        scan_u32(S.ent_cnt, S.ent_off, &S.counters[C_ENTRIES], 0, S.cap_e, &S.counters[C_RAW], S, 2, st);
        tmark(ss, "scan ent_cnt", st);
        hipLaunchKernelGGL(k_cand_emit, dim3(GRID), dim3(BS), 0, st, S);
        tmark(ss, "k_cand_emit", st);
        break;
    case PH_NARROW:
        hipLaunchKernelGGL(k_narrow, dim3(GRID), dim3(BS), 0, st, S);
        tmark(ss, "k_narrow", st);
        scan_u32(S.cand_flag, S.cand_idx, &S.counters[C_RAW], 0, S.cap_r, &S.counters[C_MANIFOLDS], S, 3, st, S.it_color,
                 S.cap_m);   // (the colours are written after the list has been read)
        tmark(ss, "scan cand_flag", st);
        hipLaunchKernelGGL(k_man_build, dim3(GRID), dim3(BS), 0, st, S, S.it_color);
        tmark(ss, "k_man_build", st);
        break;
    case PH_SCHED:
        hipLaunchKernelGGL(k_items, dim3(GRID), dim3(BS), 0, st, S);
        tmark(ss, "k_items", st);
        scan_u32(S.deg, S.deg_off, nullptr, S.nb, S.nb, nullptr, S, 4, st);
        tmark(ss, "scan deg", st);
        hipLaunchKernelGGL(k_list_fill, dim3(GRID), dim3(BS), 0, st, S);
        tmark(ss, "k_list_fill", st);
        hipLaunchKernelGGL(k_list_rank<false>, dim3(blocks_for(S.nb, BS)), dim3(BS), 0, st, S);
        tmark(ss, "k_list_rank<false>", st);
        if (sp.any_colored) {
            const size_t lds = S.nworlds <= CHAIN_WIDE_WORLDS ? COLOR_LDS : COLOR_LDS / 4;
            hipLaunchKernelGGL(k_color, dim3(S.nworlds), dim3(COLOR_THREADS), lds, st, S, (uint32_t)(lds / 4u));
            tmark(ss, "k_color", st);
        }
        if (S.nworlds > 1u) {
            hipLaunchKernelGGL(k_world_order, dim3(1), dim3(1024), 0, st, S);
            tmark(ss, "k_world_order", st);
        }
        if (sp.any_colored) {
            hipLaunchKernelGGL(k_list_rank<true>, dim3(blocks_for(S.nb, BS)), dim3(BS), 0, st, S);
            tmark(ss, "k_list_rank<true>", st);
        }
        if (sp.any_warm) {
            hipLaunchKernelGGL(k_warm_match, dim3(GRID), dim3(BS), 0, st, S, sub_steps);
            tmark(ss, "k_warm_match", st);
            hipLaunchKernelGGL(k_warm_sums, dim3(blocks_for(S.nb, BS)), dim3(BS), 0, st, S);
            tmark(ss, "k_warm_sums", st);
        }
        break;
    default: {
        const float sub_dt = dt / (float)sub_steps;
        auto pick = [&](auto warm, auto cold) { return sp.any_warm ? warm : cold; };
        const unsigned T = sp.threads;
        auto width = [&](auto narrow, auto wide, auto widest) {
            return T == CHAIN_NARROW ? narrow : T == CHAIN_COLORED ? widest : wide;
        };
        const uint32_t words = sp.lds / 4u;
        if (sub_steps > 0) {   // without sub-steps nothing of a world changes
            hipLaunchKernelGGL(pick(k_chain_build<true>, k_chain_build<false>), dim3(GRID), dim3(BS), 0, st, S, sub_dt);
            tmark(ss, "k_chain_build", st);
            if (iters > 0) {
                hipLaunchKernelGGL(width(k_chain_plan<CHAIN_NARROW>, k_chain_plan<CHAIN_THREADS>, k_chain_plan<CHAIN_COLORED>),
                                   dim3(S.nworlds), dim3(T), sp.lds, st, S, iters, words, 0u);
                tmark(ss, "k_chain_plan", st);
                if (S.chain_rest) {
                    hipLaunchKernelGGL(width(k_chain_plan<CHAIN_NARROW>, k_chain_plan<CHAIN_THREADS>, k_chain_plan<CHAIN_COLORED>),
                                       dim3(S.nworlds), dim3(T), sp.lds, st, S, iters, words, S.chain_rest);
                    tmark(ss, "k_chain_plan (rest)", st);
                }
            }
        }
        for (uint32_t s = 0; sub_steps > 0; ++s) {
            // (the first one also copies records, about four a body)
            hipLaunchKernelGGL(pick(k_chain_bodies<true>, k_chain_bodies<false>), dim3(blocks_for(s ? S.nb : 4ull * S.nb, BS)),
                               dim3(BS), 0, st, S, s, sub_steps, sub_dt);
            tmark(ss, "k_chain_bodies", st);
            if (s == sub_steps) break;
            auto run = [&](auto rest, const char* name) {
                constexpr bool REST = decltype(rest)::value;
                auto f = width(pick(k_chain_run<CHAIN_NARROW, true, REST>, k_chain_run<CHAIN_NARROW, false, REST>),
                               pick(k_chain_run<CHAIN_THREADS, true, REST>, k_chain_run<CHAIN_THREADS, false, REST>),
                               k_chain_run<CHAIN_COLORED, false, REST>);
                hipLaunchKernelGGL(f, dim3(S.nworlds), dim3(T), sp.lds, st, S, s, iters, sub_dt, words, sp.lds_nmax);
                tmark(ss, name, st);
            };
            run(std::false_type{}, "k_chain_run");
            if (S.chain_rest && iters > 0u) run(std::true_type{}, "k_chain_run (rest)");
        }
        if (sp.any_warm) {
            hipLaunchKernelGGL(k_warm_clear, dim3(blocks_for(S.nb, BS)), dim3(BS), 0, st, S);
            tmark(ss, "k_warm_clear", st);
            hipLaunchKernelGGL(k_warm_save, dim3(GRID), dim3(BS), 0, st, S);
            tmark(ss, "k_warm_save", st);
        }
        if (sub_steps == 0) {
            hipLaunchKernelGGL(k_commit_step, dim3(1), dim3(64), 0, st, S.counters);
            tmark(ss, "k_commit_step", st);
        }
        break;
    }
    }
}

void set_solve_smem_limit()
{
    auto allow = [](const void* f) { (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); };
    allow((const void*)k_color);
    allow((const void*)k_chain_plan<CHAIN_THREADS>);
    allow((const void*)k_chain_plan<CHAIN_NARROW>);
    allow((const void*)k_chain_plan<CHAIN_COLORED>);
    auto chains = [&](auto rest) {
        constexpr bool REST = decltype(rest)::value;
        allow((const void*)k_chain_run<CHAIN_COLORED, false, REST>);
        allow((const void*)k_chain_run<CHAIN_THREADS, false, REST>);
        allow((const void*)k_chain_run<CHAIN_THREADS, true, REST>);
        allow((const void*)k_chain_run<CHAIN_NARROW, false, REST>);
        allow((const void*)k_chain_run<CHAIN_NARROW, true, REST>);
    };
    chains(std::false_type{});
    chains(std::true_type{});
    for (int v = 0; v < SOLVE_TABLE; ++v) {
        if (kSolveVariants[v].fused_fn) {
            allow((const void*)kSolveVariants[v].fused_fn);
            hipFuncAttributes fa{};
            g_fused_width_ok[v] = hipFuncGetAttributes(&fa, (const void*)kSolveVariants[v].fused_fn) == hipSuccess &&
                                  fa.maxThreadsPerBlock == (int)fused_threads(v);
            int groups = 0;
            if (g_fused_groups[v].load(std::memory_order_relaxed) == 0u &&
                hipOccupancyMaxActiveBlocksPerMultiprocessor(&groups, (const void*)kSolveVariants[v].fused_fn,
                                                             (int)fused_threads(v), 0) == hipSuccess)
                g_fused_groups[v].store((uint32_t)std::max(groups, 1), std::memory_order_relaxed);
        }
    }
    (void)hipGetLastError();   // a refused attribute is not an error of a later call
}

}  // namespace r2d
