// The solver's chain as a program: the K iterations of a sub-step's items
// (constraints, then manifolds) laid out ahead of time in rows of at most 64
// lanes, which the waves then run one after another.
//
// The reference's solver is sequential: an item may run once every earlier
// item on its ordering bodies has run.  That partial order is the same in
// every sub-step of a step, so it is worked out once per step (plan_*: the
// items ready now make the next rows, which release their successors) and
// the sub-steps replay the rows (chain_lds and its relatives).  A row's lanes share no
// ordering body and every body meets its items in the reference's order, so
// the bits are the sequential loop's.  Nothing polls: a world whose rows all
// fit one wave runs them in program order, LDS serving one wave's operations
// in the order they are issued, and wider worlds put a workgroup barrier
// between rows.
//
// What bounds it is the length of the dependency chain times one row: two LDS
// reads, about 100 VALU instructions and an LDS write.  Lanes hold contact
// points, not items: the points of a two-point manifold sit in neighbouring
// lanes (the reference computes both from the same momenta and adds their
// impulses up afterwards), which halves the instructions of a row, and a
// one-point manifold (discs) costs one lane.  The 64-byte record of a row's
// points is fetched from L2 while the two rows before it run.
#pragma once

#include "r2d_device.h"

namespace r2d {

typedef float f2v __attribute__((ext_vector_type(2)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
#define R2D_LDS __attribute__((address_space(3)))
#define R2D_GLB __attribute__((address_space(1)))
typedef R2D_LDS uint32_t* LU32;
typedef R2D_LDS uint16_t* LU16;
typedef R2D_LDS u2v* LU2;
typedef R2D_LDS f2v* LF2;
typedef R2D_LDS float* LF;
typedef R2D_GLB f2v* GF2;
typedef R2D_GLB uint32_t* GU32;
typedef R2D_GLB u2v* GU2;
typedef R2D_GLB u4v* GU4;
typedef const R2D_GLB uint32_t* GCU32;
typedef const R2D_GLB u2v* GCU2;
typedef const R2D_GLB u4v* GCU4;

// ------------------------------------------------------------ point records
// 16 words.  Words 0 and 1: the two bodies and flags.
//   contact point: 2-3 normal, 4 friction, 5 Baumgarte bias of the sub-step
//     (-1: depth >= 0, or no point), 6-9 lever arms r1 r2, 10 / 11 effective
//     masses (normal, tangent), 12-13 inverse masses, 14-15 inverse inertias
//   distance joint (type 0): 2-3 direction, 4 position term, 5 / 6 power
//     limits (min, max), 12-13 inverse masses
//   offset distance joint (1): the same, 7-10 rotated offsets, 11 denominator,
//     14-15 inverse inertias
//   fixed position (2): 2-3 direction, 4 bias, 5 / 6 limits, 12 inverse mass
//   motor (3): 2 inertia, 3 target, 4 beta, 5 / 6 limits, 7 torque
constexpr uint32_t PR_INDEX = CHAIN_BODIES - 1u;
enum : uint32_t {
    PR_WRITE = 1u << 31,      // word 0 / 1, contacts: body a / b is an ordering body (its momentum is written)
                              // and this is the manifold's first point
    PR_STATIC = 1u << 30,     // word 0 / 1, contacts: the body is static (an ordering one gets "+= 0")
    PR_JOINT = 1u << 29,      // word 0
    PR_SELF = 1u << 27,       // word 0, joints: both ends on one body
    PR_SKIP = 1u << 28,       // word 0, joints: changes nothing this sub-step
    PR_WARM = 1u << 27,       // word 1, contacts: warm started (no minimum impulse)
    PR_TYPE_SHIFT = 28        // word 1, joints: type
};

// the record of a lane without a point: bias -1, no body to write
__device__ __forceinline__ u4v idle_word(int word) { return word == 1 ? u4v{0u, 0xbf800000u, 0u, 0u} : u4v{0u, 0u, 0u, 0u}; }

__device__ __forceinline__ float asf(uint32_t x) { return __uint_as_float(x); }
__device__ __forceinline__ uint32_t asu(float x) { return __float_as_uint(x); }

// ------------------------------------------------------------------ planning
// An item waits for its ordering bodies (one or two) to reach it; run, it
// releases the next item of each body's list, or the list's first item for
// the next iteration.  One round of a wave (plan_take, plan_run, plan_put)
// turns up to 64 lanes of ready items into a row.  A round is bound by its
// instructions and two LDS round trips: the entry of a ready item carries
// what the round that runs it needs, and the state word needs no decoding --
// (ordering bodies waited for) << 16 | iterations left, so a release
// subtracts 1 << 16 and made its item ready when 1 body and at least one
// iteration were left, and running an item adds its bodies and takes an
// iteration off.  An item with one ordering body releases the spare item (the
// last place), which never becomes ready.
//
// Planning state in LDS, 5 words an item: the entry (x: item | second << 16,
// y: both successors, 15 bits each, SINGLE when there is one ordering body; the
// second point of a pair counts from 1), the state, and a ring of the ready
// items' entries, which are copied as they are.  Worlds that do not fit, or
// with more items than 15 bits, keep the same in global memory (PlanGlb).
constexpr uint32_t PLAN_MAX_ITEMS = 0x7ffe;
constexpr uint32_t STATE_BODY = 1u << 16;

struct PlanEntry {
    uint32_t item, second, s0, s1;   // s1: SINGLE in the top bit when there is one ordering body
};
constexpr uint32_t SINGLE = 0x80000000u;

__host__ __device__ constexpr uint32_t plan_ring(uint32_t nit, uint32_t waves) { return nit + 64u * waves; }
// LDS words of PlanLds
__host__ __device__ constexpr uint32_t plan_lds_words(uint32_t nit, uint32_t waves)
{
    return 2u * plan_ring(nit, waves) + 3u * (nit + 1u);
}
// a state that made its item ready when a release found it
__device__ __forceinline__ bool state_ready(uint32_t old) { return old - (STATE_BODY + 1u) < STATE_BODY - 1u; }

struct PlanLds {
    typedef u2v Raw;
    LU2 ring, items;
    LU32 state;
    uint32_t ring_n;

    __device__ __forceinline__ PlanLds(LU32 p, uint32_t nit, uint32_t waves)
    {
        ring_n = plan_ring(nit, waves);
        ring = (LU2)p;                      // p is 8-byte aligned
        items = ring + ring_n;
        state = (LU32)(items + nit + 1u);
    }
    static __device__ __forceinline__ PlanEntry unpack(u2v v)
    {
        return PlanEntry{v.x & 0xffffu, v.x >> 16, v.y & 0x7fffu, ((v.y >> 16) & 0x7fffu) | (v.y & SINGLE)};
    }
    static __device__ __forceinline__ u2v pack(const PlanEntry& e)
    {
        return u2v{e.item | (e.second << 16), e.s0 | ((e.s1 & 0x7fffu) << 16) | (e.s1 & SINGLE)};
    }
    __device__ __forceinline__ void init(uint32_t j, uint32_t s0, uint32_t s1, uint32_t st, uint32_t sec)
    {
        items[j] = pack(PlanEntry{j, sec, s0, s1});
        state[j] = st;
    }
    __device__ __forceinline__ Raw read(uint32_t at) const { return ring[at]; }
    __device__ __forceinline__ void push(uint32_t at, Raw e) { ring[at] = e; }
    __device__ __forceinline__ Raw entry(uint32_t s) const { return items[s]; }
    __device__ __forceinline__ uint32_t rearm(uint32_t j, uint32_t by)
    {
        return __hip_atomic_fetch_add(&state[j], by, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ uint32_t release(uint32_t s)
    {
        return __hip_atomic_fetch_sub(&state[s], STATE_BODY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

// the same in global memory: items (succ 0, succ 1, state, second), ring of
// ready items (item, second, succ 0, succ 1)
struct PlanGlb {
    typedef PlanEntry Raw;
    static __device__ __forceinline__ PlanEntry unpack(const PlanEntry& e) { return e; }
    static __device__ __forceinline__ PlanEntry pack(const PlanEntry& e) { return e; }
    GU4 items, ring;
    uint32_t ring_n;

    __device__ __forceinline__ PlanGlb(GU4 items_, GU4 ring_, uint32_t nit, uint32_t waves)
        : items(items_), ring(ring_), ring_n(plan_ring(nit, waves))
    {
    }
    __device__ __forceinline__ void init(uint32_t j, uint32_t s0, uint32_t s1, uint32_t st, uint32_t sec)
    {
        items[j] = u4v{s0, s1, st, sec};
    }
    __device__ __forceinline__ PlanEntry read(uint32_t at) const
    {
        const u4v v = ring[at];
        return PlanEntry{v.x, v.y, v.z, v.w};
    }
    __device__ __forceinline__ void push(uint32_t at, const PlanEntry& e) { ring[at] = u4v{e.item, e.second, e.s0, e.s1}; }
    __device__ __forceinline__ GU32 state_of(uint32_t j) const { return (GU32)(items + j) + 2; }
    __device__ __forceinline__ uint32_t rearm(uint32_t j, uint32_t by)
    {
        return __hip_atomic_fetch_add(state_of(j), by, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ uint32_t release(uint32_t s)
    {
        return __hip_atomic_fetch_sub(state_of(s), STATE_BODY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ PlanEntry entry(uint32_t s) const
    {
        const GU32 p = (GU32)(items + s);
        return PlanEntry{s, p[3], p[0], p[1]};
    }
};

// A world's program: rows (first entry; entries | lanes of pairs << 8 |
// ROW_JOINTS when one is a joint), the entries (point indices: item j's first point is j,
// second points follow after the items; pairs first),
// and for worlds run by several waves the first row and the rows of each slot
// (rows of one slot run side by side, one per wave).
constexpr uint32_t ROW_JOINTS = 1u << 16;
struct Program {
    GU2 rows;
    GU32 entries;
    GU2 slots;
};

// Records in program order: entry e's four words of 16 bytes, in blocks of
// four entries, so that a row's lanes read whole 64-byte pieces.  Gathered by
// point, each of a row's four loads touches 64 cache lines, which the CU's
// one address unit takes about 256 cycles a row for: nothing to one wave (a
// row takes 890), but the bound of four or eight waves' slots (4,096-body
// pile: 106 -> 88 us a sub-step).  Joints' records, which change every
// sub-step, stay one a joint: after the entries, in the same blocks.
__device__ __forceinline__ size_t entry_at(uint32_t e) { return (size_t)(e >> 2) * 16u + (e & 3u); }
constexpr uint32_t ENTRY_WORD = 4;   // from one word of an entry to the next
__device__ __forceinline__ void entry_copy(GU4 to, uint32_t e, GCU4 recs, uint32_t point)
{
    const GCU4 q = recs + (size_t)point * 4u;
    const u4v a = q[0], b = q[1], c = q[2], d = q[3];
    const GU4 p = to + entry_at(e);
    p[0] = a; p[ENTRY_WORD] = b; p[2 * ENTRY_WORD] = c; p[3 * ENTRY_WORD] = d;
}

// A world's solve in LDS: what it works on (set by one thread), and the shared
// words of planning.
struct ChainShared {
    uint32_t w, ibase, mbeg, nj, M, base, sub_steps, iters;
    float dt;
    uint32_t free_at, free_words;   // LDS from this word on is the solve's
    uint32_t ready, pairs, live, fix, nslots, failed, taken, entries, queued[3];
    // a plan that the first chain runs behind: LDS words it keeps, rows it has written (PLANNED: all), and the
    // waves that have met (waves_meet)
    uint32_t beside, progress, met;
    uint32_t rest_slots;   // of the program after the others (StepDev::chain_rest)
    uint32_t reps, slow;   // runs of the program a sub-step; its world is slow to plan (StepDev::chain_less)
};
constexpr uint32_t PLANNED = 0x80000000u;

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }
// waits until `waves` waves of the workgroup have called it for the round-th
// time (from 1 on): a barrier of some of the waves, which all reach it
__device__ __forceinline__ void waves_meet(uint32_t* met, uint32_t waves, uint32_t round)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (lane_id() == 0u) __hip_atomic_fetch_add(met, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (__hip_atomic_load(met, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < waves * round)
        __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
__device__ __forceinline__ uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
// The arguments of an out-of-line function arrive in vector registers: what is
// the same in every lane goes back to scalar ones.
template <class P>
__device__ __forceinline__ P uniform_ptr(P p)
{
    const uint64_t x = (uint64_t)p;
    return (P)(((uint64_t)uniform((uint32_t)(x >> 32)) << 32) | uniform((uint32_t)x));
}
template <class P>
__device__ __forceinline__ P uniform_lds(P p)
{
    return (P)(uintptr_t)uniform((uint32_t)(uintptr_t)p);
}

// One round of one wave: takes ready items from ring place `first` on (at most
// `avail`, 64 lanes of points; plan_take), then writes their row's entries at
// `entry0` with pairs in the lower lanes and releases their successors
// (plan_run: the released items are in e0 / e1, r0 / r1 whether the lane
// released one).
template <class PLAN>
struct Round {
    typename PLAN::Raw self, e0, e1;
    uint32_t taken, lanes, word;   // items, points, second word of the row
    bool take, left;               // this lane's item is in the row / did not fit it
    uint32_t below, pairs;         // pairs in lower lanes / in the row
    bool r0, r1;
};

template <class PLAN>
__device__ __forceinline__ Round<PLAN> plan_take(PLAN& P, uint32_t first, uint32_t avail, uint32_t lane, uint32_t nj)
{
    Round<PLAN> R;
    const bool act = lane < avail;
    uint32_t at = first + (act ? lane : 0u);
    at = at < at - P.ring_n ? at : at - P.ring_n;   // at - ring_n wraps round to a large number below the ring's end
    R.self = P.read(at);
    const PlanEntry e = PLAN::unpack(R.self);
    const bool pair = act && e.second != 0u;
    R.below = lanes_below(__ballot(pair));
    R.take = act && lane + 1u + R.below + (pair ? 1u : 0u) <= 64u;   // lanes used through this item
    const uint64_t tm = __ballot(R.take);
    R.taken = (uint32_t)__popcll(tm);
    R.pairs = (uint32_t)__popcll(tm & __ballot(pair));
    R.lanes = R.taken + R.pairs;
    R.word = R.lanes | (R.pairs << 9) | (__ballot(R.take && e.item < nj) ? ROW_JOINTS : 0u);
    R.left = act && !R.take;
    return R;
}

// entry0: a function, called once the releases are under way (the answer of
// another LDS operation is waited for with theirs)
template <class PLAN, class ENTRY0>
__device__ __forceinline__ void plan_run(PLAN& P, Round<PLAN>& R, GU32 entries, ENTRY0 entry0, uint32_t nit, uint32_t lane)
{
    R.r0 = R.r1 = false;
    const PlanEntry e = PLAN::unpack(R.self);
    uint32_t o0 = 0u, o1 = 0u;
    if (R.take) {
        const uint32_t s1 = e.s1 & ~SINGLE;
        P.rearm(e.item, (e.s1 & SINGLE ? STATE_BODY : 2u * STATE_BODY) - 1u);
        o0 = P.release(e.s0);
        o1 = P.release(s1);
        R.e0 = P.entry(e.s0);
        R.e1 = P.entry(s1);
    }
    const uint32_t first = entry0();
    if (R.take) {
        const bool pair = e.second != 0u;
        const uint32_t pos = first + (pair ? 2u * R.below : 2u * R.pairs + (lane - R.below));
        entries[pos] = e.item;
        if (pair) entries[pos + 1u] = nit + e.second - 1u;
        R.r0 = state_ready(o0);
        R.r1 = state_ready(o1);
    }
}

template <class PLAN>
__device__ __forceinline__ void plan_put(PLAN& P, const Round<PLAN>& R, uint32_t at)
{
    const uint64_t m0 = __ballot(R.r0), m1 = __ballot(R.r1), m2 = __ballot(R.left);
    const uint32_t c0 = (uint32_t)__popcll(m0), c2 = (uint32_t)__popcll(m2);
    auto place = [&](uint32_t k) { return k < k - P.ring_n ? k : k - P.ring_n; };
    if (R.left) P.push(place(at + lanes_below(m2)), R.self);
    if (R.r0) P.push(place(at + c2 + lanes_below(m0)), R.e0);
    if (R.r1) P.push(place(at + c2 + c0 + lanes_below(m1)), R.e1);
}

// The program of a world run by one wave, planned by one wave without
// barriers; `ready` items are in the ring from its start on, `entries` are
// written already.  Returns the rows (0: the ordering data was corrupt) and
// adds the entries.
// PUBLISH: `progress` counts the rows that other waves may read (a round's
// stores, three at most, are waited for in the next round).
template <bool PUBLISH = false, class PLAN>
__device__ __forceinline__ uint32_t plan_single(PLAN& P, const Program& G, uint32_t nit, uint32_t nj, uint32_t iters,
                                                uint32_t ready, uint32_t& entries, uint32_t* progress = nullptr)
{
    auto publish = [&](uint32_t rows) {
        asm volatile("" ::: "memory");
        if (lane_id() == 0u) __hip_atomic_store(progress, rows, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t head = 0, count = ready, entry = entries, row = 0, done = 0;
    const uint32_t total = nit * iters;
    while (done < total && count) {
        Round<PLAN> R = plan_take(P, head, count < 64u ? count : 64u, lane, nj);
        R.left = false;                  // stays at the head of the ring
        if (lane == 0) G.rows[row] = u2v{entry, R.word};
        plan_run(P, R, G.entries, [&]() { return entry; }, nit, lane);
        uint32_t tail = head + count;
        if (tail >= P.ring_n) tail -= P.ring_n;
        plan_put(P, R, tail);
        asm volatile("" ::: "memory");   // the next round reads what this one wrote (LDS order)
        const uint32_t added = (uint32_t)(__popcll(__ballot(R.r0)) + __popcll(__ballot(R.r1)));
        head += R.taken;
        if (head >= P.ring_n) head -= P.ring_n;
        count += added - R.taken;
        done += R.taken;
        entry += R.lanes;
        if constexpr (PUBLISH) {
            // at most this round's last two stores are under way: the rows before it are written
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0x0f72);   // vmcnt(2)
            publish(row);
        }
        row += 1u;
    }
    if constexpr (PUBLISH) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0f70);       // vmcnt(0)
        publish((done == total ? row : 0u) | PLANNED);
    }
    entries = entry;
    return done == total ? row : 0u;
}

// The program of a world run by `waves` waves of the workgroup, planned by
// all of them: wave w takes the w-th 64 ready items.  Items that do not fit
// a row go back to the end of the ring.  A barrier per slot; called by the
// whole workgroup.  sh.taken and sh.queued start at 0, sh.entries at the
// entries written already.
template <class PLAN>
__device__ __forceinline__ uint32_t plan_multi(PLAN& P, const Program& G, uint32_t nit, uint32_t nj, uint32_t iters,
                                               uint32_t ready, uint32_t waves, ChainShared& sh)
{
    const uint32_t lane = threadIdx.x & 63u, wv = uniform(threadIdx.x >> 6);
    uint32_t head = 0, count = ready, row = 0, slot = 0;
    const uint32_t limit = nit * iters;
    for (; count && slot < limit; ++slot) {
        const uint32_t want = (count + 63u) / 64u, nrows = want < waves ? want : waves;
        const uint32_t round = slot % 3u;
        uint32_t tail = head + count;
        if (tail >= P.ring_n) tail -= P.ring_n;
        if (threadIdx.x == 0) {
            G.slots[slot] = u2v{row, nrows};
            // every wave read it (as slot - 2's count) before the last barrier; it is added to after the next
            sh.queued[(slot + 1u) % 3u] = 0u;
        }
        if (wv < nrows) {
            const uint32_t rest = count - 64u * wv;
            uint32_t first = head + 64u * wv;
            if (first >= P.ring_n) first -= P.ring_n;
            Round<PLAN> R = plan_take(P, first, rest < 64u ? rest : 64u, lane, nj);
            uint32_t e0 = 0u;
            if (lane == 0) {
                e0 = __hip_atomic_fetch_add(&sh.entries, R.lanes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add(&sh.taken, R.taken, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            plan_run(P, R, G.entries, [&]() { return e0 = uniform(e0); }, nit, lane);
            if (lane == 0) G.rows[row + wv] = u2v{e0, R.word};
            const uint32_t add = (uint32_t)(__popcll(__ballot(R.r0)) + __popcll(__ballot(R.r1)) + __popcll(__ballot(R.left)));
            uint32_t at = 0u;
            if (lane == 0)
                at = __hip_atomic_fetch_add(&sh.queued[round], add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            at = uniform(at) + tail;
            if (at >= P.ring_n) at -= P.ring_n;
            plan_put(P, R, at);
        }
        __syncthreads();
        const uint32_t used = count < 64u * nrows ? count : 64u * nrows;
        head += used;
        if (head >= P.ring_n) head -= P.ring_n;
        count = count - used + uniform(sh.queued[round]);
        row += nrows;
    }
    __syncthreads();
    return sh.taken == limit ? slot : 0u;
}

// Planned through, every item waits for the bodies it waited for at first and
// has no iterations left: with `iters` more it can be planned again.  Lanes t,
// t + stride, ... ; `ready` (0 before) counts the items that wait for nothing,
// which are in the ring from its start on.
template <class PLAN>
__device__ __forceinline__ void plan_again(PLAN& P, uint32_t nit, uint32_t iters, uint32_t t, uint32_t stride, uint32_t* ready)
{
    for (uint32_t j = t; j < nit; j += stride)
        if (P.rearm(j, iters) < STATE_BODY)
            P.push(__hip_atomic_fetch_add(ready, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP), P.entry(j));
}

// The program for the rest of a world's iterations (StepDev::chain_rest), after
// a plan of kc: its rows and slots from kc * nit on, its entries after the
// others (sh.entries).  Called by the whole workgroup after a barrier, with
// sh.taken at 0 in a world of one wave; ends with one.  sh.rest_slots is 0 if
// the ordering data was corrupt.  A function of its own: few calls need it,
// and in the planner's place it costs the others (97 worlds 283 -> 287 us a
// step).
struct PlanMemory {
    LU32 lds;          // of PlanLds, when it fits
    GU4 items, ring;   // of PlanGlb
    Program program;
};
__device__ __attribute__((noinline)) void plan_rest(PlanMemory X, bool in_lds, uint32_t nit, uint32_t nj, uint32_t kc, uint32_t rest,
                                                    uint32_t waves, R2D_LDS ChainShared* shl)
{
    ChainShared& sh = *(ChainShared*)uniform_lds(shl);
    nit = uniform(nit); nj = uniform(nj); kc = uniform(kc); rest = uniform(rest); waves = uniform(waves);
    const Program G{uniform_ptr(X.program.rows) + (size_t)kc * nit, uniform_ptr(X.program.entries),
                    uniform_ptr(X.program.slots) + (size_t)kc * nit};
    auto plan = [&](auto P) {
        if (waves > 1u) {
            if (threadIdx.x == 0) sh.ready = sh.taken = sh.queued[0] = 0u;
            __syncthreads();
            plan_again(P, nit, rest, threadIdx.x, blockDim.x, &sh.ready);
            __syncthreads();
            const uint32_t ns = plan_multi(P, G, nit, nj, rest, uniform(sh.ready), waves, sh);
            if (threadIdx.x == 0) sh.rest_slots = ns;
        } else if (threadIdx.x < 64u) {
            plan_again(P, nit, rest, lane_id(), 64u, &sh.taken);
            asm volatile("" ::: "memory");
            uint32_t entries = uniform(sh.entries);
            const uint32_t ready = uniform(__hip_atomic_load(&sh.taken, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)),
                           ns = plan_single(P, G, nit, nj, rest, ready, entries);
            if (threadIdx.x == 0) {
                sh.rest_slots = ns;
                sh.entries = entries;
            }
        }
    };
    if (uniform(in_lds)) plan(PlanLds(uniform_lds(X.lds), nit, waves));
    else plan(PlanGlb(uniform_ptr(X.items), uniform_ptr(X.ring), nit, waves));
    __syncthreads();
}

// ----------------------------------------------------------------- the chain
// momenta (x, y, angular) of a world's bodies in LDS, 16 bytes a body; the
// SPARE places after the last body take the writes that are not to be kept,
// one a lane: to one place they would be served one after another
constexpr uint32_t SPARE = 64;
typedef float f3v __attribute__((ext_vector_type(3)));
typedef R2D_LDS f3v* LF3;
typedef R2D_GLB f3v* GF3;
struct LdsMomenta {
    LF3 m;
    uint32_t none;
    __device__ __forceinline__ f3v get(uint32_t i) const { return m[i]; }
    __device__ __forceinline__ void put(uint32_t i, f3v v) const { m[i] = v; }
    __device__ __forceinline__ void put_if(bool keep, uint32_t i, f3v v) const { m[keep ? i : none + lane_id()] = v; }
};

// the same in global memory
struct GlbMomenta {
    GF3 m;
    uint32_t none;
    __device__ __forceinline__ f3v get(uint32_t i) const { return m[i]; }
    __device__ __forceinline__ void put(uint32_t i, f3v v) const { m[i] = v; }
    __device__ __forceinline__ void put_if(bool keep, uint32_t i, f3v v) const { if (keep) m[i] = v; }
};

// x of the other lane of an even / odd pair
__device__ __forceinline__ float pair_other(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xf, 0xf, false));
}

// Constraint.solve (Constraints/*.zig) from a joint record
template <class ST>
__device__ __forceinline__ void chain_joint(const u4v& q0, const u4v& q1, const u4v& q2, const u4v& q3, const ST& st, float dt)
{
    const uint32_t type = (q0.y >> PR_TYPE_SHIFT) & 3u, a = q0.x & PR_INDEX, b = q0.y & PR_INDEX;
    if (q0.x & PR_SKIP) return;
    const bool self = (q0.x & PR_SELF) != 0u;
    const float pmin = asf(q1.y), pmax = asf(q1.z);
    const f3v s1 = st.get(a);
    v2 m1 = mk(s1.x, s1.y);
    float L1 = s1.z;
    if (type <= 1u) {
        const f3v s2 = st.get(b);
        v2 m2 = mk(s2.x, s2.y);
        float L2 = s2.z;
        const v2 n = mk(asf(q0.z), asf(q0.w));
        const float pc = asf(q1.x), im1 = asf(q3.x), im2 = asf(q3.y);
        v2 dp;
        if (type == 0u) {
            // DistanceJoint.solve (DistanceJoint.zig:40-75)
            const v2 rv = sub2(scale2(m2, im2), scale2(m1, im1));
            float Jv = -(dot2(rv, n) + pc) / (im1 + im2);
            const float den = 1.0f / maxn(absf(dot2(n, rv)), GRAD_DIV_LIMIT);
            Jv = clampn(Jv, pmin * den, pmax * den);
            dp = scale2(n, Jv);
            m1 = sub2(m1, dp);
            m2 = add2(self ? m1 : m2, dp);
        } else {
            // OffsetDistanceJoint.solve (OffsetDistanceJoint.zig:44-105)
            const v2 rr1 = mk(asf(q1.w), asf(q2.x)), rr2 = mk(asf(q2.y), asf(q2.z));
            const float ii1 = asf(q3.z), ii2 = asf(q3.w);
            const float w1 = L1 * ii1, w2 = L2 * ii2;
            const v2 v1 = add2(scale2(m1, im1), mk(-rr1.y * w1, rr1.x * w1));
            const v2 v2v = add2(scale2(m2, im2), mk(-rr2.y * w2, rr2.x * w2));
            const v2 dv = sub2(v2v, v1);
            const float num = dot2(n, dv) + pc;
            const float r1xn = cross2(rr1, n), r2xn = cross2(rr2, n);
            float Jv = -num / asf(q2.w);
            const float den = 1.0f / maxn(absf(dot2(n, dv)), GRAD_DIV_LIMIT);
            Jv = clampn(Jv, pmin * den, pmax * den);
            dp = scale2(n, Jv);
            m1 = sub2(m1, dp);
            L1 = L1 - Jv * r1xn;
            m2 = add2(self ? m1 : m2, dp);
            L2 = (self ? L1 : L2) + Jv * r2xn;
        }
        // the second end last: with both ends on one body it is the sum of both
        if (!self) st.put(a, f3v{m1.x, m1.y, L1});
        st.put(b, f3v{m2.x, m2.y, type == 0u && self ? L1 : L2});
    } else if (type == 2u) {
        // FixedPositionJoint.solve (FixedPositionJoint.zig:38-72)
        const float w = asf(q3.x);
        const v2 n = mk(asf(q0.z), asf(q0.w));
        const float rv = dot2(scale2(m1, w), n);
        float Jv = -(rv - asf(q1.x)) / w;
        const float den = 1.0f / maxn(absf(rv), ALLOWED_CONSTRAINT_VALUE);
        Jv = clampn(Jv, pmin * den, pmax * den);
        m1 = add2(m1, scale2(n, Jv));
        st.put(a, f3v{m1.x, m1.y, L1});
    } else {
        // MotorJoint.solve (MotorJoint.zig:38-64)
        const float I = asf(q0.z);
        const float C = L1 / I - asf(q0.w);
        if (absf(C) < ALLOWED_CONSTRAINT_VALUE) return;
        const float bias = asf(q1.x) * C;
        const float tq = asf(q1.w);
        float Jv = tq - bias;
        const float den = 1.0f / maxn(absf(tq / I), ALLOWED_CONSTRAINT_VALUE);
        Jv = clampn(Jv, pmin * den, pmax * den);
        st.put(a, f3v{m1.x, m1.y, L1 + Jv * dt});
    }
}

// CollisionManifold.calculateImpulses (collision.zig:135-218), one point per
// lane.  Both points of a manifold work from the same momenta and their
// impulses are added in point order, so the lane of the first point takes the
// second's from its neighbour and writes the bodies.  `paired` lanes, from
// lane 0 on, hold pairs.  A separated point's impulses are zero already (its
// depth is the step's, or was reset with it), so it need only change nothing.
//
// A row is bound by its instructions (a wave issues about one every five
// cycles), so nothing here branches but on what the whole row shares: a write
// that is not to be kept goes to a spare place, a lane without a point has a
// point that does nothing (bias -1, no body to write, a spare impulse).
// fl_a, fl_b: words 0 and 1 for their flags; s1, s2, old: the bodies' momenta
// and the point's impulses, read ahead.
//
// The reference sums an impulse up from +0 and adds the sum to the bodies; it
// does so too where a point does nothing, and to a static body that is an
// ordering body it adds +0.  `fix` does that to the letter.  Without it the
// impulses are added to each other and then to the momenta, with zeros where
// a point does nothing: the same bits as long as no momentum is -0 (which no
// item makes of others), all normals and arms are finite and no ordering body
// is static, which is what the caller asks for.
template <bool WARM, class ST, class ACC>
__device__ __forceinline__ void chain_contact(const u4v& q0, const u4v& q1, const u4v& q2, const u4v& q3, uint32_t fl_a,
                                              uint32_t fl_b, float bias, const ST& st, f3v s1, f3v s2, f2v old, ACC acc,
                                              uint32_t lane, uint32_t paired, bool fix)
{
    const uint32_t a = q0.x & PR_INDEX, b = q0.y & PR_INDEX;
    const v2 n = mk(asf(q0.z), asf(q0.w)), t = rot90cw(n);
    const float fric = asf(q1.x);
    const v2 r1 = mk(asf(q1.z), asf(q1.w)), r2 = mk(asf(q2.x), asf(q2.y));
    const float om1 = s1.z * asf(q3.z), om2 = s2.z * asf(q3.w);
    const v2 v1 = add2(scale2(mk(s1.x, s1.y), asf(q3.x)), mk(-r1.y * om1, r1.x * om1));
    const v2 v2v = add2(scale2(mk(s2.x, s2.y), asf(q3.y)), mk(-r2.y * om2, r2.x * om2));
    const v2 dv = sub2(v1, v2v);
    const float pn = (dot2(dv, n) + bias) * asf(q2.z);
    const float pt = dot2(dv, t) * asf(q2.w);
    const bool go = !(bias < 0.f) && (!(pn < MIN_MANIFOLD_IMPULSE) || (WARM && (fl_b & PR_WARM) != 0u));
    const float new_pn = maxn(0.0f, old.x + pn);
    const float max_pt = fric * absf(new_pn);
    // clampn(old.y + pt, -max_pt, max_pt): a NaN of one side leaves the other
    // (fminf, and a comparison that NaN passes), -0 wins over +0 below
    const float up_pt = __builtin_fminf(old.y + pt, max_pt);
    const float new_pt = !(up_pt <= -max_pt) ? up_pt : -max_pt;
    float apn = new_pn - old.x, apt = new_pt - old.y;
    *acc = f2v{go ? new_pn : old.x, go ? new_pt : old.y};
    f3v m1, m2;
    if (__builtin_expect(!fix, 1)) {
        apn = go ? apn : 0.f;
        apt = go ? apt : 0.f;
        v2 dp = add2(scale2(n, apn), scale2(t, apt));
        float c1 = cross2(r1, dp), c2 = cross2(r2, dp);
        if (lane < paired) {
            dp.x = dp.x + pair_other(dp.x);
            dp.y = dp.y + pair_other(dp.y);
            c1 = c1 + pair_other(c1);
            c2 = c2 + pair_other(c2);
        }
        m1 = f3v{s1.x - dp.x, s1.y - dp.y, s1.z - c1};
        m2 = f3v{s2.x + dp.x, s2.y + dp.y, s2.z + c2};
    } else {
        v2 dp = add2(scale2(n, apn), scale2(t, apt));
        float c1 = cross2(r1, dp), c2 = cross2(r2, dp);
        dp.x = go ? dp.x : 0.f; dp.y = go ? dp.y : 0.f;
        c1 = go ? c1 : 0.f; c2 = go ? c2 : 0.f;
        f3v d1{0.f - dp.x, 0.f - dp.y, 0.f - c1}, d2{0.f + dp.x, 0.f + dp.y, 0.f + c2};
        if (lane < paired) {
            const float ox = pair_other(dp.x), oy = pair_other(dp.y), o1 = pair_other(c1), o2 = pair_other(c2);
            d1 = f3v{d1.x - ox, d1.y - oy, d1.z - o1};
            d2 = f3v{d2.x + ox, d2.y + oy, d2.z + o2};
        }
        if (fl_a & PR_STATIC) d1 = f3v{0.f, 0.f, 0.f};
        if (fl_b & PR_STATIC) d2 = f3v{0.f, 0.f, 0.f};
        m1 = f3v{s1.x + d1.x, s1.y + d1.y, s1.z + d1.z};
        m2 = f3v{s2.x + d2.x, s2.y + d2.y, s2.z + d2.z};
    }
    st.put_if((int32_t)fl_a < 0, a, m1);
    st.put_if((int32_t)fl_b < 0, b, m2);
}

// what the chain reads in global memory, and its sizes: points are those of
// index nj + nacc, the one that does nothing, and below; `idle` is its place
// among the entries; DIRECT programs have joint j's record at entry jbase + j
struct ChainProgram {
    GCU2 rows;
    GCU32 entries;
    GCU2 slots;
    GCU4 recs;
    uint32_t nslots, reps, nj, nacc, idle, jbase;
};
// the program after it (plan_rest): rows and slots from `rows` on
__device__ __forceinline__ ChainProgram rest_program(ChainProgram G, uint32_t rows, uint32_t nslots)
{
    G.rows += rows;
    G.slots += rows;
    G.nslots = nslots;
    G.reps = 1u;
    return G;
}

// Runs a program `reps` times over.  MULTI: the workgroup's waves run the rows
// of a slot side by side, a workgroup barrier after each slot (every wave of
// the workgroup calls it).  DIRECT: recs are in program order (entry_at),
// otherwise by point.
//
// A row is reached through loads that each need the one before (row, entry,
// record), all in L2.  The rows of 63 slots are read at once, one a lane, a
// batch ahead; entries and records run two slots ahead of the stage that uses
// them, so that a load has two slots' time to arrive.  Three buffers a stage,
// the loop unrolled by three: a buffer is never copied while its load is in
// flight.
template <class T>
struct InLds {
    static constexpr bool value = false;
};
template <>
struct InLds<LF2> {
    static constexpr bool value = true;
};
template <>
struct InLds<LdsMomenta> {
    static constexpr bool value = true;
};

template <bool MULTI, bool WARM, bool DIRECT, class ST, class ACC>
__device__ __forceinline__ void chain_run(ChainProgram G, const ST& st, ACC acc, bool fix, float dt)
{
    constexpr bool LDS_ONLY = InLds<ST>::value && InLds<ACC>::value;
    constexpr uint32_t BATCH = 63, AHEAD = 4;   // slots a batch; slots the entry stage runs ahead
    const GCU2 rows = uniform_ptr(G.rows), slots = uniform_ptr(G.slots);
    const GCU32 entries = uniform_ptr(G.entries);
    const GCU4 recs = uniform_ptr(G.recs);
    const uint32_t nslots = uniform(G.nslots), reps = uniform(G.reps), nj = uniform(G.nj), nacc = uniform(G.nacc),
                   idle = uniform(G.idle), jbase = uniform(G.jbase);
    const uint32_t lane = threadIdx.x & 63u, wave = MULTI ? uniform(threadIdx.x >> 6) : 0u;
    const uint32_t end = nslots - 1u;
    for (uint32_t rep = 0; rep < reps; ++rep) {
        uint32_t ent[3], at[3], point[3], cnt_e[3], cnt[3];
        u4v rec[3][4];
        // the rows of slots `first` + lane (past the end: the last again),
        // and in worlds of several waves, before them, the slots
        auto batch_slots = [&](uint32_t first) -> u2v {
            const uint32_t s = first + lane;
            if constexpr (MULTI) return slots[s < end ? s : end];
            return u2v{s < end ? s : end, 1u};
        };
        auto batch_rows = [&](u2v sl) -> u2v {
            const bool mine = wave < sl.y;
            u2v r = rows[sl.x + (mine ? wave : 0u)];
            if constexpr (MULTI) r.y = mine ? r.y : 0u;
            return r;
        };
        // each stage loads into buffer k; lanes without a point take the idle one
        auto load_entry = [&](u2v batch, uint32_t i, int k) {
            const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)batch.x, (int)i);
            const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)batch.y, (int)i);
            const uint32_t e = lane < (c & 0xffu) ? first + lane : idle;
            ent[k] = *(const R2D_GLB uint32_t*)((const R2D_GLB char*)entries + (size_t)(uint32_t)(e * 4u));
            at[k] = e;
            cnt_e[k] = c;
        };
        auto load_rec = [&](int k) {
            if constexpr (DIRECT) {
                const GCU4 q = recs + entry_at(ent[k] < nj ? jbase + ent[k] : at[k]);
                rec[k][0] = q[0]; rec[k][1] = q[ENTRY_WORD]; rec[k][2] = q[2 * ENTRY_WORD]; rec[k][3] = q[3 * ENTRY_WORD];
            } else {
                const GCU4 q = (GCU4)((const R2D_GLB char*)recs + (size_t)(uint32_t)(ent[k] * 64u));
                rec[k][0] = q[0]; rec[k][1] = q[1]; rec[k][2] = q[2]; rec[k][3] = q[3];
            }
            // a register of its own: shared with ent it would be moved, and so
            // waited for, in the slot that loads the next entry
            point[k] = ent[k];
            asm("" : "+v"(point[k]));
            cnt[k] = cnt_e[k];
        };
        // the first loads of every stage, as the loop's iterations -4 .. -1
        // would issue them, in its order: its waits count from either
        u2v batch = batch_rows(batch_slots(0u));
        u2v sl = batch_slots(AHEAD + BATCH);
        u2v next = batch_rows(batch_slots(AHEAD));
        load_entry(batch, 0u, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_entry(batch, 1u, 1);
        __builtin_amdgcn_sched_barrier(0);
        load_rec(0);
        load_entry(batch, 2u, 2);
        __builtin_amdgcn_sched_barrier(0);
        load_rec(1);
        load_entry(batch, 3u, 0);
        __builtin_amdgcn_sched_barrier(0);
        auto wait = [&]() {
            // the next slot reads what this one wrote
            if constexpr (MULTI) {
                if constexpr (LDS_ONLY) {
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                    __builtin_amdgcn_s_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                } else {
                    __syncthreads();
                }
            } else if constexpr (LDS_ONLY) {
                asm volatile("" ::: "memory");   // one wave's LDS operations are served in order
            } else {
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
            }
        };
        auto run_slot = [&](uint32_t i, int u) __attribute__((always_inline)) {
            // this row's LDS reads first: the fetches below are issued while
            // they are under way (joints read something harmless)
            const u4v q0 = rec[u][0], q1 = rec[u][1], q2 = rec[u][2], q3 = rec[u][3];
            const uint32_t rc = cnt[u], left = point[u] - nj;
            const uint32_t ai = left < nacc ? left : nacc;   // joints, and lanes without a point: the spare one
            const f3v s1 = st.get(q0.x & PR_INDEX), s2 = st.get(q0.y & PR_INDEX);
            const f2v old = acc[ai];
            __builtin_amdgcn_sched_barrier(0);
            load_rec((u + 2) % 3);
            load_entry(batch, i, (u + 4) % 3);
            __builtin_amdgcn_sched_barrier(0);
            auto work = [&]() __attribute__((always_inline)) {
                uint32_t fl_a = q0.x, fl_b = q0.y;
                float bias = asf(q1.y);
                if (rc & ROW_JOINTS) {
                    asm volatile("");   // one branch for the row: not folded into the lanes' test
                    const bool joint = (q0.x & PR_JOINT) != 0u;
                    if (joint) chain_joint(q0, q1, q2, q3, st, dt);
                    // as a point it does nothing
                    fl_a = joint ? 0u : fl_a;
                    fl_b = joint ? 0u : fl_b;
                    bias = joint ? -1.0f : bias;
                }
                chain_contact<WARM>(q0, q1, q2, q3, fl_a, fl_b, bias, st, s1, s2, old, acc + ai, lane, (rc >> 8) & 0xffu, fix);
            };
            if constexpr (MULTI) {
                if (rc & 0xffu) {   // this wave has a row in the slot
                    asm volatile("");
                    work();
                }
            } else {
                work();
            }
            wait();
        };
        // whole rounds of the three buffers, a batch of them at a time, then
        // what is left: a way out of the middle of the loop would make its
        // waits those of the shortest path round it (a row's fetches waited
        // for one slot after their issue)
        uint32_t rounds = nslots / 3u, s = 0;
        while (rounds) {
            batch = next;
            next = batch_rows(sl);
            sl = batch_slots(s + AHEAD + 2u * BATCH);
            const uint32_t now = rounds < BATCH / 3u ? rounds : BATCH / 3u;
            for (uint32_t i = 0; i < 3u * now; i += 3u) {
                run_slot(i, 0);
                run_slot(i + 1u, 1);
                run_slot(i + 2u, 2);
            }
            rounds -= now;
            s += 3u * now;
        }
        // (what these fetch is past the end and not used)
        if (s < nslots) run_slot(0u, 0);
        if (s + 1u < nslots) run_slot(1u, 1);
    }
}

// The chain on LDS momenta as an out-of-line call: its registers are then its
// own, whatever the step kernel holds around it.  `accg`: the accumulated
// impulses when they do not fit LDS (acc null).
template <bool MULTI, bool WARM, bool DIRECT>
__device__ __attribute__((noinline)) void chain_lds(ChainProgram G, LF3 m, uint32_t none, LF2 acc, bool fix, float dt)
{
    chain_run<MULTI, WARM, DIRECT>(G, LdsMomenta{uniform_lds(m), uniform(none)}, uniform_lds(acc), uniform(fix) != 0u, dt);
}
template <bool MULTI, bool WARM, bool DIRECT>
__device__ __attribute__((noinline)) void chain_lds_accg(ChainProgram G, LF3 m, uint32_t none, GF2 acc, bool fix, float dt)
{
    chain_run<MULTI, WARM, DIRECT>(G, LdsMomenta{uniform_lds(m), uniform(none)}, uniform_ptr(acc), uniform(fix) != 0u, dt);
}
// momenta and impulses in global memory
template <bool MULTI, bool WARM, bool DIRECT>
__device__ __attribute__((noinline)) void chain_glb(ChainProgram G, GF3 m, uint32_t none, GF2 acc, bool fix, float dt)
{
    chain_run<MULTI, WARM, DIRECT>(G, GlbMomenta{uniform_ptr(m), uniform(none)}, uniform_ptr(acc), uniform(fix) != 0u, dt);
}

}  // namespace r2d
