// Host-side entry points of the step kernels (r2d_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdio>
#include <map>
#include <string>
#include <vector>

#include "r2d_device.h"

namespace r2d {

// phase markers recorded by the optional per-step timer
enum { KT_BROAD_BEGIN = 0, KT_NARROW_BEGIN, KT_SCHED_BEGIN, KT_SOLVE_BEGIN, KT_END, KT_N };


// the four phases of one step, enqueued in this order on one stream
enum { PH_BROAD = 0, PH_NARROW, PH_SCHED, PH_SOLVE, PH_N };

// solve variants: shapes of the kernels that run worlds' programs (table in
// r2d_kernels.hip)
constexpr int SOLVE_VARIANTS = 15;
// the default for worlds that are each alone on a CU
constexpr int WIDE_VARIANT = 14;
// batches with a warm-started world take these (not tunable): several worlds
// a CU, and one
constexpr int WARM_VARIANT = SOLVE_VARIANTS, WARM_WIDE_VARIANT = SOLVE_VARIANTS + 1;
constexpr int SOLVE_TABLE = SOLVE_VARIANTS + 2;

// Iterations of a sub-step that one program covers: all of them up to 16,
// else their largest divisor from 4 to 16 (the program is then run that
// often), else 4, with a program of its own for the rest (17 = 4 x 4 + 1).  A
// program's size grows with the iterations it covers, and what a program
// covers runs overlapped: an iteration by itself costs the whole depth of the
// world's contacts.  Four take most of that away (ms a step of 16 iterations by
// programs of 1 / 4 / 16: 20-row pyramid 2.18 / 0.79 / 0.51, 60 rows 10.0 /
// 4.7 / 2.7, world of 387 bodies 0.58 / 0.61 / 0.60, 97 worlds 0.78 / 0.80 /
// 0.80, 4,096-body pile 1.47 / 1.24 / 1.54).  17 iterations, one at a time and by fours: pyramids of 20 and 60
// rows 2.29 -> 0.96 and 9.5 -> 5.2 ms, 4,096-body pile 1.43 -> 1.34; shallow
// worlds pay for planning more, 387 bodies 0.61 -> 0.65, 97 worlds 0.79 -> 0.88.
constexpr uint32_t CHAIN_ITERS_MAX = 16, CHAIN_ITERS_ENOUGH = 4;
struct ChainSplit {
    uint32_t each, rest;   // iterations of the program, and of the one that ends a sub-step
    uint32_t room() const { return each + rest; }
};
// most: a smaller bound where memory holds no more (CHAIN_SHORT: fours, and
// ones; 1: ones)
constexpr uint32_t CHAIN_SHORT = 2 * CHAIN_ITERS_ENOUGH - 1;
inline ChainSplit chain_split(size_t iters, uint32_t most = CHAIN_ITERS_MAX)
{
    if (iters == 0 || most < CHAIN_SHORT) return ChainSplit{1u, 0u};
    if (iters <= most) return ChainSplit{(uint32_t)iters, 0u};
    for (uint32_t k = most; k >= CHAIN_ITERS_ENOUGH; --k)
        if (iters % k == 0) return ChainSplit{k, 0u};
    return ChainSplit{CHAIN_ITERS_ENOUGH, (uint32_t)(iters % CHAIN_ITERS_ENOUGH)};
}

// Iterations of the programs of worlds that are slow to plan, in a step of one
// sub-step, which runs what it plans that one time: their largest divisor up
// to a quarter of them (up to two, of three to eleven; one, of two), or 0: as
// the other worlds.  Slow are plans in global memory and, in the one-kernel
// step, plans by several waves; one wave's first chain runs behind its planner.
// One sub-step of 8 iterations by programs of 8 and of 2, and before there were
// programs: a disturbed 4,096-body pile of more items than LDS plans 2.75, 1.18
// and 2.00 ms a step, 1,000 bodies 521, 355 and 509 us.  (All worlds by such
// programs: deep ones lose more than their plan costs, a rope of 900 links
// 1,160 us a step of 4 iterations, then 2,840.)
inline uint32_t chain_less(size_t sub_steps, size_t iters, uint32_t each)
{
    if (sub_steps != 1) return 0u;
    for (size_t k = iters == 2 ? 1 : iters / 4 < 2 ? 2 : iters / 4; k > 0; --k)
        if (iters % k == 0) return k < each ? (uint32_t)k : 0u;
    return 0u;
}

// Waves that run a world's rows: one for each `rows` rows of 64 its items fill
// (a pile's chain is 90-150 slots deep for 4 iterations).  In the one-kernel
// step a slot of several waves costs about two rows of one, so they pay from
// 96 rows on (97 worlds x 8 steps, when this line was drawn: 3.40 ms, with 48
// 4.45 ms; 2.26 now).  In the separate
// launches, records in program order, wider is better down to a wave for 32
// rows (solve of a 4,096-body pile, 96 / 48 / 24 rows: 529 / 499 / 498 us;
// coloured 417 / 311 / 308).
// Whether several pay in the one-kernel step is asked of four iterations at
// most: more of them make a program longer, not wider.  Asked of all, sixteen
// iterations took several waves from 384 items on (20-row pyramid 954 us a
// step, now 512; 387 bodies 988 and 602; 97 worlds 1,340 and 802).
constexpr uint32_t FUSED_WAVE_ROWS = 96, CHAIN_WAVE_ROWS = 32, FUSED_WAVE_ITERS = 4;
__host__ __device__ inline uint32_t chain_waves(uint32_t nit, uint32_t iters, uint32_t most, uint32_t rows)
{
    const uint32_t w = (uint32_t)(((uint64_t)nit * iters / 64u + rows - 1u) / rows);
    return w < 1u ? 1u : (w < most ? w : most);
}
__host__ __device__ inline uint32_t fused_waves(uint32_t nit, uint32_t iters, uint32_t most)
{
    const bool several = chain_waves(nit, iters < FUSED_WAVE_ITERS ? iters : FUSED_WAVE_ITERS, most, FUSED_WAVE_ROWS) > 1u;
    return several ? chain_waves(nit, iters, most, FUSED_WAVE_ROWS) : 1u;
}

// The separate launches' chain: batches of at most this many worlds (one per
// CU) take wide workgroups and all of LDS.
constexpr size_t CHAIN_WIDE_WORLDS = 256;
constexpr size_t CHAIN_LDS = 159 * 1024, CHAIN_LDS_MIN = 16 * 1024, CHAIN_LDS_BODY = 40;

// how one batch's solve phase is launched
struct SolvePlan {
    uint32_t lds = 0;          // dynamic LDS of a world's workgroup
    uint32_t lds_nmax = 0;     // bodies a world may have to keep its momenta in LDS
    uint32_t threads = 0;      // of the chain's workgroups
    uint32_t any_colored = 0;  // some world uses the coloured schedule
    uint32_t any_warm = 0;     // some world is warm started
};
// chosen: the variant that the caller chose (-1: none); lds_limit: largest
// world (bodies) that keeps its momenta in LDS (0: as many as LDS holds);
// allow_wide: small batches may take wide chains whose caller chose none
SolvePlan plan_solve(int chosen, const uint32_t* nbodies, size_t nw, uint32_t lds_limit, bool any_colored,
                     bool any_warm, bool allow_wide = true);

// Optional per-kernel timing (a context created with R2D_TRACE_KERNELS set):
// an event after every launch, summed per kernel name; the steps run eagerly.
struct KernelTrace {
    struct Mark {
        const char* name;
        hipEvent_t ev;
    };
    std::vector<Mark> marks;
    std::vector<hipEvent_t> pool;
    std::map<std::string, std::pair<double, uint64_t>> totals;
    void mark(const char* name, hipStream_t st);
    void flush();                 // synchronise and add the recorded intervals
    void report(FILE* f);
    ~KernelTrace();
};

// the context's stream
struct Streams {
    hipStream_t main;
    KernelTrace* trace;
};

// enqueue one phase of a batched step (phases in PH_* order on ss.main)
void launch_phase(const StepDev& S, const Streams& ss, int phase, float dt, uint32_t sub_steps, uint32_t iters,
                  const SolvePlan& sp);

void scan_u32(const uint32_t* in, uint32_t* out, const uint32_t* n_dev, uint32_t n_const, uint32_t cap,
              uint32_t* total_dev, const StepDev& S, int which, hipStream_t st, uint32_t* where = nullptr,
              uint32_t where_cap = 0);

void set_solve_smem_limit();

// Whole steps per workgroup (k_fused) for worlds of at most FUSED_NMAX bodies
// in the reference order; the variant picks threads and workgroups a CU.
constexpr uint32_t FUSED_NMAX = 1024;
bool fused_available(int variant);
// dynamic LDS of the fused kernel for a world of n bodies and tb hash buckets
size_t fused_lds_bytes(uint32_t n, uint32_t tb);
uint32_t fused_threads(int variant);
// workgroups of it that a compute unit's registers hold
uint32_t fused_groups(int variant);
// one workgroup per world (S.w_order), up to nsteps steps per world (S.w_done)
// the fused kernel of a variant as compiled (registers, LDS, scratch): for error reports
hipError_t fused_attributes(int variant, hipFuncAttributes* out);
void launch_fused(const StepDev& S, int variant, uint32_t nworlds, float dt, uint32_t sub_steps, uint32_t iters,
                  uint32_t nsteps, size_t lds, hipStream_t st);

}  // namespace r2d
