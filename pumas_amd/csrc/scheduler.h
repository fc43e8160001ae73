/*
 * The wavefront scheduler of the transport: its kernel arguments, tables in
 * LDS, history records and queues, shared by the kernels of pumas_gpu.hip and
 * the stepping kernel (k_step.h).
 */
#ifndef PUMAS_SCHEDULER_H
#define PUMAS_SCHEDULER_H

#include <hip/hip_runtime.h>

#include "../../include/pumas_gpu.h"
#include "engine_transport.h"

using namespace pg;

/* Dynamic LDS of the FP32-bulk stepping kernel: a copy of the single
 * precision tables, made by each block at its start. */
extern __shared__ float pg_lds_floats[];

/* A table column in that copy, as an offset in floats. Reads compile to LDS
 * loads (ds_read) addressed from the symbol, so the table view holding these
 * offsets stays in the kernel arguments (scalar registers). */
struct LdsFloats {
        uint32_t off;

        PG_FN float operator[](int i) const { return pg_lds_floats[off + i]; }
        PG_FN LdsFloats operator+(int k) const
        {
                return LdsFloats{ off + (uint32_t)k };
        }
};

using LdsTables = FloatTablesT<LdsFloats>;

/* The same for the FP64 stepping kernel: the tables read by every step. */
extern __shared__ double pg_lds_doubles[];

struct LdsDoubles {
        uint32_t off;

        PG_FN double operator[](int i) const { return pg_lds_doubles[off + i]; }
        PG_FN double operator*() const { return pg_lds_doubles[off]; }
        PG_FN LdsDoubles operator+(int k) const
        {
                return LdsDoubles{ off + (uint32_t)k };
        }
        PG_FN bool operator==(const LdsDoubles & o) const
        {
                return off == o.off;
        }
};

/* The members of PhysicsView that the per-step lookups read (CEL range,
 * stopping power and its inverse, straggling, DEL cross section, MSC and
 * EHS parameters), as columns of the LDS copy. */
struct LdsStepTables {
        static constexpr bool by_rows = false;
        int n_energies, n_materials;
        double mass;
        LdsDoubles K, X, X_dK, K_dX, dE, dE_dK, Omega, Omega_dK;
        LdsDoubles CS, CS_dK, Mu0, Mu0_dK, Ms1, Ms1_dK, Lb, a_max, b_max;
        const int16_t * k_coarse; /* in HBM, as PhysicsView::k_coarse */
        int k_bin0, k_nbins;
        /* The stepping kernel's lookups rarely miss far: no coarse index
         * code in it. */
        static constexpr bool coarse_index = false;
};

/* The row tables, the whole LDS copy of the FP64 kernels with energy loss. */
struct LdsRowColumn {
        PG_FN double operator[](int i) const { return pg_lds_doubles[i]; }
};

using LdsRowTables = RowTables<LdsRowColumn>;

/* ------------------------------------------------------------------------
 * Transport kernels: a wavefront scheduler over per-phase queues.
 *
 * A batch runs in rounds. k_init loads every history and runs the entry
 * logic of pumas_context_transport; histories that need stepping get a
 * record (their Walker, in HBM) and a slot in the step queue. Each round
 * then runs two kernels:
 *   k_step  persistent; a lane takes a slot from the step queue and steps
 *           that history in registers, elastic hard scatterings (EHS)
 *           included, until it ends or reaches an inelastic DEL vertex,
 *           then writes it back and appends its slot to the DEL queue (one
 *           atomic per wavefront); free lanes refill by ballot;
 *   k_del   one lane per queued DEL, all lanes on the same sampling code;
 *           the histories go back to the next round's step queue.
 * EHS vertices (~16% of the steps of a muon in rock) are batched inside the
 * stepping wavefront: lanes that reach one wait until enough others do.
 * DEL vertices (~0.2% of the steps at a 5% cutoff) leave the wavefront in the
 * rounds of large batches, and leave the stepping loop in the other rounds:
 * the DEL samplers are the largest code of the path (exact DCS models, polar
 * angles, rejection loops) and would hold the stepping kernel's registers
 * for every step. A history's operations are the reference's, in its
 * order; only the interleaving across histories differs, and the random
 * stream of a history is keyed by its id, so results do not depend on the
 * schedule.
 * ------------------------------------------------------------------------ */
enum {
        C_TAKEN = 0, /* step queue entries taken in this round */
        C_STEPS,     /* Monte Carlo steps of finished histories */
        C_ERROR,     /* first error code raised by a history */
        C_STEP_N0,   /* step queue lengths (ping-pong) */
        C_STEP_N1,
        C_DEL_N,     /* DEL queue length */
        C_STATUS,    /* histories ended with HISTORY_STEP_LIMIT, then */
        C_STATUS_LOOP,   /* HISTORY_LOOP_LIMIT and */
        C_STATUS_TARGET, /* HISTORY_NO_TARGET */
        C_COUNT = 12
};

struct KernelArgs {
        PhysicsView p;
        ModelView mv;
        FloatTables ft;
        LdsTables ftl;          /* ft in the stepping kernel's LDS copy */
        LdsStepTables stl;      /* FP64 step tables in the LDS copy */
        LdsRowTables rowl;      /* or the row tables, in the lean kernels' */
        /* The LDS copy of the stepping kernel: up to three pieces, each
         * `n4` 16 B words from `src` to LDS word `dst`. */
        struct {
                const float4 * src;
                uint32_t dst, n4;
        } lds_piece[3];
        int n_lds_pieces;
        Config c;
        pg_geometry g;
        struct pumas_state * states;
        uint64_t n;
        uint64_t seed;
        uint64_t first;
        enum pumas_event * events;
        int32_t * media;
        uint32_t * steps;
        uint32_t * draws;
        int32_t * rc;
        int max_steps;
        int ehs_batch;
        uint32_t resident_lanes; /* of the stepping launch */
        uint64_t wave_del_max;   /* histories of a round up to which DELs are
                                    applied in the wavefronts */
        int lanes_per_wave;      /* lanes of a wavefront taking histories */
        int lanes_auto;          /* fewer in the rounds that fit (k_step) */
        int tail_del;            /* as pumas_gpu_options.tail_del */
        Recorder rec;
        unsigned long long * counters;
        Walker * records;     /* [n] histories in flight */
        uint32_t * q_step[2]; /* [n] step queues (ping-pong) */
        uint32_t * q_del;     /* [n] */
};

/* The arguments are read in place from the kernarg segment (scalar loads of
 * uniform data): naming the by-value parameter's members by reference would
 * make a per-lane scratch copy of it. */
#define KERNEL_ARGS(args)                                                      \
        (void)(args);                                                          \
        const KernelArgs & a =                                                 \
            *(const KernelArgs *)__builtin_amdgcn_kernarg_segment_ptr()

/* Store the end state of history i at `s` and its outputs. `cold` holds the
 * members that a lean engine leaves in the record (`w` itself otherwise). */
__device__ __forceinline__ void walker_store(const KernelArgs & a, uint64_t i,
    const Walker & w, const Walker & cold, struct pumas_state * s)
{
        const Track & t = w.t;
        const int rc = cold.rc;
        s->charge = cold.t.charge;
        s->energy = t.energy;
        s->distance = t.distance;
        s->grammage = t.grammage;
        s->time = t.time;
        s->weight = t.weight;
        s->position[0] = t.pos[0];
        s->position[1] = t.pos[1];
        s->position[2] = t.pos[2];
        s->direction[0] = t.dir[0];
        s->direction[1] = t.dir[1];
        s->direction[2] = t.dir[2];
        s->decayed = cold.t.decayed;
        if (a.events) a.events[i] = (enum pumas_event)cold.event;
        if (a.media) {
                a.media[2 * i] = cold.media0;
                a.media[2 * i + 1] = cold.end_medium;
        }
        if (a.steps) a.steps[i] = t.steps;
        if (a.draws) a.draws[i] = t.rng.count;
        if (a.rc) a.rc[i] = rc;
        if (rc >= HISTORY_STEP_LIMIT)
                atomicAdd(a.counters + C_STATUS + (rc - HISTORY_STEP_LIMIT),
                    1ull);
        else if (rc != RETURN_SUCCESS)
                atomicCAS(a.counters + C_ERROR, 0ull, (unsigned long long)rc);
}

/* Write a history of a lean engine back to its record: the members that it
 * keeps in registers. */
template <bool F32>
__device__ __forceinline__ void walker_save(Walker * r, const Walker & w)
{
        r->t.energy = w.t.energy;
        r->t.distance = w.t.distance;
        r->t.grammage = w.t.grammage;
        r->t.time = w.t.time;
        r->t.weight = w.t.weight;
        for (int i = 0; i < 3; i++) {
                r->t.pos[i] = w.t.pos[i];
                r->t.dir[i] = w.t.dir[i];
        }
        r->t.step_first = w.t.step_first;
        r->t.step_event = w.t.step_event;
        r->t.step_foreseen = w.t.step_foreseen;
        r->t.step_invlb1 = w.t.step_invlb1;
        r->t.randn_done = w.t.randn_done;
        r->t.randn_next = w.t.randn_next;
        r->t.ix = w.t.ix;
        if constexpr (F32) r->t.fx = w.t.fx;
        r->t.rng.count = w.t.rng.count;
        r->t.rng.next_lo = w.t.rng.next_lo;
        r->t.rng.next_hi = w.t.rng.next_hi;
        r->t.steps = w.t.steps;
        r->t.max_steps = w.t.max_steps;
        r->phase = w.phase;
        r->medium = w.medium;
        r->material = w.material;
        r->straight = w.straight;
        r->step_index = w.step_index;
        r->step_max_type = w.step_max_type;
        r->density = w.density;
        r->step_max_medium = w.step_max_medium;
        r->step_max_locals = w.step_max_locals;
        r->ti = w.ti;
        r->dei = w.dei;
        r->grammage_max = w.grammage_max;
}

__device__ __forceinline__ uint64_t lanes_below()
{
        const int lane = threadIdx.x & 63;
        return (lane == 0) ? 0ull : (~0ull >> (64 - lane));
}

/* Append `slot` to `queue` for the lanes where `pred` holds: one atomic per
 * wavefront, positions by prefix count. Called by all lanes of the wave. */
__device__ __forceinline__ void queue_append(unsigned long long * count,
    uint32_t * queue, bool pred, uint32_t slot)
{
        const uint64_t m = __ballot(pred);
        if (!m) return;
        const int leader = __ffsll((unsigned long long)m) - 1;
        unsigned long long base = 0;
        if ((int)(threadIdx.x & 63) == leader)
                base = atomicAdd(count, (unsigned long long)__popcll(m));
        base = __shfl(base, leader, 64);
        if (pred) queue[base + __popcll(m & lanes_below())] = slot;
}

/* Sum a per-lane step tally over the wave into the global counter. */
__device__ __forceinline__ void steps_flush(
    const KernelArgs & a, unsigned long long acc)
{
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
        if ((threadIdx.x & 63) == 0 && acc) atomicAdd(a.counters + C_STEPS, acc);
}

/*
 * Schedule of the stepping rounds. Slabs forward FP64, and the same with
 * backward voxels (1 % cutoff, a DEL every 20 steps), 256 CUs x 512 lanes.
 *
 * WAVE_DEL_ROUNDS: a round of at most so many times the resident lanes has its
 * DELs in the wavefronts, so that it ends the batch; a larger one queues them
 * for a kernel that runs 64 of them per wavefront. 1 (and queued until the
 * step queue is exhausted): 2x10^5 muons 147 ms, 10^6 354, 3x10^6 809, voxels
 * 10^6 121; 2: 74, 324, 782, 119; 4: 77, 306, 775, 121; 8: 77, 292, 771, 139.
 * DEL_BATCH, DEL_WAIT: such DELs run when so many lanes, or as many as the
 * others in flight, wait for one, or after so many steps of the others, as
 * one lane's DEL costs the wavefront as much as many lanes'. At once: voxels
 * 5x10^4 35.9 ms, terrain 10^5 62.1; 8, 32: 27.6, 55.7; 24, 48: 26.6, 55.9.
 * HAND_OVER: in a larger round, a wavefront with fewer than so many of 64
 * lanes left, once the step queue is exhausted, puts its histories in the next
 * round's queue, instead of stepping them until the last one ends: 0: 10^6
 * muons 379 ms, voxels 10^6 179, terrain 6x10^5 200; 32: 354, 128, 137; 48:
 * 377, 126, 131. Not before HAND_OVER_AFTER steps, so that every round makes
 * progress.
 * PACK_LANES: a round that fits with more than so many lanes per wavefront, and
 * in half of the wavefronts of each 512 lane block, is put in that half: one
 * wavefront per SIMD with twice the lanes. In infinite media and slabs: 30011
 * muons 48.2 -> 45.2 ms, 60000 53.4 -> 48.6, 17000 to 64000 histories 2 to 22 %
 * in every energy loss mode and precision; below it loses: 3000 29.8 -> 32.7,
 * 10000 38.6 -> 40.6. In terrains and voxel grids (PACK_LANES_GRID), whose
 * locations load per lane, it loses longer: 24000 histories, mixed losses,
 * terrain 43.4 -> 48.7 ms, voxels 22.3 -> 25.2, straggled 37.8 -> 40.5 and 19.0
 * -> 20.9, 40000 43.0 -> 43.9 and 22.5 -> 23.1; 50021 voxel histories 24.7 ->
 * 24.1, 64000 46.9 -> 44.6 and 25.5 -> 24.8.
 */
constexpr uint64_t WAVE_DEL_ROUNDS = 4;
constexpr int DEL_BATCH = 24;
constexpr int DEL_WAIT = 48;
constexpr int HAND_OVER = 40;
constexpr int HAND_OVER_AFTER = 32;
constexpr uint32_t PACK_LANES = 8;
constexpr uint32_t PACK_LANES_GRID = 22;

/* The stepping kernel of a launch, in an energy loss mode, with the tables in
 * LDS or in HBM (step_*.hip: compiled apart, which is most of the build's
 * time). */
using StepKernel = void (*)(KernelArgs, int);

template <bool F32, bool RECORD>
StepKernel step_kernel(int energy_loss, bool lds);

#endif
