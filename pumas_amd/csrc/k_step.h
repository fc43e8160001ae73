/*
 * The stepping kernel, and its choice for a launch. Included by the files that
 * compile it, one per precision.
 */
#ifndef PUMAS_K_STEP_H
#define PUMAS_K_STEP_H

#include <type_traits>

#include "scheduler.h"

/* The kernel arguments at `args` (the kernarg segment), the same for every
 * lane: in scalar registers, so that their members are scalar loads also in
 * out-of-line code. */
__device__ __forceinline__ const KernelArgs & uniform_args(
    const KernelArgs * args)
{
        typedef const __attribute__((address_space(4))) KernelArgs cargs;
        const uint64_t v = (uint64_t)args;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        return *(const KernelArgs *)(cargs *)(((uint64_t)hi << 32) | lo);
}

/* The pending DELs of a stepping wavefront's histories, on their records.
 * Out of line: the DEL samplers are the largest code of the path. */
template <bool F32>
__device__ __noinline__ void del_wave(
    const KernelArgs * args, uint32_t slot, bool pending)
{
        const KernelArgs & a = uniform_args(args);
        if (!pending) return;
        const EngineT<F32> eng = { a.p, a.mv, a.c, a.g, a.ft, a.p, a.rec };
        Walker w = a.records[slot];
        eng.walker_del(w);
        a.records[slot] = w;
}

/*
 * Stepping: persistent over the step queue of round `parity`. In a round of at
 * most a.wave_del_max histories (or always, a.tail_del > 0) a wavefront
 * applies the DELs of its histories itself instead of queueing them for the
 * next round: the last histories of a batch, and small batches, then run to
 * their end without a round barrier per DEL.
 *
 * The DELs run outside of the stepping loop, on the records: the wavefront
 * saves its histories, calls the DEL code and reloads them, so that nothing
 * of the stepping loop is live in registers across the call. As compiled, the
 * kernels with DELs spill 63 to 90 registers around the call and none in the
 * loop, those without DELs (CSDA, no energy loss) none at all. Variants with the
 * call inside of the loop spilled 200 to 1400 registers on every step.
 */
template <bool F32, bool LDS, bool RECORD, int SCHEME>
__global__ void __launch_bounds__(512, 2) k_step(KernelArgs args, int parity)
{
        KERNEL_ARGS(args);
        /* With LDS, the tables of the step lookups in the working precision
         * are read from a copy in LDS: the FP32 mirrors (FP32-bulk), the row
         * tables (FP64 with energy loss) or the packed FP64 step
         * tables. */
        using FT = typename std::conditional<LDS && F32, LdsTables,
            FloatTables>::type;
        constexpr bool ROWS = LDS && !F32 && (SCHEME >= MODE_CSDA);
        using ST = typename std::conditional<ROWS, LdsRowTables,
            typename std::conditional<LDS, LdsStepTables,
                PhysicsView>::type>::type;
        const FT * ft;
        const ST * st;
        if constexpr (LDS && F32)
                ft = &a.ftl;
        else
                ft = &a.ft;
        if constexpr (ROWS)
                st = &a.rowl;
        else if constexpr (LDS)
                st = &a.stl;
        else
                st = &a.p;
        const EngineT<F32, FT, ST, true, SCHEME, RECORD> eng = { a.p, a.mv, a.c,
                a.g, *ft, *st, a.rec, a.records };
        /* The modes with inelastic DELs. The others have no DEL call, and
         * spill nothing around it (10^6 muons, CSDA: 205 -> 196 ms, FP32 186
         * -> 181). */
        constexpr bool DELS = SCHEME > MODE_CSDA;
        const uint64_t below = lanes_below();
        const uint32_t * in = a.q_step[parity];
        const unsigned long long n_in = a.counters[C_STEP_N0 + parity];
        if (n_in == 0) return;
        if constexpr (LDS) {
                /* The copy (tens of KB to 160 KB, read from L2 by every
                 * block of the launch), in 16 B words. */
                float4 * lds = (float4 *)pg_lds_floats;
                for (int k = 0; k < a.n_lds_pieces; k++) {
                        const float4 * src = a.lds_piece[k].src;
                        float4 * dst = lds + a.lds_piece[k].dst;
                        for (uint32_t i = threadIdx.x; i < a.lds_piece[k].n4;
                             i += blockDim.x)
                                dst[i] = src[i];
                }
                __syncthreads();
        }
        uint32_t slot = 0;
        bool exhausted = false;
        /* A round that fits in the resident lanes: each wavefront takes its
         * share of the queue once, and the queue has nothing more for it.
         * (Taken from the shared counter instead, a wavefront learns that
         * only when it asks again, with a lane freed by its first DEL: with
         * one history per wavefront every DEL cost a round.) The shares are
         * spread over all wavefronts, first over the blocks, then over the
         * wavefronts of a block, unless the caller asked for a number of
         * lanes. */
        const bool fits = n_in <= a.resident_lanes;
        uint32_t waves = gridDim.x * (blockDim.x >> 6);
        const bool grid =
            (a.g.kind == GEO_TERRAIN) || (a.g.kind == GEO_VOXELS);
        if ((blockDim.x == 512) &&
            (n_in > waves * (grid ? PACK_LANES_GRID : PACK_LANES)) &&
            (n_in <= waves * 32))
                waves /= 2;
        const int lanes = (fits && a.lanes_auto) ?
            (int)((n_in + waves - 1) / waves) :
            a.lanes_per_wave;
        const bool lane_on = (int)(threadIdx.x & 63) < lanes;
        const bool wave_del = (a.tail_del > 0) ||
            ((a.tail_del == 0) && (n_in <= a.wave_del_max));
        /* Lanes below which the histories left are handed over. */
        const int keep = (wave_del || fits) ? 0 : (lanes * HAND_OVER) / 64;
        unsigned long long steps_acc = 0;
        bool held = false; /* the lane has a history, saved in its record */
        uint64_t del_mask = 0; /* lanes with a DEL to apply here */
        int del_wait = 0;
        bool finished = false;
        do {
                Walker w;
                w.phase = PHASE_EMPTY;
                if (held) w = a.records[slot];
                for (int it = 0;; it++) {
                        /* Hand over the histories that left the stepping
                         * phase. */
                        const bool done = w.phase == PHASE_DONE;
                        const bool del = w.phase == PHASE_DEL;
                        if (done) {
                                walker_store(a, slot, w, a.records[slot],
                                    a.states + slot);
                                steps_acc += w.t.steps;
                        }
                        const bool to_del = DELS && del && !wave_del;
                        uint64_t dels = DELS ? __ballot(del && wave_del) : 0;
                        if (dels) {
                                const int others = __popcll(
                                    __ballot((w.phase == PHASE_STEP) ||
                                        (w.phase == PHASE_EHS)));
                                const int waiting = __popcll(dels);
                                if ((waiting < others) &&
                                    (waiting < DEL_BATCH) &&
                                    (++del_wait <= DEL_WAIT))
                                        dels = 0; /* not yet */
                                else
                                        del_wait = 0;
                        }
                        bool to_step = false;
                        if (keep && exhausted && (it > HAND_OVER_AFTER)) {
                                const bool left = (w.phase == PHASE_STEP) ||
                                    (w.phase == PHASE_EHS);
                                to_step = left &&
                                    (__popcll(__ballot(left)) < keep);
                        }
                        const bool save = to_del || to_step ||
                            (dels && (w.phase != PHASE_EMPTY) && !done);
                        if (save)
                                walker_save<F32>(a.records + slot, w);
                        queue_append(
                            a.counters + C_DEL_N, a.q_del, to_del, slot);
                        queue_append(a.counters + C_STEP_N0 + (parity ^ 1),
                            a.q_step[parity ^ 1], to_step, slot);
                        if (dels) {
                                /* DELs in the wavefront, below. */
                                held = save;
                                del_mask = dels;
                                break;
                        }
                        if (done || to_del || to_step)
                                w.phase = PHASE_EMPTY;

                        /* Refill the free lanes from the step queue. */
                        if (!exhausted) {
                                const uint64_t free_lanes = __ballot(
                                    (w.phase == PHASE_EMPTY) && lane_on);
                                if (free_lanes) {
                                        const int count = __popcll(free_lanes);
                                        unsigned long long base = 0;
                                        if (fits) {
                                                base = (unsigned long long)
                                                    lanes *
                                                    ((threadIdx.x >> 6) *
                                                            gridDim.x +
                                                        blockIdx.x);
                                                exhausted = true;
                                        } else {
                                                const int leader =
                                                    __ffsll((unsigned long
                                                        long)free_lanes) - 1;
                                                if ((int)(threadIdx.x & 63) ==
                                                    leader)
                                                        base = atomicAdd(
                                                            a.counters +
                                                                C_TAKEN,
                                                            count);
                                                base = __shfl(
                                                    base, leader, 64);
                                                if (base + count >= n_in)
                                                        exhausted = true;
                                        }
                                        if ((w.phase == PHASE_EMPTY) &&
                                            lane_on) {
                                                const unsigned long long k =
                                                    base +
                                                    __popcll(
                                                        free_lanes & below);
                                                if (k < n_in) {
                                                        slot = in[k];
                                                        w = a.records[slot];
                                                }
                                        }
                                }
                        }
                        if (!__ballot((w.phase == PHASE_STEP) ||
                                (w.phase == PHASE_EHS))) {
                                if (exhausted) {
                                        finished = true;
                                        break;
                                }
                                continue;
                        }
                        /* In scalar registers: the same for every history. */
                        w.t.rng.k0 = (uint32_t)a.seed;
                        w.t.rng.k1 = (uint32_t)(a.seed >> 32);
                        w.t.rng.stream = STREAM_TRANSPORT;
                        w.slot = slot;
                        if (w.phase == PHASE_STEP) eng.walker_step(w);

                        /* Elastic hard scatterings, on ~16% of the steps of
                         * a muon in rock, run once enough lanes wait for one
                         * (half of the lanes in flight, at most a.ehs_batch)
                         * or none can step, so that the wavefront runs that
                         * code with most lanes busy. */
                        const uint64_t ehs = __ballot(w.phase == PHASE_EHS);
                        const uint64_t stepping =
                            __ballot(w.phase == PHASE_STEP);
                        const int waiting = __popcll(ehs);
                        const int in_flight = waiting + __popcll(stepping);
                        const int batch =
                            (in_flight + 1) / 2 < a.ehs_batch ?
                            (in_flight + 1) / 2 :
                            a.ehs_batch;
                        if (ehs && ((waiting >= batch) || !stepping)) {
                                if (w.phase == PHASE_EHS) eng.walker_ehs(w);
                        }
                }
                if constexpr (DELS) {
                        if (!finished)
                                del_wave<F32>(&a, slot,
                                    (del_mask >> (threadIdx.x & 63)) & 1);
                }
        } while (!finished);
        steps_flush(a, steps_acc);
}

/* The stepping kernel of a launch: compiled for its energy loss mode, and with
 * or without a frame recorder. In one kernel for every mode, which launches with
 * a recorder, with the tables in HBM or without energy loss took, 10^6 muons
 * through the slabs: recorder, CSDA 252 ms (FP32 247) instead of 199 (186), no
 * loss 66 (65) instead of 51 (44); HBM, CSDA 277 (288) instead of 216 (193). With
 * the recorder's code in all of them, launches without one lose 1 to 6 %. */
template <bool F32, bool LDS, bool RECORD>
StepKernel step_kernel_mode(int energy_loss)
{
        switch (energy_loss) {
        case MODE_STRAGGLED:
                return k_step<F32, LDS, RECORD, MODE_STRAGGLED>;
        case MODE_MIXED:
                return k_step<F32, LDS, RECORD, MODE_MIXED>;
        case MODE_CSDA:
                return k_step<F32, LDS, RECORD, MODE_CSDA>;
        default:
                return k_step<F32, LDS, RECORD, SCHEME_NONE>;
        }
}

template <bool F32, bool RECORD>
StepKernel step_kernel(int energy_loss, bool lds)
{
        return lds ? step_kernel_mode<F32, true, RECORD>(energy_loss) :
                     step_kernel_mode<F32, false, RECORD>(energy_loss);
}

#endif
