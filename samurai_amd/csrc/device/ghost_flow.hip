// update_ghost_mr as one dataflow launch.
//
// The update is a chain of stages (per level, finest first: outer ghosts, then
// the projection into the level below; then the predictions, coarsest level
// first), 37 of them on a 2D L4..12 mesh.  Most ghosts do not need that
// order: a ghost waits only for the ghosts it reads, and on graded meshes 94 %
// of them read cells or ghosts that read cells (2D L4..12: 41 K and 40 K of
// 87 K ghosts at depth 1 and 2, the deepest at 10).  So every ghost is written
// exactly once, by a lane that waits for its own sources: k_ghost_reset stores
// a mark in every ghost the update writes, then k_ghost_flow computes all of
// them in one grid, each lane loading its sources again while one still holds
// the mark.  The values travel through 8-byte agent-scope stores and loads, so
// a source is seen either as the mark or as its final value: no flags, no
// fences, no barriers.
//
// Bound: latency, launch + index chain + one store-to-load trip per depth.
// The stages were bound by their launches (3 to 4 us each) and, for the small
// ones, by a block barrier and a chain of five dependent loads per stage.
// update_ghost_mr + upwind, one step: 2D L4..12 (158 K cells) 27 us against 90
// with a launch per stage, 3D L2..8 (234 K cells) 36 against 96, 2D L2..7
// (5.9 K cells) 19 against 26.
//
// Every wait ends.  Blocks take their place in the order of the ghosts from a
// counter (the ticket), and the order keeps every source before its readers
// where the cells tile the box (the other meshes keep the staged launches), so
// the lowest unfinished wave waits for nothing that is not done; and a wave
// gives up after FlowWait::rounds looks and uses what it has read (the right
// value when a cell itself holds the bits of the mark; otherwise the fault words
// say so).
#include "flow_ops.hpp"

namespace smr::dev
{
    namespace
    {
        // projection_op_ (op_project_at) on waited-for sources
        template <int DIM>
        __device__ __forceinline__ bool flow_project(const List& l, int64_t c, bool active, double* u, const FlowWait& w)
        {
            constexpr int NR     = 1 << (DIM - 1);
            constexpr double inv = 1.0 / double(1 << DIM);
            double* dst          = nullptr;
            const double* row[NR];
            if (active)
            {
                const Cell cell  = locate(l, c);
                const int64_t* b = bases(l, cell.run);
                dst              = u + b[0] + cell.x;
#pragma unroll
                for (int r = 0; r < NR; ++r)
                {
                    row[r] = u + b[1 + r] + 2 * cell.x;
                }
            }
            auto at = [&](int k) { return row[k >> 1] + (k & 1); };
            Sources<2 * NR, decltype(at)> s;
            auto attempt = [&](bool last)
            {
                if (!s.ready(at) && !last)
                {
                    return false;
                }
                double sum = 0;
#pragma unroll
                for (int r = 0; r < NR; ++r)
                {
                    sum += s.v[2 * r] + s.v[2 * r + 1];
                }
                publish(dst, sum * inv);
                return true;
            };
            return until_done(active, w, attempt);
        }

        // prediction_op <s,false> (op_predict_fine_at) on waited-for sources
        template <int DIM, int S>
        __device__ __forceinline__ bool flow_predict(const List& l, int64_t c, bool active, double* u, const FlowWait& w)
        {
            constexpr int NY = 2 * S + 1, NZ = DIM == 3 ? NY : 1, N = NZ * NY * NY;
            double* dst = nullptr;
            const double* row[NZ * NY];
            int px = 0, py = 0, pz = 0;
            if (active)
            {
                const Cell cell  = locate(l, c);
                const int64_t* b = bases(l, cell.run);
                dst              = u + b[0] + cell.x;
                px               = cell.x & 1;
                py               = cell.y & 1;
                pz               = cell.z & 1;
#pragma unroll
                for (int r = 0; r < NZ * NY; ++r)
                {
                    row[r] = u + b[1 + r] + (cell.x >> 1) - S;
                }
            }
            auto at = [&](int k) { return row[k / NY] + k % NY; };
            Sources<N, decltype(at)> s;
            auto attempt = [&](bool last)
            {
                if (!s.ready(at) && !last)
                {
                    return false;
                }
                double v;
                if constexpr (S == 0)
                {
                    v = s.v[0];
                }
                else
                {
                    v = 0;
#pragma unroll
                    for (int rz = 0; rz < NZ; ++rz)
                    {
#pragma unroll
                        for (int ry = 0; ry < 3; ++ry)
                        {
#pragma unroll
                            for (int sx = 0; sx < 3; ++sx)
                            {
                                const double f = s.v[(rz * 3 + ry) * 3 + sx];
                                double coeff   = 1.;
                                coeff *= pcoef(px, sx);
                                coeff *= pcoef(py, ry);
                                if constexpr (DIM == 3)
                                {
                                    coeff *= pcoef(pz, rz);
                                }
                                v += f * coeff;
                            }
                        }
                    }
                }
                publish(dst, v);
                return true;
            };
            return until_done(active, w, attempt);
        }

        // the item of wave w: the last one whose first wave is at most w
        // (at most 64 items, one per lane)
        __device__ __forceinline__ int item_of(const GhostFlow& f, int w)
        {
            const int lane   = int(threadIdx.x & 63);
            const bool ok    = lane < f.nitems && f.wave0[lane] <= w;
            const uint64_t m = __ballot(ok);
            return __builtin_amdgcn_readfirstlane(63 - __clzll(m));
        }

        // stores the mark in the ghosts of wave w of the update
        __device__ __forceinline__ void reset_wave(const GhostFlow& f, int w, double* u)
        {
            const int k     = item_of(f, w);
            const int64_t c = int64_t(f.c0[k]) + int64_t(w - f.wave0[k]) * 64 + int(threadIdx.x & 63);
            if (c >= f.c1[k])
            {
                return;
            }
            int64_t dst;
            if (f.op[k] == SEQ_RECIPES)
            {
                dst = f.rec[4 * c];
            }
            else
            {
                const List& l   = f.op[k] == SEQ_PROJECT ? f.proj : f.pred;
                const int64_t r = l.cellrun[c];
                dst             = l.base[r * l.ntaps] + l.iv[5 * r] + (c - l.pref[r]);
            }
            u[dst] = __longlong_as_double((long long)kMark);
        }

        __device__ __forceinline__ bool in_list(const List& l, int64_t slot)
        {
            for (int64_t r = 0; r < l.nruns; ++r)
            {
                const int64_t x = slot - l.base[r * l.ntaps];
                if (x >= l.iv[5 * r] && x < l.iv[5 * r + 1])
                {
                    return true;
                }
            }
            return false;
        }

        // whether slot holds the mark and the update does not write it
        __device__ __forceinline__ bool marked_input(const GhostFlow& f, const double* u, int64_t slot)
        {
            if (!marked(look_again(u + slot)) || in_list(f.proj, slot) || in_list(f.pred, slot))
            {
                return false;
            }
            for (int k = 0; k < f.nitems; ++k)
            {
                for (int32_t c = f.op[k] == SEQ_RECIPES ? f.c0[k] : f.c1[k]; c < f.c1[k]; ++c)
                {
                    if (f.rec[4 * int64_t(c)] == slot)
                    {
                        return false;
                    }
                }
            }
            return true;
        }

        // a wave that gave up, on ghost c of item k: a fault, unless some wave
        // waited for an input that holds the mark
        template <int DIM, int S>
        __device__ __forceinline__ void gave_up(const GhostFlow& f, int k, int64_t c, bool active, const double* u, const FlowWait& w)
        {
            report_fault(w, FAULT_GHOSTS);
            if (!active)
            {
                return;
            }
            // the sources are located anew, so that the wait holds no registers
            // for this (kept from before it: 126 -> 166 in 3D)
            asm volatile("" : "+v"(c));
            bool input = false;
            if (f.op[k] == SEQ_RECIPES)
            {
                const int4 r = reinterpret_cast<const int4*>(f.rec)[c];
                for (int q = 0; q < r.y >> 8; ++q)
                {
                    input = input || marked_input(f, u, q == 0 ? r.z : f.rsrc[r.w + q]);
                }
            }
            else
            {
                const bool fine    = f.op[k] == SEQ_PROJECT;
                const List& l      = fine ? f.proj : f.pred;
                const Cell cell    = locate(l, c);
                const int64_t* row = bases(l, cell.run);
                const int n        = fine ? 2 : 2 * S + 1;
                const int32_t x0   = fine ? 2 * cell.x : (cell.x >> 1) - S;
                for (int q = 0; q < n * (l.ntaps - 1); ++q)
                {
                    input = input || marked_input(f, u, row[1 + q / n] + x0 + q % n);
                }
            }
            if (input)
            {
                excuse_faults(w);
            }
        }

        // computes the ghosts of wave w
        template <int DIM, int S>
        __device__ __forceinline__ void flow_wave(const GhostFlow& f, int w, double* u, double bc, const FlowWait& fw)
        {
            const int k       = item_of(f, w);
            const int64_t c   = int64_t(f.c0[k]) + int64_t(w - f.wave0[k]) * 64 + int(threadIdx.x & 63);
            const bool active = c < f.c1[k];
            bool late;
            switch (f.op[k])
            {
                case SEQ_RECIPES: late = flow_recipe(f.rec, f.rsrc, c, active, u, bc, fw); break;
                case SEQ_PROJECT: late = flow_project<DIM>(f.proj, c, active, u, fw); break;
                default: late = flow_predict<DIM, S>(f.pred, c, active, u, fw); break;
            }
            if (late)
            {
                gave_up<DIM, S>(f, k, c, active, u, fw);
            }
        }

        // marks every ghost of the update and clears its ticket
        __global__ __launch_bounds__(256) void k_ghost_reset(GhostFlow f, double* u, int64_t nref)
        {
            if (blockIdx.x == 0 && threadIdx.x == 0)
            {
                *reinterpret_cast<unsigned*>(u + nref) = 0;
            }
            const int w = int(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
            if (w < f.nwaves)
            {
                reset_wave(f, w, u);
            }
        }

        // at most this many threads in a block (one ticket each)
        constexpr int FLOW_BLOCK = 512;

        template <int DIM, int S>
        __global__ __launch_bounds__(FLOW_BLOCK) void k_ghost_flow(GhostFlow f, double* u, int64_t nref, double bc, FlowWait fw)
        {
            __shared__ unsigned ticket;
            if (threadIdx.x == 0)
            {
                ticket = atomicAdd(reinterpret_cast<unsigned*>(u + nref), 1u);
            }
            __syncthreads();
            const int w = __builtin_amdgcn_readfirstlane(int(ticket * (blockDim.x >> 6) + (threadIdx.x >> 6)));
            if (w < f.nwaves)
            {
                flow_wave<DIM, S>(f, w, u, bc, fw);
            }
        }

        // ---- many fields per launch: the waves of one after the other ----

        // blocks of the batched launch: thousands of tickets, so the largest
        constexpr int BATCH_BLOCK = 1024;

        // the instance of wave w: the last one with pref[k] <= w, 64 looked at
        // per step
        __device__ __forceinline__ int instance_of(const int64_t* pref, int n, int64_t w)
        {
            const int lane = int(threadIdx.x & 63);
            int lo = 0; // pref[lo] <= w throughout
            while (n > 64)
            {
                const int step   = (n + 63) >> 6;
                const int k      = lo + lane * step;
                const uint64_t m = __ballot(k < lo + n && pref[k] <= w);
                const int next   = lo + (63 - __clzll(m)) * step;
                n                = min(step, lo + n - next);
                lo               = next;
            }
            const uint64_t m = __ballot(lane < n && pref[lo + lane] <= w);
            return __builtin_amdgcn_readfirstlane(lo + (63 - __clzll(m)));
        }

        __global__ __launch_bounds__(256) void k_ghost_reset_batch(const FlowInstance* inst, const int64_t* pref, int n, int64_t nwaves, unsigned* ticket)
        {
            if (blockIdx.x == 0 && threadIdx.x == 0)
            {
                *ticket = 0;
            }
            const int64_t w = int64_t(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
            if (w < nwaves)
            {
                const int k = instance_of(pref, n, w);
                reset_wave(inst[k].f, int(w - pref[k]), inst[k].u);
            }
        }

        template <int DIM, int S>
        __global__ __launch_bounds__(BATCH_BLOCK) void k_ghost_flow_batch(const FlowInstance* inst, const int64_t* pref, int n, int64_t nwaves,
                                                                          unsigned* ticket, FlowWait fw)
        {
            __shared__ unsigned t;
            if (threadIdx.x == 0)
            {
                t = atomicAdd(ticket, 1u);
            }
            __syncthreads();
            const int64_t w = int64_t(__builtin_amdgcn_readfirstlane(int(t))) * (BATCH_BLOCK / 64) + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
            if (w < nwaves)
            {
                const int k = instance_of(pref, n, w);
                flow_wave<DIM, S>(inst[k].f, int(w - pref[k]), inst[k].u, inst[k].bc, fw);
            }
        }
    } // namespace

    void ghost_flow(int dim, int ps, const GhostFlow& f, double* u, int64_t nref, double bc, const FlowWait& w, hipStream_t s)
    {
        if (f.nwaves <= 0)
        {
            return;
        }
        // blocks queue about 10 ns each for their tickets, and small grids
        // spread better in small blocks (update + upwind, 256 / 512 / 1024
        // threads: 170 waves 19.0 / 19.9 / 20.8 us, 1.4 K waves 27.6 / 26.8 /
        // 27.7, 3D 1.8 K waves 37.6 / 36.0 / 37.0)
        const unsigned W = f.nwaves <= 512 ? 4 : FLOW_BLOCK / 64;
        const dim3 g((unsigned(f.nwaves) + W - 1) / W), b(W * 64);
        hipLaunchKernelGGL(k_ghost_reset, dim3(unsigned((f.nwaves + 3) / 4)), dim3(256), 0, s, f, u, nref);
        if (dim == 2 && ps == 0)
        {
            hipLaunchKernelGGL((k_ghost_flow<2, 0>), g, b, 0, s, f, u, nref, bc, w);
        }
        else if (dim == 2)
        {
            hipLaunchKernelGGL((k_ghost_flow<2, 1>), g, b, 0, s, f, u, nref, bc, w);
        }
        else if (ps == 0)
        {
            hipLaunchKernelGGL((k_ghost_flow<3, 0>), g, b, 0, s, f, u, nref, bc, w);
        }
        else
        {
            hipLaunchKernelGGL((k_ghost_flow<3, 1>), g, b, 0, s, f, u, nref, bc, w);
        }
    }

    void ghost_flow_batch(int dim, int ps, const FlowInstance* inst, const int64_t* wpref, int n, int64_t nwaves, unsigned* ticket, const FlowWait& w,
                          hipStream_t s)
    {
        if (nwaves <= 0)
        {
            return;
        }
        constexpr int W = BATCH_BLOCK / 64;
        const dim3 g(unsigned((nwaves + W - 1) / W)), b(BATCH_BLOCK);
        hipLaunchKernelGGL(k_ghost_reset_batch, dim3(unsigned((nwaves + 3) / 4)), dim3(256), 0, s, inst, wpref, n, nwaves, ticket);
        if (dim == 2 && ps == 0)
        {
            hipLaunchKernelGGL((k_ghost_flow_batch<2, 0>), g, b, 0, s, inst, wpref, n, nwaves, ticket, w);
        }
        else if (dim == 2)
        {
            hipLaunchKernelGGL((k_ghost_flow_batch<2, 1>), g, b, 0, s, inst, wpref, n, nwaves, ticket, w);
        }
        else if (ps == 0)
        {
            hipLaunchKernelGGL((k_ghost_flow_batch<3, 0>), g, b, 0, s, inst, wpref, n, nwaves, ticket, w);
        }
        else
        {
            hipLaunchKernelGGL((k_ghost_flow_batch<3, 1>), g, b, 0, s, inst, wpref, n, nwaves, ticket, w);
        }
    }
} // namespace smr::dev
