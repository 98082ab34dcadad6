// Frozen-mesh time steps and their adjoint as dataflow launches.
//
// On a frozen mesh every value of every step is written once and its sources
// are known, so a whole checkpoint segment (`steps` time steps of all
// instances: ghosts, then the upwind update of the cells, step after step) is
// one launch over `steps` state arrays in which each lane waits for its own
// sources (flow_ops.hpp); the adjoint of the segment is another.  The
// operations are table driven: one record of storage slots per ghost and cell,
// over the concatenated storages of all instances, so a lane reaches its
// values with two dependent loads.
//
// The adjoint value of a slot is the transposed upwind stencil at a cell (or,
// at a ghost, the contributions of the cells beside it) plus, for every
// forward stage that reads the slot from the last one on, the weighted adjoint
// values of the ghosts that stage computes from it: the sums and their order
// are those of the staged adjoint (adjoint.hpp), whose results are the same
// bits.
//
// Bound: the latency of a wave's few loads times the waves per step (22 K for
// 851 K cells and their ghosts, 8 K of them resident at a time), 23 us per
// forward step; a launch per stage took 225 us, a checkpoint segment of 10
// steps forward and backward now 0.8 ms instead of 7.6.
#include "flow_ops.hpp"

namespace smr::dev
{
    namespace
    {
        // Threads of a block.  Blocks queue for their tickets, about 10 ns each:
        // 100 steps of 32 instances (851 K cells) and their adjoint took 19.5 ms
        // with blocks of 256, 12.3 with 512, 10.3 with 1024 and 9.4 with blocks
        // that take their own index instead (whose order the hardware does not
        // promise).  A ticket for several rounds of a block is slower (17 ms
        // for 2, 41 for 4): the later rounds hold up what follows them.
        constexpr int FB = 1024;

        // words of a projection, prediction and cell record
        constexpr int proj_words(int dim) { return dim == 2 ? 4 : 8; }
        constexpr int pred_words(int dim, int s) { return s == 0 ? 2 : (dim == 2 ? 4 : 12); }
        constexpr int cell_words(int dim) { return dim == 2 ? 4 : 8; }

        // the wave's place in the order of the work
        __device__ __forceinline__ int64_t take_wave(unsigned* ticket)
        {
            __shared__ unsigned t;
            if (threadIdx.x == 0)
            {
                t = atomicAdd(ticket, 1u);
            }
            __syncthreads();
            return int64_t(__builtin_amdgcn_readfirstlane(int(t))) * (FB / 64) + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
        }

        // array j of a segment: the first and the last one are kept apart
        __device__ __forceinline__ double* segment_array(const FlowArrays& a, int j, int64_t n)
        {
            return j == 0 ? a.first : (j == a.steps ? a.last : a.between + int64_t(j - 1) * n);
        }

        template <int DIM, int S>
        __device__ __forceinline__ bool ghost_project(const int32_t* __restrict__ tab, int64_t c, bool active, double* u, const FlowWait& w)
        {
            constexpr int NR     = 1 << (DIM - 1);
            constexpr double inv = 1.0 / double(1 << DIM);
            int32_t r[1 + NR]    = {};
            if (active)
            {
#pragma unroll
                for (int k = 0; k < 1 + NR; ++k)
                {
                    r[k] = tab[proj_words(DIM) * c + k];
                }
            }
            auto at = [&](int k) { return u + r[1 + (k >> 1)] + (k & 1); };
            Sources<2 * NR, decltype(at)> s;
            auto attempt = [&](bool last)
            {
                if (!s.ready(at) && !last)
                {
                    return false;
                }
                double sum = 0;
#pragma unroll
                for (int q = 0; q < NR; ++q)
                {
                    sum += s.v[2 * q] + s.v[2 * q + 1];
                }
                publish(u + r[0], sum * inv);
                return true;
            };
            return until_done(active, w, attempt);
        }

        template <int DIM, int S>
        __device__ __forceinline__ bool ghost_predict(const int32_t* __restrict__ tab, int64_t c, bool active, double* u, const FlowWait& w)
        {
            constexpr int NY = 2 * S + 1, NZ = DIM == 3 ? NY : 1;
            int32_t r[1 + NZ * NY] = {};
            if (active)
            {
#pragma unroll
                for (int k = 0; k < 1 + NZ * NY; ++k)
                {
                    r[k] = tab[pred_words(DIM, S) * c + k];
                }
            }
            auto at = [&](int k) { return u + r[1 + k / NY] + k % NY; };
            Sources<NZ * NY * NY, decltype(at)> s;
            auto attempt = [&](bool last)
            {
                if (!s.ready(at) && !last)
                {
                    return false;
                }
                double v = s.v[0];
                if constexpr (S == 1)
                {
                    const int px = (r[0] >> 28) & 1, py = (r[0] >> 29) & 1, pz = (r[0] >> 30) & 1;
                    v            = 0;
#pragma unroll
                    for (int k = 0; k < NZ * 9; ++k)
                    {
                        double coeff = 1.;
                        coeff *= pcoef(px, k % 3);
                        coeff *= pcoef(py, (k / 3) % 3);
                        if constexpr (DIM == 3)
                        {
                            coeff *= pcoef(pz, k / 9);
                        }
                        v += s.v[k] * coeff;
                    }
                }
                publish(u + (r[0] & kFlowSlotMask), v);
                return true;
            };
            return until_done(active, w, attempt);
        }

        // cell record: own slot, the rows below and above (2D) and in front
        // and behind (3D) at this x, then level | ghost neighbours << 5 |
        // instance << 11
        template <int DIM>
        struct CellRec
        {
            int32_t own, row[2 * DIM - 2], word;
            __device__ __forceinline__ void load(const int32_t* __restrict__ tab, int64_t c)
            {
                if constexpr (DIM == 2)
                {
                    const int4 v = reinterpret_cast<const int4*>(tab)[c];
                    own          = v.x;
                    row[0]       = v.y;
                    row[1]       = v.z;
                    word         = v.w;
                }
                else
                {
                    const int4 v = reinterpret_cast<const int4*>(tab)[2 * c], q = reinterpret_cast<const int4*>(tab)[2 * c + 1];
                    own    = v.x;
                    row[0] = v.y;
                    row[1] = v.z;
                    row[2] = v.w;
                    row[3] = q.x;
                    word   = q.y;
                }
            }
            // neighbour d: x - 1, x + 1, y - 1, y + 1, z - 1, z + 1
            __device__ __forceinline__ int32_t neighbour(int d) const { return d < 2 ? own + 2 * d - 1 : row[d - 2]; }
            __device__ __forceinline__ bool ghost(int d) const { return (word >> (5 + d)) & 1; }
            __device__ __forceinline__ int level() const { return word & 31; }
            __device__ __forceinline__ int instance() const { return word >> 11; }
        };

        template <int DIM>
        __device__ __forceinline__ bool cell_upwind(const AdjointFlow& f, int64_t c, bool active, const double* u, double* out, const FlowWait& w)
        {
            CellRec<DIM> r{};
            FlowParam p{};
            if (active)
            {
                r.load(f.cell, c);
                p = f.par[r.instance()];
            }
            auto at = [&](int k) { return u + (k == 0 ? r.own : r.neighbour(k - 1)); };
            Sources<2 * DIM + 1, decltype(at)> s;
            auto attempt = [&](bool last)
            {
                if (!s.ready(at) && !last)
                {
                    return false;
                }
                const double uc = s.v[0];
                const double FL = flux_h(.5 * p.a[0], .5 * fabs(p.a[0]), s.v[1], uc);
                const double FR = flux_h(.5 * p.a[0], .5 * fabs(p.a[0]), uc, s.v[2]);
                const double FD = flux_h(.5 * p.a[1], .5 * fabs(p.a[1]), s.v[3], uc);
                const double FU = flux_h(.5 * p.a[1], .5 * fabs(p.a[1]), uc, s.v[4]);
                double S;
                if constexpr (DIM == 2)
                {
                    S = -FL + FR + -FD + FU;
                }
                else
                {
                    const double FF = flux_h(.5 * p.a[2], .5 * fabs(p.a[2]), s.v[2 * DIM - 1], uc);
                    const double FB = flux_h(.5 * p.a[2], .5 * fabs(p.a[2]), uc, s.v[2 * DIM]);
                    S               = -FL + FR + -FD + FU + -FF + FB;
                }
                publish(out + r.own, uc - p.dt * (S * double(1 << r.level())));
                return true;
            };
            return until_done(active, w, attempt);
        }

        // a.steps time steps: the ghosts of each state, then the next state's
        // cells (not the last one's without `last`)
        template <int DIM, int S>
        __global__ __launch_bounds__(FB) void k_adj_forward(AdjointFlow f, FlowArrays a, int last, unsigned* ticket, FlowWait fw)
        {
            const int64_t g = take_wave(ticket);
            const int j     = int(g / f.nwaves);
            if (j >= a.steps)
            {
                return;
            }
            const int w      = int(g - int64_t(j) * f.nwaves);
            const int lane   = int(threadIdx.x & 63);
            const bool ok    = lane < f.nitems && f.wave0[lane] <= w;
            const uint64_t m = __ballot(ok);
            const int k      = __builtin_amdgcn_readfirstlane(63 - __clzll(m));
            const int64_t c  = int64_t(f.c0[k]) + int64_t(w - f.wave0[k]) * 64 + lane;
            const bool act   = c < f.c1[k];
            double* u        = segment_array(a, j, f.n);
            bool late        = false;
            switch (f.op[k])
            {
                case FLOW_RECIPES:
                {
                    double bc = 0;
                    if (act)
                    {
                        const int4 r = reinterpret_cast<const int4*>(f.rec)[c];
                        bc           = (r.y & 255) == 1 ? f.par[r.w].bc : 0.0;
                    }
                    late = flow_recipe(f.rec, f.rsrc, c, act, u, bc, fw);
                    break;
                }
                case FLOW_PROJECT: late = ghost_project<DIM, S>(f.proj, c, act, u, fw); break;
                case FLOW_PREDICT: late = ghost_predict<DIM, S>(f.pred, c, act, u, fw); break;
                default:
                    if (j + 1 < a.steps || last)
                    {
                        late = cell_upwind<DIM>(f, c, act, u, segment_array(a, j + 1, f.n), fw);
                    }
                    break;
            }
            if (late)
            {
                report_fault(fw, FAULT_ADJOINT);
            }
        }

        // m += the contributions of the forward stages that read the slot of
        // operation q, from entry k on; false while one is awaited
        struct Gather
        {
            int32_t k, end;
            double group = 0;
            __device__ __forceinline__ bool run(const AdjointFlow& f, const double* mu, double& m, bool last)
            {
                for (; k < end; ++k)
                {
                    const int32_t e = f.esrc[k];
                    const double* p = mu + (e & kFlowSlotMask);
                    double x        = look(p);
                    if (marked(x))
                    {
                        x = look_again(p);
                        if (marked(x) && !last)
                        {
                            return false;
                        }
                    }
                    group += f.ew[k] * x;
                    if (e < 0)
                    {
                        m += group;
                        group = 0;
                    }
                }
                return true;
            }
        };

        // a.steps adjoint steps: per step the ghosts' adjoint values, then the
        // cells' of the step before
        template <int DIM>
        __global__ __launch_bounds__(FB) void k_adj_backward(AdjointFlow f, FlowArrays a, unsigned* ticket, FlowWait fw)
        {
            const int64_t g   = take_wave(ticket);
            const int64_t nwg = (f.naghost + 63) / 64, nw = nwg + (f.ncells + 63) / 64;
            const int j       = int(g / nw);
            if (j >= a.steps)
            {
                return;
            }
            const int64_t w = g - int64_t(j) * nw;
            const int lane  = int(threadIdx.x & 63);
            double* lam     = segment_array(a, j, f.n);
            if (w < nwg)
            {
                // the cells whose neighbour in direction d this ghost is
                const int64_t q = w * 64 + lane;
                const bool act  = q < f.naghost;
                int32_t dst = 0, cells[6] = {-1, -1, -1, -1, -1, -1};
                FlowParam p{};
                double kk = 0, m = 0;
                Gather in{0, 0};
                if (act)
                {
                    const int4 r0 = reinterpret_cast<const int4*>(f.aghost)[2 * q], r1 = reinterpret_cast<const int4*>(f.aghost)[2 * q + 1];
                    dst      = r0.x;
                    cells[0] = r0.z;
                    cells[1] = r0.w;
                    cells[2] = r1.x;
                    cells[3] = r1.y;
                    cells[4] = r1.z;
                    cells[5] = r1.w;
                    p        = f.par[r0.y >> 5];
                    kk       = p.dt * ldexp(1.0, r0.y & 31);
                    in.k     = f.rowptr[q];
                    in.end   = f.rowptr[q + 1];
                }
                int d = 0;
                auto attempt = [&](bool last)
                {
#pragma unroll
                    for (int e = 0; e < 2 * DIM; ++e)
                    {
                        if (e == d)
                        {
                            if (cells[e] >= 0)
                            {
                                double x = look(lam + cells[e]);
                                if (marked(x))
                                {
                                    x = look_again(lam + cells[e]);
                                    if (marked(x) && !last)
                                    {
                                        return false;
                                    }
                                }
                                const double aa = p.a[e >> 1];
                                m += (e & 1) ? -kk * fmin(aa, 0.0) * x : kk * fmax(aa, 0.0) * x;
                            }
                            ++d;
                        }
                    }
                    if (!in.run(f, lam, m, last))
                    {
                        return false;
                    }
                    publish(lam + dst, m);
                    return true;
                };
                const bool late = until_done(act, fw, attempt);
                if (late)
                {
                    report_fault(fw, FAULT_ADJOINT);
                }
                return;
            }
            const int64_t c = (w - nwg) * 64 + lane;
            const bool act  = c < f.ncells;
            CellRec<DIM> r{};
            FlowParam p{};
            Gather in{0, 0};
            if (act)
            {
                r.load(f.cell, c);
                p      = f.par[r.instance()];
                in.k   = f.rowptr[f.naghost + c];
                in.end = f.rowptr[f.naghost + c + 1];
            }
            double* out = segment_array(a, j + 1, f.n);
            // lam of a ghost neighbour is zero (its slot holds the ghost's
            // adjoint value): the cell's own value stands in for the wait
            auto at = [&](int k) { return lam + (k == 0 || r.ghost(k - 1) ? r.own : r.neighbour(k - 1)); };
            Sources<2 * DIM + 1, decltype(at)> s;
            bool begun = false;
            double m   = 0;
            auto attempt = [&](bool last)
            {
                if (!begun)
                {
                    if (!s.ready(at) && !last)
                    {
                        return false;
                    }
                    const double k = p.dt * ldexp(1.0, r.level());
                    double v[2 * DIM];
#pragma unroll
                    for (int d = 0; d < 2 * DIM; ++d)
                    {
                        v[d] = r.ghost(d) ? 0.0 : s.v[1 + d];
                    }
                    double self = fabs(p.a[0]) + fabs(p.a[1]);
                    if constexpr (DIM == 3)
                    {
                        self += fabs(p.a[2]);
                    }
                    m = (1.0 - k * self) * s.v[0];
#pragma unroll
                    for (int d = 0; d < DIM; ++d)
                    {
                        m += k * fmax(p.a[d], 0.0) * v[2 * d + 1] - k * fmin(p.a[d], 0.0) * v[2 * d];
                    }
                    begun = true;
                }
                if (!in.run(f, lam, m, last))
                {
                    return false;
                }
                publish(out + r.own, m);
                return true;
            };
            const bool late = until_done(act, fw, attempt);
            if (late)
            {
                report_fault(fw, FAULT_ADJOINT);
            }
        }

        // the velocity-gradient terms of a.steps adjoint steps (all values in
        // place): step j pairs adjoint array j with state s.steps - 1 - j
        template <int DIM>
        __global__ __launch_bounds__(256) void k_adj_velocity(AdjointFlow f, FlowArrays lam, FlowArrays st, int st0, double* ga)
        {
            const int64_t c = int64_t(blockIdx.x) * 256 + threadIdx.x;
            if (c >= f.ncells)
            {
                return;
            }
            CellRec<DIM> r;
            r.load(f.cell, c);
            const FlowParam p = f.par[r.instance()];
            const double k    = p.dt * ldexp(1.0, r.level());
            double acc[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d)
            {
                acc[d] = ga[DIM * c + d];
            }
            for (int j = 0; j < lam.steps; ++j)
            {
                const double li  = segment_array(lam, j, f.n)[r.own];
                const double* un = segment_array(st, st0 - j, f.n);
                const double uc  = un[r.own];
#pragma unroll
                for (int d = 0; d < DIM; ++d)
                {
                    acc[d] += -k * li * (dflux_da(p.a[d], uc, un[r.neighbour(2 * d + 1)]) - dflux_da(p.a[d], un[r.neighbour(2 * d)], uc));
                }
            }
#pragma unroll
            for (int d = 0; d < DIM; ++d)
            {
                ga[DIM * c + d] = acc[d];
            }
        }

        // marks: every slot the launch writes (kind 1 cell, 2 ghost) of the
        // arrays between, the ghosts of the first; the other slots of the
        // arrays between are zero
        __global__ __launch_bounds__(256) void k_adj_marks(const uint8_t* __restrict__ kind, FlowArrays a, int64_t n, unsigned* ticket)
        {
            if (blockIdx.x == 0 && threadIdx.x == 0)
            {
                *ticket = 0;
            }
            const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
            if (i >= n)
            {
                return;
            }
            const uint8_t q   = kind[i];
            const double mark = __longlong_as_double((long long)kMark);
            if (q == 2)
            {
                a.first[i] = mark;
            }
            for (int j = 1; j < a.steps; ++j)
            {
                a.between[int64_t(j - 1) * n + i] = q ? mark : 0.0;
            }
        }

        // compact cell vectors: to = 1 from the array, 0 into it (stored quiet, so
        // that no cell of an array holds the bits of the mark)
        __global__ __launch_bounds__(256) void k_adj_cells(const int32_t* __restrict__ cell, int words, int64_t ncells, double* array, double* compact,
                                                           int to)
        {
            const int64_t c = int64_t(blockIdx.x) * 256 + threadIdx.x;
            if (c >= ncells)
            {
                return;
            }
            double* p = array + cell[words * c];
            if (to)
            {
                compact[c] = *p;
            }
            else
            {
                publish(p, compact[c]);
            }
        }

        unsigned blocks_of(int64_t n, int block)
        {
            return unsigned((n + block - 1) / block);
        }
    } // namespace

    void adjoint_flow_cells(const AdjointFlow& f, double* array, double* compact, bool to_compact, hipStream_t s)
    {
        if (f.ncells > 0)
        {
            hipLaunchKernelGGL(k_adj_cells, dim3(blocks_of(f.ncells, 256)), dim3(256), 0, s, f.cell, cell_words(f.dim), f.ncells, array, compact,
                               to_compact ? 1 : 0);
        }
    }

    void adjoint_flow_forward(const AdjointFlow& f, const FlowArrays& a, bool last, unsigned* ticket, const FlowWait& w, hipStream_t s)
    {
        if (f.ncells <= 0)
        {
            return;
        }
        hipLaunchKernelGGL(k_adj_marks, dim3(blocks_of(f.n, 256)), dim3(256), 0, s, f.kind, a, f.n, ticket);
        const dim3 g(blocks_of(int64_t(f.nwaves) * a.steps, FB / 64)), b(FB);
        if (f.dim == 2 && f.ps == 0)
        {
            hipLaunchKernelGGL((k_adj_forward<2, 0>), g, b, 0, s, f, a, int(last), ticket, w);
        }
        else if (f.dim == 2)
        {
            hipLaunchKernelGGL((k_adj_forward<2, 1>), g, b, 0, s, f, a, int(last), ticket, w);
        }
        else if (f.ps == 0)
        {
            hipLaunchKernelGGL((k_adj_forward<3, 0>), g, b, 0, s, f, a, int(last), ticket, w);
        }
        else
        {
            hipLaunchKernelGGL((k_adj_forward<3, 1>), g, b, 0, s, f, a, int(last), ticket, w);
        }
    }

    void adjoint_flow_backward(const AdjointFlow& f, const FlowArrays& a, unsigned* ticket, const FlowWait& w, hipStream_t s)
    {
        if (f.ncells <= 0)
        {
            return;
        }
        hipLaunchKernelGGL(k_adj_marks, dim3(blocks_of(f.n, 256)), dim3(256), 0, s, f.kind, a, f.n, ticket);
        const int64_t nw = (f.naghost + 63) / 64 + (f.ncells + 63) / 64;
        const dim3 g(blocks_of(nw * a.steps, FB / 64)), b(FB);
        if (f.dim == 2)
        {
            hipLaunchKernelGGL(k_adj_backward<2>, g, b, 0, s, f, a, ticket, w);
        }
        else
        {
            hipLaunchKernelGGL(k_adj_backward<3>, g, b, 0, s, f, a, ticket, w);
        }
    }

    void adjoint_flow_velocity(const AdjointFlow& f, const FlowArrays& lam, const FlowArrays& st, int st0, double* ga, hipStream_t s)
    {
        if (f.ncells <= 0)
        {
            return;
        }
        const dim3 g(blocks_of(f.ncells, 256)), b(256);
        if (f.dim == 2)
        {
            hipLaunchKernelGGL(k_adj_velocity<2>, g, b, 0, s, f, lam, st, st0, ga);
        }
        else
        {
            hipLaunchKernelGGL(k_adj_velocity<3>, g, b, 0, s, f, lam, st, st0, ga);
        }
    }
} // namespace smr::dev
