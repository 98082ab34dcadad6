// The maximum pass of the tags (mr/operators.hpp:22-96, per level from the
// finest down) as one dataflow launch: a coarse cell waits until none of its
// children is open, i.e. still has a pass of its own to come.
//
// k_tag_open opens every coarse cell of the list (a bit of its tag byte that
// no rule uses), k_tag_flow closes them, finest level first: blocks take their
// place from a counter, so the lowest unfinished wave waits for nothing that is
// not done, and a wave gives up waiting after FlowWait::rounds looks (which
// only a broken order would make it do: the fault words say so).  The tags
// travel through agent-scope byte loads and stores.
//
// Bound: latency, a store-to-load trip per level.  The staged form is a launch
// per level of more than 2048 coarse cells and one block for the others.
// 3D L2..8: 6.2 us after the opening, against three launches of 3.8 us and
// 8.0 for the block; 2D L4..12: about 13 us for both launches against seven
// of 3.7 us and 10.4 for the block.
#include "flow_ops.hpp"

namespace smr::dev
{
    namespace
    {
        constexpr int TB         = 256;
        constexpr unsigned kOpen = 0x80;

        __global__ __launch_bounds__(TB) void k_tag_open(List l, uint8_t* tag, unsigned* ticket)
        {
            const int64_t c = int64_t(blockIdx.x) * TB + threadIdx.x;
            if (c == 0)
            {
                *ticket = 0;
            }
            if (c < l.ncells)
            {
                const Cell cell = locate(l, c);
                uint8_t* t      = tag + bases(l, cell.run)[0] + cell.x;
                *t              = uint8_t(*t | kOpen);
            }
        }

        template <int DIM>
        __global__ __launch_bounds__(TB) void k_tag_flow(List l, uint8_t* tag, unsigned* ticket, FlowWait fw)
        {
            __shared__ unsigned place;
            if (threadIdx.x == 0)
            {
                place = atomicAdd(ticket, 1u);
            }
            __syncthreads();
            // the list holds the coarse levels in ascending order
            const int64_t c   = l.ncells - 1 - (int64_t(place) * TB + threadIdx.x);
            const bool active = c >= 0;
            constexpr int NR  = 1 << (DIM - 1);
            uint8_t* own      = nullptr;
            uint8_t* row[NR];
            unsigned v = 0;
            if (active)
            {
                const Cell cell  = locate(l, c);
                const int64_t* b = bases(l, cell.run);
                own              = tag + b[0] + cell.x;
                v                = *own & ~kOpen;
#pragma unroll
                for (int r = 0; r < NR; ++r)
                {
                    row[r] = tag + b[1 + r] + 2 * cell.x;
                }
            }
            auto attempt = [&](bool last)
            {
                unsigned t[2 * NR], any = 0, all = 2;
#pragma unroll
                for (int k = 0; k < 2 * NR; ++k)
                {
                    t[k] = __hip_atomic_load(row[k >> 1] + (k & 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    any |= t[k];
                    all &= t[k];
                }
                if ((any & kOpen) && !last)
                {
                    return false;
                }
                // a child that is kept keeps the others, and the
                // cell; the children go together or not at all
                const bool keep = any & 1;
#pragma unroll
                for (int k = 0; k < 2 * NR; ++k)
                {
                    const unsigned w = keep ? t[k] | 1u : (all ? t[k] : t[k] & ~2u);
                    if (w != t[k])
                    {
                        __hip_atomic_store(row[k >> 1] + (k & 1), uint8_t(w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
                __hip_atomic_store(own, uint8_t(keep || all ? v | 1u : v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return true;
            };
            const bool late = until_done(active, fw, attempt);
            if (late)
            {
                report_fault(fw, FAULT_TAGS);
            }
        }
    } // namespace

    void tag_flow(int dim, const List& l, uint8_t* tag, unsigned* ticket, const FlowWait& w, hipStream_t s)
    {
        if (l.ncells <= 0)
        {
            return;
        }
        const dim3 g(unsigned((l.ncells + TB - 1) / TB)), b(TB);
        hipLaunchKernelGGL(k_tag_open, g, b, 0, s, l, tag, ticket);
        if (dim == 2)
        {
            hipLaunchKernelGGL(k_tag_flow<2>, g, b, 0, s, l, tag, ticket, w);
        }
        else
        {
            hipLaunchKernelGGL(k_tag_flow<3>, g, b, 0, s, l, tag, ticket, w);
        }
    }
} // namespace smr::dev
