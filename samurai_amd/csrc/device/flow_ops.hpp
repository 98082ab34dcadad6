// Waiting for values inside a launch: a slot that the launch will write holds
// a mark until its value arrives, and a lane that reads it looks again while
// it sees the mark (ghost_flow.hip, adjoint_flow.hip).
//
// The values travel through 8-byte agent-scope stores and loads, so a source
// is seen either as the mark or as its final value: no flags and no fences.
// Every wait ends: the launches hand out their work in an order in which every
// source precedes its readers (the lowest unfinished wave waits for nothing
// that is not done), and a wave gives up after FlowWait::rounds looks and uses
// what it has read.  That is right where a value the launch only reads holds
// the bits of the mark; otherwise the order was broken, and the context's fault
// words say so.
#pragma once

#include "cell_ops.hpp"

namespace smr::dev
{
    // a signalling NaN: arithmetic results are never signalling, and a
    // copied value with these very bits is stored quiet
    constexpr unsigned long long kMark = 0x7FF05A3C96E1D2B4ull;
    constexpr unsigned long long kQuiet = 0x0008000000000000ull;

    __device__ __forceinline__ bool marked(double v)
    {
        return (unsigned long long)__double_as_longlong(v) == kMark;
    }

    // the first look at a source: any cache may answer, since a line that
    // is out of date holds the mark
    __device__ __forceinline__ double look(const double* p)
    {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    __device__ __forceinline__ double look_again(const double* p)
    {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    __device__ __forceinline__ void publish(double* p, double v)
    {
        if (marked(v))
        {
            v = __longlong_as_double((long long)(kMark | kQuiet));
        }
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // a wave has given up on a value that its launch writes
    __device__ __forceinline__ void report_fault(const FlowWait& w, int code)
    {
        __hip_atomic_store(w.fault, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }

    // a wave has waited for a value that holds the bits of the mark itself.  What
    // waits for that wave has given up about when it did, and has its NaN anyway
    __device__ __forceinline__ void excuse_faults(const FlowWait& w)
    {
        __hip_atomic_store(w.fault + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }

    // runs attempt(last) on the lanes not yet done until all of them are: it
    // returns true once the lane has published (always when last).  Whether the
    // wave gave up: known from the rounds alone, so that the wait keeps no
    // account of who missed what (with one per lane the adjoint steps took
    // 12.6 ms instead of 11.6).
    template <class F>
    __device__ __forceinline__ bool until_done(bool active, const FlowWait& w, F&& attempt)
    {
        bool done = !active;
        int spin  = 0;
        for (; !__all(done); ++spin)
        {
            if (!done)
            {
                done = attempt(spin >= w.rounds);
            }
        }
        return spin > w.rounds;
    }

    // N sources held in registers; true when none of them is marked
    template <int N, class Addr>
    struct Sources
    {
        double v[N];
        bool fresh = true;
        __device__ __forceinline__ bool ready(const Addr& at)
        {
            bool ok = true;
#pragma unroll
            for (int k = 0; k < N; ++k)
            {
                if (fresh)
                {
                    v[k] = look(at(k));
                }
                else if (marked(v[k]))
                {
                    v[k] = look_again(at(k));
                }
            }
#pragma unroll
            for (int k = 0; k < N; ++k)
            {
                ok = ok && !marked(v[k]);
            }
            fresh = false;
            return ok;
        }
    };

    // op_recipe on waited-for sources; (dst, op | n << 8, first source,
    // first of the n sources in src).  The sources are taken one after the
    // other as they come, in the recipe's order.
    __device__ __forceinline__ bool flow_recipe(const int32_t* __restrict__ rec, const int32_t* __restrict__ src, int64_t c, bool active,
                                                double* u, double bc, const FlowWait& w)
    {
        int4 r{};
        if (active)
        {
            r = reinterpret_cast<const int4*>(rec)[c];
        }
        const int op = r.y & 255, n = r.y >> 8;
        double acc = 0;
        int k      = 0;
        bool first = true;
        auto attempt = [&](bool last)
        {
            for (; k < n; ++k)
            {
                const double* p = u + (k == 0 ? r.z : src[r.w + k]);
                double x        = first ? look(p) : look_again(p);
                if (marked(x) && first)
                {
                    x = look_again(p);
                }
                if (marked(x) && !last)
                {
                    first = false;
                    return false;
                }
                first = true;
                if (op == 0)
                {
                    acc = x;
                }
                else if (op == 1)
                {
                    acc = 2 * bc - x;
                }
                else if (op == 2)
                {
                    acc += x;
                }
                else if (k == 0)
                {
                    acc = x;
                }
                else if (n == 3)
                {
                    // u0 - u1 * 3 + u2 * 3
                    acc = k == 1 ? acc - x * 3.0 : acc + x * 3.0;
                }
                else
                {
                    // u0 - u1 * 5 + u2 * 10 - u3 * 10 + u4 * 5
                    const double w = x * (k == 1 || k == 4 ? 5.0 : 10.0);
                    acc            = (k & 1) ? acc - w : acc + w;
                }
            }
            if (op == 2 && n > 0)
            {
                acc /= n;
            }
            publish(u + r.x, acc);
            return true;
        };
        return until_done(active, w, attempt);
    }
} // namespace smr::dev
