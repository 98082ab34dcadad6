// The flux-based convection operators on the cells of a mesh: a kernel that
// knows, per cell and side, what lies across the face, and adds the cell's
// interface terms in the reference's order.
//
// Across a face of a cell of level l lies a cell of the same level, a coarser
// cell, finer cells, or the boundary.  Except for finer cells, the interface's
// stencil is the cell and the slot beside it at level l (a cell or a ghost),
// and the factor the same: only the order of the terms depends on the kind.
// Finer cells bring 2^(dim-1) interfaces between slots of level l + 1, which a
// small table holds.  So a cell costs its run, a word of side kinds and the
// values; the order of the terms per direction d is (host/convection.cpp):
//   1. faces to cells of the same level (linear operator along x: right face
//      first; otherwise left face first, the order of the interfaces),
//   2. left, then right face to a coarser cell,
//   3. right, then left face to finer cells,
//   4. right, then left boundary face.
//
// Bound: latency of about four dependent loads, as the upwind step: the words of
// the fine sides are loaded together, then the values of a direction.  The
// ordered per-cell term lists this replaces cost 24 B per term to read and
// were built on the host (14.5 ms for 141 K cells of a 2D L4..12 mesh).  Whole
// calls on small meshes of prediction radius 0 (term lists / one fine face after
// the other and the output cleared by a launch of its own / as below): 2D L2..6
// 17.4 / 18.5 / 16.0 us, 3D L2..4 19.2 / 22.5 / 17.9 (Burgers) and 53.1 / 61.9 /
// 51.2 (velocity field, four ghost updates).
#include "cell_ops.hpp"

namespace smr::dev
{
    namespace
    {
        constexpr int CB = 256;

        enum Side : int
        {
            SIDE_SAME   = 0,
            SIDE_COARSE = 1,
            SIDE_FINE   = 2,
            SIDE_BOUNDARY = 3,
            SIDE_NONE   = 4 // no interface (a jump of more than one level)
        };

        __device__ __forceinline__ int side_of(int32_t word, int s) { return (word >> (3 * s)) & 7; }

        // slot of cell (level, x .. x + span - 1, y, z) at x, all in one run;
        // -1 if absent.  `row` is the row of the last hit: the next row of a
        // stencil is mostly the one after it
        __device__ __forceinline__ int64_t slot_of(const Table& t, int level, int32_t x, int32_t y, int32_t z, int span, int64_t& row)
        {
            if (level < 0 || level > 20)
            {
                return -1;
            }
            const int64_t key = row_key(y, z), first = t.row_off[level], end = t.row_off[level + 1];
            int64_t r = row + 1;
            if (row < first || r >= end || t.row_key[r] != key)
            {
                int64_t lo = first, hi = end;
                while (lo < hi)
                {
                    const int64_t mid = (lo + hi) >> 1;
                    if (t.row_key[mid] < key)
                    {
                        lo = mid + 1;
                    }
                    else
                    {
                        hi = mid;
                    }
                }
                r = lo;
                if (r >= end || t.row_key[r] != key)
                {
                    return -1;
                }
            }
            row       = r;
            int64_t a = t.rp[r], b = t.rp[r + 1];
            const int64_t k0 = a;
            while (a < b)
            {
                const int64_t mid = (a + b) >> 1;
                if (t.run_s[mid] <= x)
                {
                    a = mid + 1;
                }
                else
                {
                    b = mid;
                }
            }
            const int64_t k = a - 1;
            return k >= k0 && x + span <= t.run_e[k] ? t.run_idx[k] + x : -1;
        }

        // leaf[slot] = 1 for the cells and past the nref slots (0 beforehand)
        __global__ __launch_bounds__(CB) void k_leaf_flags(List l, uint8_t* leaf, int64_t nref)
        {
            const int64_t c = int64_t(blockIdx.x) * CB + threadIdx.x;
            if (c < conv_leaf_bytes(nref) - nref)
            {
                leaf[nref + c] = 1;
            }
            if (c < l.ncells)
            {
                const Cell cell = locate(l, c);
                leaf[bases(l, cell.run)[0] + cell.x] = 1;
            }
        }

        // side kinds of every cell, and the slots across its faces to finer
        // cells: fine_at[c] is the first of the cell's entries in fine, per
        // such side (in the order of the sides) one slot per face along x (the
        // slot inside the cell's face, its neighbour in x being the other
        // one), two along y and z (inside, outside) per pair of faces in x;
        // -1 where no interface is
        template <int DIM>
        __global__ __launch_bounds__(CB) void k_side_kinds(List l, Table t, const uint8_t* __restrict__ leaf, int32_t* word, int32_t* fine_at,
                                                           int32_t* fine, unsigned long long* used, int64_t room, int* fault)
        {
            constexpr int NF = 1 << (DIM - 1); // entries of a side
            const int64_t c   = int64_t(blockIdx.x) * CB + threadIdx.x;
            const bool active = c < l.ncells;
            int32_t w = 0, n = 0;
            bool fail = false;
            int32_t slots[2 * DIM * NF];
            if (active)
            {
                const Cell cell  = locate(l, c);
                const int64_t* b = bases(l, cell.run);
                const int side   = 1 << cell.level;
                const int32_t p[3] = {cell.x, cell.y, cell.z};
                for (int s = 0; s < 2 * DIM; ++s)
                {
                    const int d = s >> 1, up = s & 1;
                    int kind = SIDE_NONE;
                    if (p[d] == (up ? side - 1 : 0))
                    {
                        kind = SIDE_BOUNDARY;
                    }
                    else if (leaf[d == 0 ? b[0] + cell.x + 2 * up - 1 : b[s - 1] + cell.x])
                    {
                        kind = SIDE_SAME;
                    }
                    else
                    {
                        int64_t row = -2;
                        int32_t q[3] = {p[0], p[1], p[2]};
                        q[d] += 2 * up - 1;
                        const int64_t k = slot_of(t, cell.level - 1, q[0] >> 1, q[1] >> 1, q[2] >> 1, 1, row);
                        if (k >= 0 && leaf[k])
                        {
                            kind = SIDE_COARSE;
                        }
                        else
                        {
                            // the children at the face (inside) and their neighbours across it
                            bool any = false;
                            int32_t e[NF];
                            const int lf = cell.level + 1;
                            row          = -2;
                            if (d == 0)
                            {
#pragma unroll
                                for (int f = 0; f < NF; ++f)
                                {
                                    const int32_t xi = 2 * p[0] + up;
                                    const int64_t k0 = slot_of(t, lf, xi - 1 + up, 2 * p[1] + (f & 1), 2 * p[2] + (f >> 1), 2, row);
                                    const int64_t in = k0 + 1 - up, out = k0 + up;
                                    const bool ok    = k0 >= 0 && leaf[out];
                                    e[f]             = ok ? int32_t(in) : -1;
                                    any              = any || ok;
                                }
                            }
                            else
                            {
#pragma unroll
                                for (int f = 0; f < NF / 2; ++f)
                                {
                                    int32_t y = 2 * p[1] + (d == 1 ? up : f), z = DIM == 3 ? 2 * p[2] + (d == 2 ? up : f) : 0;
                                    const int32_t yo = y + (d == 1 ? 2 * up - 1 : 0), zo = z + (d == 2 ? 2 * up - 1 : 0);
                                    const int64_t in  = slot_of(t, lf, 2 * p[0], y, z, 2, row);
                                    const int64_t out = slot_of(t, lf, 2 * p[0], yo, zo, 2, row);
                                    // both faces of a pair are there on graded meshes
                                    const bool ok = in >= 0 && out >= 0 && leaf[out] && leaf[out + 1];
                                    if (out >= 0 && (leaf[out] || leaf[out + 1]) && !ok)
                                    {
                                        fail = true;
                                    }
                                    e[2 * f]     = ok ? int32_t(in) : -1;
                                    e[2 * f + 1] = ok ? int32_t(out) : -1;
                                    any          = any || ok;
                                }
                            }
                            if (any)
                            {
                                kind = SIDE_FINE;
#pragma unroll
                                for (int f = 0; f < NF; ++f)
                                {
                                    slots[n + f] = e[f];
                                }
                                n += NF;
                            }
                        }
                    }
                    w |= kind << (3 * s);
                }
            }
            // one reservation per wave
            const int lane = int(threadIdx.x & 63);
            int32_t incl   = n;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1)
            {
                const int32_t v = __shfl_up(incl, o);
                incl += lane >= o ? v : 0;
            }
            const int32_t total    = __shfl(incl, 63);
            unsigned long long at0 = 0;
            if (lane == 0 && total > 0)
            {
                at0 = atomicAdd(used, (unsigned long long)total);
            }
            at0              = __shfl(at0, 0);
            const int64_t at = int64_t(at0) + incl - n;
            if (!active)
            {
                return;
            }
            if (at + n > room)
            {
                fail    = true;
                w       = 0;
                n       = 0;
            }
            if (fail)
            {
                __hip_atomic_store(fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            word[c]    = w;
            fine_at[c] = int32_t(at);
            for (int k = 0; k < n; ++k)
            {
                fine[at + k] = slots[k];
            }
        }

        // scalar non-linear upwind flux of f(u) = u * u
        // (schemes/fv/operators/convection_nonlin.hpp:54-67)
        __device__ __forceinline__ double burgers_flux(double ul, double ur)
        {
            const double v = 0.5 * (ul + ur);
            return v >= 0 ? ul * ul : ur * ur;
        }

        // the term of an interface between slots sl and sr along d with the
        // signed factor f (linear: the velocity in it)
        template <int OP>
        __device__ __forceinline__ double interface_term(const ConvFields& a, int d, int64_t sl, int64_t sr, double f, bool from_left)
        {
            if constexpr (OP == CONV_LINEAR)
            {
                return f * a.u[from_left ? sl : sr];
            }
            else if constexpr (OP == CONV_BURGERS)
            {
                return burgers_flux(a.u[sl], a.u[sr]) * f;
            }
            else
            {
                // w = 0.5 * (v_d[left] + v_d[right]) (convection_lin.hpp:210-226)
                const double* v    = d == 0 ? a.v[0] : (d == 1 ? a.v[1] : a.v[2]);
                const double w     = 0.5 * (v[sl] + v[sr]);
                // both loaded, so that neither waits for w
                const double ul = a.u[sl], ur = a.u[sr];
                return (f * w) * (w >= 0 ? ul : ur);
            }
        }

        // the terms of a side to finer cells (up: the right one), loaded at once:
        // one per entry, in the order in which they are added
        template <int DIM, int OP>
        struct FineTerms
        {
            static constexpr int NF = 1 << (DIM - 1);
            double t[NF];
            bool ok[NF];
            __device__ __forceinline__ void load(const ConvFields& a, int d, const int32_t (&e)[NF], bool up, double f, bool from_left)
            {
#pragma unroll
                for (int k = 0; k < NF; ++k)
                {
                    // along x an entry is a face, else two are a pair of faces
                    const int32_t first = d == 0 ? e[k] : e[k & ~1];
                    ok[k]               = first >= 0;
                    const int64_t in    = ok[k] ? (d == 0 ? first : first + (k & 1)) : 0;
                    const int64_t o     = ok[k] ? (d == 0 ? first + (up ? 1 : -1) : e[k | 1] + (k & 1)) : 0;
                    t[k]                = interface_term<OP>(a, d, up ? in : o, up ? o : in, f, from_left);
                }
            }
            __device__ __forceinline__ void add(double& acc, int d) const
            {
                if (OP == CONV_LINEAR && d != 0)
                {
#pragma unroll
                    for (int k = 0; k < NF; k += 2)
                    {
                        acc = ok[k] ? acc + (t[k] + t[k + 1]) : acc;
                    }
                    return;
                }
#pragma unroll
                for (int k = 0; k < NF; ++k)
                {
                    acc = ok[k] ? acc + t[k] : acc;
                }
            }
        };

        template <int DIM, int OP>
        __device__ __forceinline__ void convect_cell(const List& l, const ConvSides& sd, const ConvFields& a, int64_t c, double* __restrict__ out)
        {
            constexpr int NF   = 1 << (DIM - 1);
            const int32_t word = sd.word[c];
            const int32_t* fe  = sd.fine + sd.fine_at[c];
            const Cell cell    = locate(l, c);
            const int64_t* b   = bases(l, cell.run);
            const int64_t own  = b[0] + cell.x;
            const double fa    = double(int64_t(1) << cell.level);   // h^(dim-1) / h^dim
            const double ff    = fa / double(NF);                    // (h/2)^(dim-1) / h^dim: a face to a finer cell
            // the entries of all sides to finer cells, NF words each
            int32_t entry[2 * DIM][NF];
#pragma unroll
            for (int s = 0; s < 2 * DIM; ++s)
            {
                if (side_of(word, s) == SIDE_FINE)
                {
                    __builtin_memcpy(entry[s], __builtin_assume_aligned(fe, 4 * NF), 4 * NF);
                    fe += NF;
                }
            }
            double acc = 0;
#pragma unroll
            for (int d = 0; d < DIM; ++d)
            {
                const int64_t left = d == 0 ? own - 1 : b[2 * d - 1] + cell.x, right = d == 0 ? own + 1 : b[2 * d] + cell.x;
                const int kl = side_of(word, 2 * d), kr = side_of(word, 2 * d + 1);
                const double v = OP == CONV_LINEAR ? a.vel[d] : 1.0;
                if (OP == CONV_LINEAR && v == 0.0)
                {
                    continue; // no terms
                }
                // linear: the upwind side carries the velocity; the left
                // cell of an interface adds, the right one subtracts
                const bool from_left = v >= 0;
                const double fc = OP == CONV_LINEAR ? fa * v : fa;
                double tl = 0, tr = 0; // the terms of the left and right face
                if (kl != SIDE_FINE && kl != SIDE_NONE)
                {
                    tl = interface_term<OP>(a, d, left, own, -fc, from_left);
                }
                if (kr != SIDE_FINE && kr != SIDE_NONE)
                {
                    tr = interface_term<OP>(a, d, own, right, fc, from_left);
                }
                FineTerms<DIM, OP> fl, fr;
                if (kr == SIDE_FINE)
                {
                    fr.load(a, d, entry[2 * d + 1], true, OP == CONV_LINEAR ? ff * v : ff, from_left);
                }
                if (kl == SIDE_FINE)
                {
                    fl.load(a, d, entry[2 * d], false, OP == CONV_LINEAR ? -ff * v : -ff, from_left);
                }
                if (OP == CONV_LINEAR && d == 0)
                {
                    if (kr == SIDE_SAME)
                    {
                        acc += tr;
                    }
                    if (kl == SIDE_SAME)
                    {
                        acc += tl;
                    }
                }
                else
                {
                    if (kl == SIDE_SAME)
                    {
                        acc += tl;
                    }
                    if (kr == SIDE_SAME)
                    {
                        acc += tr;
                    }
                }
                if (kl == SIDE_COARSE)
                {
                    acc += tl;
                }
                if (kr == SIDE_COARSE)
                {
                    acc += tr;
                }
                if (kr == SIDE_FINE)
                {
                    fr.add(acc, d);
                }
                if (kl == SIDE_FINE)
                {
                    fl.add(acc, d);
                }
                if (kr == SIDE_BOUNDARY)
                {
                    acc += tr;
                }
                if (kl == SIDE_BOUNDARY)
                {
                    acc += tl;
                }
            }
            out[own] = acc;
        }

        // the first blocks take the cells; the others, 8 slots a thread, zero the
        // slots that are no cells (a clearing of the whole output ahead of the
        // launch was another 2 us of a small mesh's 18).  No bound on the registers:
        // 68 instead of 88 for the 3D velocity field took uniform L7 from 51.1 to
        // 46.6 us, but small meshes, which wait for their loads together, from 51.5
        // to 54.7 (L2..4) and 88.4 to 92.3 (L2..5).
        template <int DIM, int OP>
        __global__ __launch_bounds__(CB) void k_convection(List l, ConvSides sd, ConvFields a, double* __restrict__ out, unsigned cell_blocks)
        {
            if (blockIdx.x < cell_blocks)
            {
                const int64_t c = int64_t(blockIdx.x) * CB + threadIdx.x;
                if (c < l.ncells)
                {
                    convect_cell<DIM, OP>(l, sd, a, c, out);
                }
                return;
            }
            const int64_t s0 = 8 * (int64_t(blockIdx.x - cell_blocks) * CB + threadIdx.x);
            if (s0 >= sd.nref)
            {
                return;
            }
            const uint64_t cells = *reinterpret_cast<const uint64_t*>(sd.leaf + s0);
#pragma unroll
            for (int k = 0; k < 8; ++k)
            {
                if (!((cells >> (8 * k)) & 1))
                {
                    out[s0 + k] = 0.0;
                }
            }
        }

        unsigned blocks(int64_t n)
        {
            return unsigned((n + CB - 1) / CB);
        }

        template <int DIM>
        void launch(int op, const List& l, const ConvSides& sd, const ConvFields& a, double* out, hipStream_t s)
        {
            const unsigned nc = blocks(l.ncells);
            const dim3 g(nc + blocks((sd.nref + 7) / 8)), b(CB);
            switch (op)
            {
                case CONV_LINEAR: hipLaunchKernelGGL((k_convection<DIM, CONV_LINEAR>), g, b, 0, s, l, sd, a, out, nc); break;
                case CONV_BURGERS: hipLaunchKernelGGL((k_convection<DIM, CONV_BURGERS>), g, b, 0, s, l, sd, a, out, nc); break;
                default: hipLaunchKernelGGL((k_convection<DIM, CONV_FIELD>), g, b, 0, s, l, sd, a, out, nc); break;
            }
        }
    } // namespace

    void conv_sides(int dim, const List& l, const Table& t, uint8_t* leaf, int64_t nref, int32_t* word, int32_t* fine_at, int32_t* fine, double* used,
                    int64_t room, int* fault, hipStream_t s)
    {
        if (l.ncells <= 0)
        {
            return;
        }
        zero_u8(leaf, conv_leaf_bytes(nref), s);
        zero_f64(used, 1, s);
        hipLaunchKernelGGL(k_leaf_flags, dim3(blocks(l.ncells)), dim3(CB), 0, s, l, leaf, nref);
        auto* count = reinterpret_cast<unsigned long long*>(used);
        if (dim == 2)
        {
            hipLaunchKernelGGL(k_side_kinds<2>, dim3(blocks(l.ncells)), dim3(CB), 0, s, l, t, leaf, word, fine_at, fine, count, room, fault);
        }
        else
        {
            hipLaunchKernelGGL(k_side_kinds<3>, dim3(blocks(l.ncells)), dim3(CB), 0, s, l, t, leaf, word, fine_at, fine, count, room, fault);
        }
    }

    void convection(int dim, int op, const List& l, const ConvSides& sd, const ConvFields& a, double* out, hipStream_t s)
    {
        if (l.ncells <= 0)
        {
            return;
        }
        if (dim == 2)
        {
            launch<2>(op, l, sd, a, out, s);
        }
        else
        {
            launch<3>(op, l, sd, a, out, s);
        }
    }
} // namespace smr::dev
