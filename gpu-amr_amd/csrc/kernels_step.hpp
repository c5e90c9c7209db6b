// kernels_step.hpp -- the leaf-patch upwind update with the halo gather fused
// in, the padded (halo-exchanged) view, and the refinement criteria.
//
// State in HBM: one buffer of n^R interior doubles per leaf slot (compact,
// 4 KiB per 8^3 patch, 2 KiB per 16^2 patch), leaves in Morton order.  Ghost
// values are not stored: each workgroup gathers the ghost layer of its patch
// from the neighbours' interiors through the device neighbour table, with the
// reference's same / finer (mean) / coarser (injection) rules, into LDS.
//
// Bodies that work on one item alone are __host__ __device__, so that they run
// on the CPU item by item; kernels whose lanes share LDS or registers run there
// as a whole, a launch lane by lane (the tests do both).
#pragma once

#include "device_common.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace amrhip
{

// Per-launch step constants.  dtdx[l][d] = dt / cell_size(l)[d] and
// hs[d] = 0.5 * |v_d| are formed on the host with the same IEEE operations
// the reference performs per cell (amr_solver.hpp:333,
// AdvectionPhysics.hpp:61-65).
struct step_params
{
    double   vel[3];
    double   hs[3];
    double   dtdx[kMaxLevels][3];
    uint32_t reverse; // walk this launch's leaves backwards (sweep_item)
};

// Leaf (or run) of workgroup b: each XCD owns the same contiguous range in
// every launch (xcd_item), walked backwards when `reverse` is set.
// Consecutive steps alternate the direction, so that a step starts on the
// leaves the previous one wrote last -- the lines most likely still in the
// memory-side cache (8^3 step, 32768 leaves: 57 us alternating against 65 us
// always forward) -- while a tree small enough for the XCDs' L2s keeps finding
// its leaves in the L2 that wrote them.  Items >= count are skipped by the
// caller.  `walk` is walk_of(items, reverse): an argument of its own ahead of
// the constants, so that the hardware hands it to the wave with the pointers
// (kernel arguments up to the first structure arrive in scalar registers; a
// load of them would stand before the kernel's first load of data).
__device__ inline uint32_t sweep_item(uint32_t b, uint32_t walk)
{
    const uint32_t per = walk >> 1, j = b / kXcds;
    return (b % kXcds) * per + ((walk & 1) ? per - 1 - j : j);
}

inline uint32_t walk_of(uint64_t items, uint32_t reverse) { return xcd_grid(items) / kXcds * 2 + (reverse & 1u); }

// Output store of a step kernel.  The default is a store at agent scope: it
// goes through L2 to the memory side at once, where a plain store leaves a
// dirty line that the end of the kernel has to write back, with the next
// step waiting behind it.  us per step, plain -> agent scope: 512 leaves of
// 8^3 4.46 -> 4.07, 484 of 16^2 2.95 -> 2.84, 22500 of 8^3 36.5 -> 35.6, 1765
// of 12x10x6 12.8 -> 11.9; single-level 8^3 two-step launches unchanged.  The
// non-temporal form streams the new state past L2 so that L2 keeps the input
// lines that neighbouring leaves' ghost gathers re-read.
template <bool NT>
__device__ inline void store_cell(double* p, double v)
{
    if constexpr (NT)
        __builtin_nontemporal_store(v, p);
    else
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Where a launch's step constants come from: its own argument, one entry of a
// table in device memory (a captured launch, whose constants change between
// replays) or, for a batch of concatenated trees, the entry of the leaf's
// instance.
enum : int
{
    FROM_LAUNCH = 0,
    FROM_TABLE  = 1,
    PER_LEAF    = 2,
};

// A leaf's step constants.  Its key and instance are read at the top of a
// kernel, next to the leaf's face records, and the constants they select
// before the ghosts arrive: read after them they were two or three more round
// trips to memory, one behind the other, in kernels bound by such chains (8^3
// step of 22500 adapted leaves 39.4 -> 35.3 us, 16^2 step of a batch of 74000
// leaves 82 -> 79 us).
template <int R>
struct step_consts
{
    double dtdx[R], vel[R], hs[R];
};

template <int FROM>
__device__ inline uint32_t leaf_instance(const uint32_t* __restrict__ inst, uint32_t leaf)
{
    if constexpr (FROM == PER_LEAF) return inst[leaf];
    return 0;
}

template <int FROM, int R>
__device__ inline step_consts<R> leaf_consts(step_params const& prm, const step_params* __restrict__ table,
                                             uint32_t who, int lv)
{
    step_consts<R> c;
    auto           take = [&](step_params const& P) {
#pragma unroll
        for (int d = 0; d < R; ++d)
        {
            c.dtdx[d] = P.dtdx[lv][d];
            c.vel[d]  = P.vel[d];
            c.hs[d]   = P.hs[d];
        }
    };
    if constexpr (FROM == FROM_LAUNCH)
        take(prm);
    else
        take(table[who]);
    return c;
}

// Ghost value of the cell with layout coordinates c (c[dim] lies outside
// [0, n(dim)): >= n(dim) on the positive side, < 0 on the negative side) of
// the leaf whose direction-`dir` neighbour record is (L, meta).  Restates
// halo_exchange_impl_t::{same_t, finer_t, coarser_t}
// (include/ndtree/patch_utils.hpp:315-441) in compact coordinates:
//   same    -> neighbour cell at the wrapped normal coordinate;
//   finer   -> mean of the 2^R fine cells, summed from 0.0 in row-major order;
//   coarser -> injection of the coarse cell under the contact quadrant.
// The fine cells' base coordinate along every dim d is (2 v) mod n(d), as
// the reference's device twin takes it (src/cuda/halo_exchange.cu:174-176).
// Its CPU rule reduces every dim mod n(dim) of the face normal
// (patch_utils.hpp:358), the same for square patches only; for other shapes
// that rule addresses cells outside the fine patch's interior.
template <int R, class BX>
__host__ __device__ inline double ghost_value(BX const& B, const double* __restrict__ u, const face_link& L,
                                              uint32_t meta, int dir, const int* c)
{
    const int  dim = dir >> 1;
    const bool pos = (dir & 1) != 0;
    const int  nrm = pos ? c[dim] - B.n(dim) : c[dim] + B.n(dim); // reference's from_idxs[dim]
    switch (rel_of(meta))
    {
        case REL_SAME:
        {
            int cc[R];
            for (int d = 0; d < R; ++d) cc[d] = (d == dim) ? nrm : c[d];
            return u[static_cast<size_t>(L.ids[0]) * B.ni() + B.lin(cc)];
        }
        case REL_COARSER:
        {
            int cc[R];
            for (int d = 0; d < R; ++d)
                cc[d] = static_cast<int>(quad_of(meta, d)) * B.half(d) + ((d == dim) ? nrm : c[d]) / 2;
            return u[static_cast<size_t>(L.ids[0]) * B.ni() + B.lin(cc)];
        }
        case REL_FINER:
        {
            int k = 0, bit = 0, base[R];
            for (int d = 0; d < R; ++d)
            {
                const int v = (d == dim) ? nrm : c[d];
                base[d]     = B.fine(v, d);
                if (d != dim)
                {
                    k |= B.half_of(c[d], d) << bit;
                    ++bit;
                }
            }
            const double* q   = u + static_cast<size_t>(L.ids[k]) * B.ni();
            double        sum = 0.0;
            for (int o = 0; o < box<R>::F; ++o)
            {
                int cc[R];
                for (int d = 0; d < R; ++d) cc[d] = base[d] + ((o >> (R - 1 - d)) & 1);
                sum += q[B.lin(cc)];
            }
            return sum / static_cast<double>(box<R>::F);
        }
        default: return 0.0;
    }
}

template <int R, int N>
__host__ __device__ inline double ghost_value(const double* __restrict__ u, const face_link& L, uint32_t meta, int dir,
                                              const int* c)
{
    constexpr box<R> B = box<R>::cube(N);
    return ghost_value<R>(B, u, L, meta, dir, c);
}

// LDS tile of the patch plus one ghost layer: (N+2)^R doubles.
template <int R, int N>
struct tile_shape
{
    static constexpr int TP = N + 2;
    static constexpr int TS = (R == 2) ? TP * TP : TP * TP * TP;
    __host__ __device__ static int idx(const int* c)
    {
        int l = 0;
        for (int d = 0; d < R; ++d) l = l * TP + (c[d] + 1);
        return l;
    }
    // stride of layout dim j inside the tile
    __host__ __device__ static constexpr int stride(int j)
    {
        return (R == 3 && j == 0) ? TP * TP : (j == R - 1 ? 1 : TP);
    }
};

// Interior cell i of the leaf into the tile.
template <int R, int N>
__host__ __device__ inline void stage_interior(double* tile, const double* __restrict__ up, int i)
{
    int c[R];
    patch_shape<R, N>::coords(i, c);
    tile[tile_shape<R, N>::idx(c)] = up[i];
}

// Ghost item g in [0, 2R * N^(R-1)): direction g / N^(R-1), tangential
// position g % N^(R-1) in row-major order over the non-normal dims.
// Returns the direction and sets c to the (padded-frame) cell of ghost item g.
template <int R, int N>
__host__ __device__ inline int ghost_cell(int g, int* c)
{
    using S       = patch_shape<R, N>;
    const int dir = g / S::FACE, dim = dir >> 1;
    int       r   = g % S::FACE;
    for (int d = R - 1; d >= 0; --d)
    {
        if (d == dim) continue;
        c[d] = r % N;
        r /= N;
    }
    c[dim] = (dir & 1) ? N : -1;
    return dir;
}

template <int R, int N>
__host__ __device__ inline void stage_ghost(double* tile, const double* __restrict__ u, uint32_t leaf,
                                            const face_link* __restrict__ links, const uint32_t* __restrict__ metas,
                                            int g)
{
    int            c[R];
    const int      dir             = ghost_cell<R, N>(g, c);
    const size_t   e               = static_cast<size_t>(leaf) * patch_shape<R, N>::NDIR + dir;
    tile[tile_shape<R, N>::idx(c)] = ghost_value<R, N>(u, links[e], metas[e], dir, c);
}

// Index into u of the one interior cell that gives the ghost value of cell c
// when the direction-`dir` neighbour (slot nb) is same-level (copy) or
// coarser (injection): ghost_value's single-cell rules.
template <int R, class BX>
__host__ __device__ inline size_t ghost_source(BX const& B, int32_t nb, uint32_t meta, int dir, const int* c)
{
    const int  dim    = dir >> 1;
    const int  nrm    = (dir & 1) ? c[dim] - B.n(dim) : c[dim] + B.n(dim);
    const bool coarse = rel_of(meta) == REL_COARSER;
    int        cc[R];
    for (int d = 0; d < R; ++d)
    {
        const int v = (d == dim) ? nrm : c[d];
        cc[d]       = coarse ? static_cast<int>(quad_of(meta, d)) * B.half(d) + v / 2 : v;
    }
    return static_cast<size_t>(nb) * B.ni() + B.lin(cc);
}

template <int R, int N>
__host__ __device__ inline size_t ghost_source(int32_t nb, uint32_t meta, int dir, const int* c)
{
    constexpr box<R> B = box<R>::cube(N);
    return ghost_source<R>(B, nb, meta, dir, c);
}

// Value of cell c of `leaf` (layout coordinates, at most one of them outside
// the patch): the interior cell, or the ghost value by the face rules.
template <int R, class BX>
__host__ __device__ inline double cell_or_ghost(BX const& B, const double* __restrict__ u, uint32_t leaf,
                                                const face_link* __restrict__ links,
                                                const uint32_t* __restrict__ metas, const int* c)
{
    for (int d = 0; d < R; ++d)
        if (c[d] < 0 || c[d] >= B.n(d))
        {
            const int    dir = 2 * d + (c[d] >= B.n(d) ? 1 : 0);
            const size_t e   = static_cast<size_t>(leaf) * box<R>::NDIR + dir;
            return ghost_value<R>(B, u, links[e], metas[e], dir, c);
        }
    return u[static_cast<size_t>(leaf) * B.ni() + B.lin(c)];
}

// A leaf's face records: relation/quadrant word and neighbour slots per
// direction, read with one batch of scalar loads.
template <int R>
__device__ inline void load_faces(const face_link* __restrict__ L, const uint32_t* __restrict__ M, uint32_t* m,
                                  int4* nb)
{
#pragma unroll
    for (int k = 0; k < 2 * R; ++k)
    {
        m[k]  = M[k];
        nb[k] = int4{ L[k].ids[0], L[k].ids[1], L[k].ids[2], L[k].ids[3] };
    }
}

// Whether none of a leaf's faces has finer neighbours (every ghost is then a
// single cell and the gathers below issue all their loads back to back).
template <int R>
__device__ inline bool single_cell_ghosts(const uint32_t* m)
{
    uint32_t finer = 0;
#pragma unroll
    for (int k = 0; k < 2 * R; ++k) finer |= (rel_of(m[k]) == REL_FINER) ? 1u : 0u;
    return finer == 0;
}

// Ghost cell c of direction DIR with finer neighbours nb: ghost_value's
// finer rule, the fine slot picked by selects.
template <int DIR>
__device__ inline double fine_mean_3d8(const double* __restrict__ u, int4 nb, const int* c)
{
    constexpr box<3> B   = box<3>::cube(8);
    constexpr int    dim = DIR >> 1;
    int              k = 0, bit = 0, cc[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        cc[d] = (d == dim) ? ((DIR & 1) ? 0 : 6) : B.fine(c[d], d);
        if (d != dim)
        {
            k |= B.half_of(c[d], d) << bit;
            ++bit;
        }
    }
    const int32_t slot = (k & 2) ? ((k & 1) ? nb.w : nb.z) : ((k & 1) ? nb.y : nb.x);
    const double* q    = u + static_cast<size_t>(slot) * B.ni() + B.lin(cc);
    double        f[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) f[o] = q[((o >> 2) & 1) * 64 + ((o >> 1) & 1) * 8 + (o & 1)];
    double sum = 0.0;
#pragma unroll
    for (int o = 0; o < 8; ++o) sum += f[o];
    return sum / 8.0;
}

// The six ghost values of a lane of the 3D wave layout (lane = 8 hi + lo),
// from the leaf's face records (m, nb): g[0], g[1] = -z / +z of the column
// (y, x) = (hi, lo); g[2], g[3] = the (z, x) = (hi, lo) cell of the -y / +y
// face; g[4], g[5] = the (z, y) = (hi, lo) cell of the -x / +x face (skipped
// unless wanted).  The single-cell ghosts are loaded back to back for all
// faces (a face with finer neighbours reads a cell it then drops): a
// per-face switch on the relation makes the compiler wait for every
// outstanding load before each face.
__device__ inline void gather_ghosts_3d8(const double* __restrict__ u, const uint32_t* m, const int4* nb, int hi,
                                         int lo, bool want_xm, bool want_xp, double* g)
{
    const int c[6][3] = { { -1, hi, lo }, { 8, hi, lo }, { hi, -1, lo }, { hi, 8, lo }, { hi, lo, -1 }, { hi, lo, 8 } };
    size_t src[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) src[k] = ghost_source<3, 8>(nb[k].x, m[k], k, c[k]);
#pragma unroll
    for (int k = 0; k < 4; ++k) g[k] = u[src[k]];
    g[4] = want_xm ? u[src[4]] : 0.0;
    g[5] = want_xp ? u[src[5]] : 0.0;
    if (single_cell_ghosts<3>(m)) return;
    if (rel_of(m[0]) == REL_FINER) g[0] = fine_mean_3d8<0>(u, nb[0], c[0]);
    if (rel_of(m[1]) == REL_FINER) g[1] = fine_mean_3d8<1>(u, nb[1], c[1]);
    if (rel_of(m[2]) == REL_FINER) g[2] = fine_mean_3d8<2>(u, nb[2], c[2]);
    if (rel_of(m[3]) == REL_FINER) g[3] = fine_mean_3d8<3>(u, nb[3], c[3]);
    if (rel_of(m[4]) == REL_FINER && want_xm) g[4] = fine_mean_3d8<4>(u, nb[4], c[4]);
    if (rel_of(m[5]) == REL_FINER && want_xp) g[5] = fine_mean_3d8<5>(u, nb[5], c[5]);
}

// The cells that give the ghost of cell t of face q, as a lane of the 2D wave
// layout gathers it (lane = 16 q + t): the one of a same-level or coarser
// neighbour or, next to finer neighbours, the 2 x 2 block of one of them, from
// its first cell on.
struct ghost_cells_2d16
{
    size_t first;
    bool   finer;

    __device__ ghost_cells_2d16(const uint32_t* ms, const int4* nbs, int q, int t)
    {
        using S = patch_shape<2, 16>;
        int c[2];
        c[0] = (q == 0) ? -1 : (q == 1) ? 16 : t;
        c[1] = (q == 2) ? -1 : (q == 3) ? 16 : t;
        // the lane's own face record, selected from the four uniform ones
        uint32_t m   = ms[0];
        int32_t  nb  = nbs[0].x;
        int32_t  id1 = nbs[0].y; // second fine slot of a face with finer neighbours
#pragma unroll
        for (int k = 1; k < 4; ++k)
        {
            m   = q == k ? ms[k] : m;
            nb  = q == k ? nbs[k].x : nb;
            id1 = q == k ? nbs[k].y : id1;
        }
        finer = false;
        if (single_cell_ghosts<2>(ms))
        {
            first = ghost_source<2, 16>(nb, m, q, c);
            return;
        }
        finer = rel_of(m) == REL_FINER;
        if (finer)
        {
            // ghost_value's finer rule: fine neighbour t / 8 of the face,
            // cells (2 t) % 16 + {0, 1} along the face, the two layers next
            // to it
            const int dim = q >> 1, nrm = (q & 1) ? c[dim] - 16 : c[dim] + 16;
            int       base[2];
            for (int d = 0; d < 2; ++d) base[d] = (((d == dim) ? nrm : c[d]) * 2) % 16;
            const int32_t fine = (t / S::HALF) ? id1 : nb;
            first              = static_cast<size_t>(fine) * S::NI + S::lin(base);
        }
        else
            first = ghost_source<2, 16>(nb, m, q, c);
    }

    // The ghost value where the leaf has finer neighbours.  Branch-free over
    // the relation, so that the wave's loads are all in flight at once: every
    // lane loads the four cells a finer neighbour's mean needs -- a
    // same-level or coarser neighbour's single cell four times -- and keeps
    // the mean (summed from 0.0 in row-major order, as ghost_value) or the
    // first value.
    __device__ double value(const double* __restrict__ u) const
    {
        double v[4];
#pragma unroll
        for (int o = 0; o < 4; ++o) v[o] = u[first + (finer ? (o >> 1) * 16 + (o & 1) : 0)];
        double sum = 0.0;
#pragma unroll
        for (int o = 0; o < 4; ++o) sum += v[o];
        return finer ? sum / 4.0 : v[0];
    }
};

__device__ inline double gather_ghost_2d16(const double* __restrict__ u, const uint32_t* ms, const int4* nbs, int q,
                                           int t)
{
    const ghost_cells_2d16 cells(ms, nbs, q, t);
    return single_cell_ghosts<2>(ms) ? u[cells.first] : cells.value(u);
}

// The value of lane l - 1 (row_shr) or l + 1 (row_shl) within the lane's
// 16-lane DPP row.  In both wave layouts x runs along consecutive lanes of a
// row, so this is the x neighbour; a lane whose neighbour would come from
// outside its row (or from the other x row of a 3D row) is an x boundary lane,
// which takes its ghost value instead: such lanes read 0 here (bound_ctrl),
// so the move needs no copy of the old value.  A VALU move, where __shfl
// goes through the LDS unit.  Like every cross-lane read it must run with
// all lanes active: evaluate it as a statement of its own, never as an
// operand of ?: (which would run it only in the lanes taking that branch,
// reading the others as invalid).
__device__ inline double lane_minus1(double v)
{
    const uint64_t b  = __builtin_bit_cast(uint64_t, v);
    const int      lo = static_cast<int>(b), hi = static_cast<int>(b >> 32);
    const int      l  = __builtin_amdgcn_update_dpp(0, lo, 0x111, 0xF, 0xF, true); // row_shr:1
    const int      h  = __builtin_amdgcn_update_dpp(0, hi, 0x111, 0xF, 0xF, true);
    return __builtin_bit_cast(double, (static_cast<uint64_t>(static_cast<uint32_t>(h)) << 32) | static_cast<uint32_t>(l));
}

// v = *p in the lanes where `take` holds, p pointing into LDS: a volatile
// LDS read inside the branch, so the compiler keeps it a ds_read under the
// lane mask (the other lanes keep v) instead of a read by every lane and a
// 64-bit select (two VALU instructions).  Used where a boundary lane
// replaces a cross-lane value with one from LDS; the LDS writes it reads
// must be ordered before it by a barrier or leaf_sync.
__device__ inline void take_lds_if(bool take, const double* p, double& v)
{
    typedef __attribute__((address_space(3))) const volatile double lds_double;
    if (__builtin_expect(take, 1)) v = *(lds_double*)(p);
}

__device__ inline double lane_plus1(double v)
{
    const uint64_t b  = __builtin_bit_cast(uint64_t, v);
    const int      lo = static_cast<int>(b), hi = static_cast<int>(b >> 32);
    const int      l  = __builtin_amdgcn_update_dpp(0, lo, 0x101, 0xF, 0xF, true); // row_shl:1
    const int      h  = __builtin_amdgcn_update_dpp(0, hi, 0x101, 0xF, 0xF, true);
    return __builtin_bit_cast(double, (static_cast<uint64_t>(static_cast<uint32_t>(h)) << 32) | static_cast<uint32_t>(l));
}

// Upwind update of one cell from its neighbours along each physical axis d
// (lo[d] = u_L, hi[d] = u_R): the expression order of
// amr_solver::time_step_cpu (amr_solver.hpp:302-347) and
// AdvectionPhysics::rusanovFlux (AdvectionPhysics.hpp:45-66):
//   total = 0; total -= dt/dx_d * (F(u, u_R) - F(u_L, u)) for d = x, y(, z);
//   F(a, b) = 0.5 * (a v + b v) - (0.5 |v|) (b - a); out = u + total.
__host__ __device__ inline double upwind_flux(double a, double b, double v, double hs)
{
    return 0.5 * (a * v + b * v) - hs * (b - a);
}

// The update from the cell's face fluxes, fL[d] = F(u_L, u), fR[d] = F(u, u_R).
// A face flux is the same bits whether computed for the cell on its left or
// on its right, so kernels may evaluate each face once.
template <int R>
__host__ __device__ inline double update_from_fluxes(double uc, const double* fL, const double* fR, const double* dtdx)
{
    double total = 0.0;
    for (int d = 0; d < R; ++d) total -= dtdx[d] * (fR[d] - fL[d]);
    return uc + total;
}

template <int R>
__host__ __device__ inline double upwind_update(double uc, const double* lo, const double* hi, const double* dtdx,
                                                const double* vel, const double* hs)
{
    double fL[R], fR[R];
    for (int d = 0; d < R; ++d)
    {
        fL[d] = upwind_flux(lo[d], uc, vel[d], hs[d]);
        fR[d] = upwind_flux(uc, hi[d], vel[d], hs[d]);
    }
    return update_from_fluxes<R>(uc, fL, fR, dtdx);
}

// Upwind update of interior cell i from the staged tile.
template <int R, int N>
__host__ __device__ inline double upwind_cell(const double* tile, int i, const double* dtdx, const double* vel,
                                              const double* hs)
{
    using T = tile_shape<R, N>;
    int c[R];
    patch_shape<R, N>::coords(i, c);
    const int t = T::idx(c);
    double    lo[R], hi[R];
    for (int d = 0; d < R; ++d)
    {
        const int s = T::stride(R - 1 - d); // physical axis d
        lo[d]       = tile[t - s];
        hi[d]       = tile[t + s];
    }
    return upwind_update<R>(tile[t], lo, hi, dtdx, vel, hs);
}

// max over layout dims of max(|u[c+s]-u[c]|, |u[c]-u[c-s]|) for cell i.
template <int R, int N>
__host__ __device__ inline double gradient_cell(const double* tile, int i)
{
    using T = tile_shape<R, N>;
    int c[R];
    patch_shape<R, N>::coords(i, c);
    const int t = T::idx(c);
    double    g = 0.0;
    for (int j = 0; j < R; ++j)
    {
        const int s = T::stride(j);
        g           = fmax(g, fmax(fabs(tile[t + s] - tile[t]), fabs(tile[t] - tile[t - s])));
    }
    return g;
}

// Cell i of the padded view ((n(d) + 2h) per dim, row-major): interior copy,
// face halo gathered; *kind = 0 interior, 1 face halo, 2 edge/corner (value 0).
template <int R, class BX>
__host__ __device__ inline double padded_value(BX const& B, int h, const double* __restrict__ u, uint32_t leaf,
                                               const face_link* __restrict__ links,
                                               const uint32_t* __restrict__ metas, int i, int* kind)
{
    int c[R], r = i, outside = 0, odim = 0;
    for (int d = R - 1; d >= 0; --d)
    {
        const int p = B.n(d) + 2 * h;
        c[d]        = r % p - h;
        r /= p;
        if (c[d] < 0 || c[d] >= B.n(d))
        {
            ++outside;
            odim = d;
        }
    }
    *kind = outside < 2 ? outside : 2;
    if (outside == 0) return u[static_cast<size_t>(leaf) * B.ni() + B.lin(c)];
    if (outside == 1)
    {
        const int    dir = 2 * odim + (c[odim] >= B.n(odim) ? 1 : 0);
        const size_t e   = static_cast<size_t>(leaf) * box<R>::NDIR + dir;
        return ghost_value<R>(B, u, links[e], metas[e], dir, c);
    }
    return 0.0;
}

template <int R, int N, int H>
__host__ __device__ inline double padded_value(const double* __restrict__ u, uint32_t leaf,
                                               const face_link* __restrict__ links,
                                               const uint32_t* __restrict__ metas, int i, int* kind)
{
    constexpr box<R> B = box<R>::cube(N);
    return padded_value<R>(B, H, u, leaf, links, metas, i, kind);
}

__host__ __device__ inline int8_t decide(double value, int level, double rthr, double cthr, int min_level,
                                         int max_level)
{
    if (value > rthr && level < max_level) return 1;
    if (value < cthr && level > min_level) return 2;
    return 0;
}

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

template <int R, int N, int NT>
__device__ inline void stage_tile(double* tile, const double* __restrict__ u, uint32_t leaf,
                                  const face_link* __restrict__ links, const uint32_t* __restrict__ metas)
{
    using S          = patch_shape<R, N>;
    const double* up = u + static_cast<size_t>(leaf) * S::NI;
    for (int i = threadIdx.x; i < S::NI; i += NT) stage_interior<R, N>(tile, up, i);
    for (int g = threadIdx.x; g < S::NDIR * S::FACE; g += NT) stage_ghost<R, N>(tile, u, leaf, links, metas, g);
}

// ---------------------------------------------------------------------------
// LDS tiles of patches whose extents are launch arguments: the patch plus one
// ghost layer, (n(d) + 2) cells per dim, row-major.
// ---------------------------------------------------------------------------
constexpr size_t kBoxTileBytes = 64 * 1024; // largest of them

template <int R>
struct box_tile
{
    int st[R]; // stride of layout dim d

    template <class BX>
    __host__ __device__ explicit box_tile(BX const& B)
    {
        st[R - 1] = 1;
        for (int d = R - 1; d > 0; --d) st[d - 1] = st[d] * (B.n(d) + 2);
    }
    __host__ __device__ int idx(const int* c) const
    {
        int l = 0;
        for (int d = 0; d < R; ++d) l += (c[d] + 1) * st[d];
        return l;
    }
    template <class BX>
    __host__ __device__ static int cells(BX const& B)
    {
        int l = 1;
        for (int d = 0; d < R; ++d) l *= B.n(d) + 2;
        return l;
    }
};

// Ghost item g (0 <= g < 2 face(D)) of the two faces normal to layout dim D:
// its cell c, and the side (0 negative, 1 positive).  D is a constant, so the
// coordinates stay in registers.
template <int R, int D, class BX>
__host__ __device__ inline int face_pair_item(BX const& B, int g, int* c)
{
    const int fc = B.face(D), side = g >= fc ? 1 : 0, f = side ? g - fc : g;
    if constexpr (R == 2)
        c[1 - D] = f;
    else
    {
        constexpr int hi = D == 0 ? 1 : 0, lo = D == 2 ? 1 : 2;
        c[hi]            = B.quot(f, lo);
        c[lo]            = f - c[hi] * B.n(lo);
    }
    c[D] = side ? B.n(D) : -1;
    return side;
}

// ghost_source for a face normal to the constant dim D.
template <int R, int D, class BX>
__host__ __device__ inline size_t face_source(BX const& B, int32_t nb, uint32_t meta, int side, const int* c)
{
    const bool coarse = rel_of(meta) == REL_COARSER;
    int        cc[R];
    for (int d = 0; d < R; ++d)
    {
        const int v = (d == D) ? (side ? c[D] - B.n(D) : c[D] + B.n(D)) : c[d];
        cc[d]       = coarse ? static_cast<int>(quad_of(meta, d)) * B.half(d) + v / 2 : v;
    }
    return static_cast<size_t>(nb) * B.ni() + B.lin(cc);
}

// First of the 2^R fine cells under ghost cell c of a face normal to D with
// finer neighbours ids (a vector, whose elements a select picks: an array
// indexed by a lane's value would live in scratch memory).
template <int R, int D, class BX>
__host__ __device__ inline size_t face_fine_source(BX const& B, int4 ids, int side, const int* c)
{
    int k = 0, bit = 0, cc[R];
    for (int d = 0; d < R; ++d)
    {
        cc[d] = B.fine((d == D) ? (side ? c[D] - B.n(D) : c[D] + B.n(D)) : c[d], d);
        if (d != D)
        {
            k |= B.half_of(c[d], d) << bit;
            ++bit;
        }
    }
    int32_t nb = (k & 1) ? ids.y : ids.x;
    if constexpr (R == 3) nb = (k & 2) ? ((k & 1) ? ids.w : ids.z) : nb;
    return static_cast<size_t>(nb) * B.ni() + B.lin(cc);
}

__host__ __device__ inline int4 link_ids(const face_link* __restrict__ L) { return *reinterpret_cast<const int4*>(L); }

// Offset of the o-th of those cells (row-major) from the first.
template <int R, class BX>
__host__ __device__ inline int fine_offset(BX const& B, int o)
{
    int l = 0;
    for (int d = 0; d < R; ++d) l += ((o >> (R - 1 - d)) & 1) * B.stride(d);
    return l;
}

// The NV values of the face-ghost cell c (fields fstride apart) of a face with
// record (L, meta) by ghost_value's rules.
template <int R, int NV, int D, class BX>
__device__ inline void face_values(BX const& B, const double* __restrict__ u, size_t fstride, int4 L, uint32_t meta,
                                   int side, const int* c, double* out)
{
    if (rel_of(meta) != REL_FINER)
    {
        const size_t at = face_source<R, D>(B, L.x, meta, side, c);
#pragma unroll
        for (int v = 0; v < NV; ++v) out[v] = u[v * fstride + at];
        return;
    }
    const size_t first = face_fine_source<R, D>(B, L, side, c);
    double       sum[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) sum[v] = 0.0;
#pragma unroll
    for (int o = 0; o < (1 << R); ++o)
#pragma unroll
        for (int v = 0; v < NV; ++v) sum[v] += u[v * fstride + first + fine_offset<R>(B, o)];
#pragma unroll
    for (int v = 0; v < NV; ++v) out[v] = sum[v] / static_cast<double>(1 << R);
}

// The NV values (fields fstride apart) of the cell before (SIDE 0) or after
// (SIDE 1) cell c of `leaf` along layout dim D: a cell of the patch or, past
// its last one, the face's ghost.
template <int R, int NV, int D, int SIDE, class BX>
__host__ __device__ inline void neighbour_values(BX const& B, const double* __restrict__ u, size_t fstride,
                                                 uint32_t leaf, const face_link* __restrict__ links,
                                                 const uint32_t* __restrict__ metas, const int* c, double* out)
{
    if (SIDE ? c[D] + 1 < B.n(D) : c[D] > 0)
    {
        const size_t at = static_cast<size_t>(leaf) * B.ni() + (B.lin(c) + (SIDE ? B.stride(D) : -B.stride(D)));
#pragma unroll
        for (int v = 0; v < NV; ++v) out[v] = u[v * fstride + at];
        return;
    }
    int g[R];
    for (int d = 0; d < R; ++d) g[d] = c[d];
    g[D]                = SIDE ? B.n(D) : -1;
    const size_t   e    = static_cast<size_t>(leaf) * box<R>::NDIR + (2 * D + SIDE);
    const uint32_t meta = metas[e];
    const int4     L    = link_ids(links + e);
    if (rel_of(meta) != REL_FINER)
    {
        const size_t at = face_source<R, D>(B, L.x, meta, SIDE, g);
#pragma unroll
        for (int v = 0; v < NV; ++v) out[v] = u[v * fstride + at];
        return;
    }
    // face_values' sums, the cells up to 20 at a time in flight: left to
    // itself the compiler keeps registers by waiting for them one by one
    constexpr int F = 1 << R, BATCH = NV * F <= 20 ? F : F / 2;
    const size_t  first = face_fine_source<R, D>(B, L, SIDE, g);
    double        sum[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) sum[v] = 0.0;
#pragma unroll
    for (int o0 = 0; o0 < F; o0 += BATCH)
    {
        double f[BATCH][NV];
#pragma unroll
        for (int o = 0; o < BATCH; ++o)
#pragma unroll
            for (int v = 0; v < NV; ++v) f[o][v] = u[v * fstride + first + fine_offset<R>(B, o0 + o)];
#ifdef __HIP_DEVICE_COMPILE__
        __builtin_amdgcn_sched_barrier(0);
#endif
#pragma unroll
        for (int o = 0; o < BATCH; ++o)
#pragma unroll
            for (int v = 0; v < NV; ++v) sum[v] += f[o][v];
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) out[v] = sum[v] / static_cast<double>(F);
}

// The upwind update of interior cell i of `leaf` with its neighbours read
// from memory (interior cells, or ghost values at the patch boundary): the
// same operands as upwind_cell on a staged tile, for patches of any shape.
template <int R, class BX>
__host__ __device__ inline double upwind_cell_direct(BX const& B, const double* __restrict__ u, uint32_t leaf,
                                                     const face_link* __restrict__ links,
                                                     const uint32_t* __restrict__ metas, int i, const double* dtdx,
                                                     const double* vel, const double* hs)
{
    int c[R];
    B.coords(i, c);
    double lo[R], hi[R];
    auto   along = [&](auto dim) {
        constexpr int J = decltype(dim)::value; // layout dim of physical axis R - 1 - J
        neighbour_values<R, 1, J, 0>(B, u, 0, leaf, links, metas, c, &lo[R - 1 - J]);
        neighbour_values<R, 1, J, 1>(B, u, 0, leaf, links, metas, c, &hi[R - 1 - J]);
    };
    along(std::integral_constant<int, 0>{});
    along(std::integral_constant<int, 1>{});
    if constexpr (R == 3) along(std::integral_constant<int, 2>{});
    return upwind_update<R>(u[static_cast<size_t>(leaf) * B.ni() + i], lo, hi, dtdx, vel, hs);
}

// gradient_cell with the neighbours read from memory (any patch shape).
template <int R, class BX>
__host__ __device__ inline double gradient_cell_direct(BX const& B, const double* __restrict__ u, uint32_t leaf,
                                                       const face_link* __restrict__ links,
                                                       const uint32_t* __restrict__ metas, int i)
{
    int c[R];
    B.coords(i, c);
    const double uc = u[static_cast<size_t>(leaf) * B.ni() + i];
    double       g  = 0.0;
    auto         along = [&](auto dim) {
        constexpr int J = decltype(dim)::value;
        double        um, up;
        neighbour_values<R, 1, J, 0>(B, u, 0, leaf, links, metas, c, &um);
        neighbour_values<R, 1, J, 1>(B, u, 0, leaf, links, metas, c, &up);
        g = fmax(g, fmax(fabs(up - uc), fabs(uc - um)));
    };
    along(std::integral_constant<int, 0>{});
    along(std::integral_constant<int, 1>{});
    if constexpr (R == 3) along(std::integral_constant<int, 2>{});
    return g;
}

// How a workgroup of NT threads walks the cells of a patch: `layers` layers of
// layout dim 0 at a time, one cell per thread, so that a thread keeps its
// column (the other coordinates) and steps along dim 0 with two additions per
// cell; `passes` times.  Chosen on the host (box_walk_for).
struct box_walk
{
    int32_t layers, passes;
};

// The walk of a patch (box_walk) and its workgroup size: the one of 64,
// 128, 256 (512 from 2048 cells on) threads that spends the fewest thread
// slots in at most four passes, the smaller one of equals, else the
// largest.  0 when a layer has more cells than the largest workgroup.
template <int R>
int box_walk_for(box<R> const& B, box_walk& W)
{
    const int cols = B.face(0), most = B.ni() >= 2048 ? 512 : 256;
    int       best = 0, slots = 0;
    for (int nt = 64; nt <= most; nt *= 2)
    {
        if (cols > nt) continue;
        const int layers = B.n(0) < nt / cols ? B.n(0) : nt / cols;
        const int passes = (B.n(0) + layers - 1) / layers;
        if (best && (passes * nt >= slots) && !(W.passes > 4)) continue;
        best  = nt;
        slots = passes * nt;
        W     = box_walk{ layers, passes };
    }
    return best;
}

// One thread's walk: active while k < passes and cell(k) is in the patch.
template <int R>
struct box_column
{
    int  i0, di; // patch cell of pass 0, step per pass
    int  t0, dt; // the same in the tile
    int  z0, dz; // layer
    bool on;

    template <class BX>
    __device__ box_column(BX const& B, box_tile<R> const& T, box_walk const& W)
    {
        const int cols = B.face(0), tid = threadIdx.x;
        di             = W.layers * cols;
        on             = tid < di;
        i0             = on ? tid : 0;
        dz             = W.layers;
        dt             = dz * T.st[0];
        int c[R];
        B.coords(i0, c); // W.layers <= n(0): a cell of the patch
        z0 = c[0];
        t0 = T.idx(c);
    }
};

// Stages every field's tile of `leaf` (field v at tile + v * cells): the
// patch and its face ghosts, edges and corners untouched.  Bound by the two
// dependent loads of a ghost (its face record, then its cell), so the first
// NT items of each face pair and CH cells per thread are loaded before any is
// stored, the face pairs starting on different waves.
template <int R, int NT, int NV, int CH, class BX>
__device__ inline void stage_box(BX const& B, box_tile<R> const& T, box_column<R> const& col, box_walk const& W,
                                 double* tile, const double* __restrict__ u, size_t fstride, uint32_t leaf,
                                 const face_link* __restrict__ links, const uint32_t* __restrict__ metas)
{
    const int        cells = box_tile<R>::cells(B), tid = threadIdx.x;
    const double*    own   = u + static_cast<size_t>(leaf) * B.ni();
    const face_link* L     = links + static_cast<size_t>(leaf) * box<R>::NDIR;
    const uint32_t*  M     = metas + static_cast<size_t>(leaf) * box<R>::NDIR;
    // this thread's first ghost item of each face pair and its record
    int      gc[R][R], item[R], side[R];
    uint32_t meta[R];
    int4     link[R];
    auto     first_item = [&](auto dim) {
        constexpr int D     = decltype(dim)::value;
        constexpr int shift = (D * NT / R) / 64 * 64;
        item[D]             = (tid + NT - shift) % NT;
        const bool on       = item[D] < 2 * B.face(D);
        side[D]             = face_pair_item<R, D>(B, on ? item[D] : 0, gc[D]);
        meta[D]             = M[2 * D + side[D]];
        link[D]             = link_ids(L + 2 * D + side[D]);
    };
    first_item(std::integral_constant<int, 0>{});
    first_item(std::integral_constant<int, 1>{});
    if constexpr (R == 3) first_item(std::integral_constant<int, 2>{});
    double r[CH][NV];
    auto   load_cells = [&](int k0) {
#pragma unroll
        for (int k = 0; k < CH; ++k)
        {
            const int i = col.z0 + (k0 + k) * col.dz < B.n(0) ? col.i0 + (k0 + k) * col.di : col.i0;
#pragma unroll
            for (int v = 0; v < NV; ++v) r[k][v] = own[v * fstride + i];
        }
    };
    auto store_cells = [&](int k0) {
#pragma unroll
        for (int k = 0; k < CH; ++k)
            if (col.on && col.z0 + (k0 + k) * col.dz < B.n(0))
            {
#pragma unroll
                for (int v = 0; v < NV; ++v) tile[v * cells + col.t0 + (k0 + k) * col.dt] = r[k][v];
            }
    };
    load_cells(0);
    // single-cell ghosts of every face pair at once, then, in a wave that
    // has finer neighbours, the 2^R fine cells (the cells of all face pairs
    // at once took 84 instead of 60 registers in 3D and was 4 % slower)
    size_t at[R];
    at[0] = face_source<R, 0>(B, link[0].x, meta[0], side[0], gc[0]);
    at[1] = face_source<R, 1>(B, link[1].x, meta[1], side[1], gc[1]);
    if constexpr (R == 3) at[2] = face_source<R, 2>(B, link[2].x, meta[2], side[2], gc[2]);
    double g[R][NV];
    bool   fine[R], any_fine = false;
#pragma unroll
    for (int d = 0; d < R; ++d)
    {
#pragma unroll
        for (int v = 0; v < NV; ++v) g[d][v] = u[v * fstride + at[d]];
        fine[d]  = rel_of(meta[d]) == REL_FINER;
        any_fine = any_fine || fine[d];
    }
    if (__any(any_fine))
    {
        at[0] = fine[0] ? face_fine_source<R, 0>(B, link[0], side[0], gc[0]) : at[0];
        at[1] = fine[1] ? face_fine_source<R, 1>(B, link[1], side[1], gc[1]) : at[1];
        if constexpr (R == 3) at[2] = fine[2] ? face_fine_source<R, 2>(B, link[2], side[2], gc[2]) : at[2];
        constexpr int F = 1 << R;
#pragma unroll
        for (int d = 0; d < R; ++d)
            if (fine[d])
            {
                double sum[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) sum[v] = 0.0;
#pragma unroll
                for (int o = 0; o < F; ++o)
#pragma unroll
                    for (int v = 0; v < NV; ++v) sum[v] += u[v * fstride + at[d] + fine_offset<R>(B, o)];
#pragma unroll
                for (int v = 0; v < NV; ++v) g[d][v] = sum[v] / static_cast<double>(F);
            }
    }
    store_cells(0);
#pragma unroll
    for (int d = 0; d < R; ++d)
        if (item[d] < 2 * B.face(d))
        {
#pragma unroll
            for (int v = 0; v < NV; ++v) tile[v * cells + T.idx(gc[d])] = g[d][v];
        }
    // what is left of larger patches
    for (int k = CH; k < W.passes; k += CH)
    {
        load_cells(k);
        store_cells(k);
    }
    auto rest = [&](auto dim) {
        constexpr int D = decltype(dim)::value;
        for (int q = item[D] + NT; q < 2 * B.face(D); q += NT)
        {
            int       c[R];
            const int sd = face_pair_item<R, D>(B, q, c);
            double    w[NV];
            face_values<R, NV, D>(B, u, fstride, link_ids(L + 2 * D + sd), M[2 * D + sd], sd, c, w);
#pragma unroll
            for (int v = 0; v < NV; ++v) tile[v * cells + T.idx(c)] = w[v];
        }
    };
    rest(std::integral_constant<int, 0>{});
    rest(std::integral_constant<int, 1>{});
    if constexpr (R == 3) rest(std::integral_constant<int, 2>{});
}

// Upwind update of tile cell t from a staged tile.
template <int R>
__device__ inline double upwind_tile_cell(const double* tile, box_tile<R> const& T, int t, const double* dtdx,
                                          const double* vel, const double* hs)
{
    double lo[R], hi[R];
#pragma unroll
    for (int d = 0; d < R; ++d)
    {
        lo[d] = tile[t - T.st[R - 1 - d]];
        hi[d] = tile[t + T.st[R - 1 - d]];
    }
    return upwind_update<R>(tile[t], lo, hi, dtdx, vel, hs);
}

// One time step for every leaf; one workgroup per leaf patch
// (XCD-contiguous ranges).
template <int R, int N, int NT, int FROM>
__global__ __launch_bounds__(NT) void k_step(const double* __restrict__ u, double* __restrict__ un,
                                             const uint64_t* __restrict__ keys,
                                             const face_link* __restrict__ links,
                                             const uint32_t* __restrict__ metas, uint32_t nleaves, uint32_t walk, step_params prm,
    const step_params* __restrict__ table, const uint32_t* __restrict__ inst)
{
    using S = patch_shape<R, N>;
    __shared__ double tile[tile_shape<R, N>::TS];
    const uint32_t leaf = sweep_item(blockIdx.x, walk);
    if (leaf >= nleaves) return;
    const uint32_t who = leaf_instance<FROM>(inst, leaf);
    const int      lv  = key_level(keys[leaf]);
    stage_tile<R, N, NT>(tile, u, leaf, links, metas);
    const step_consts<R> C = leaf_consts<FROM, R>(prm, table, who, lv);
    __syncthreads();
    double* out = un + static_cast<size_t>(leaf) * S::NI;
    // Through L2 (store_cell) only where a step writes enough for it: us per
    // step, plain / through, 64^2: 64 leaves 8.5 / 10.2, 256 11.6 / 12.6, 484
    // 14.8 / 13.6, 1024 19.7 / 17.2; of the small patches 484 leaves of 8^2 6.7 / 7.1, 2339 of
    // 4^3 (three steps) 33.6 / 35.8 us, 12692 of 4^3 12.3 / 12.8.
    const bool through = S::NI >= 4096 && nleaves >= 400;
    for (int i = threadIdx.x; i < S::NI; i += NT)
    {
        const double v = upwind_cell<R, N>(tile, i, C.dtdx, C.vel, C.hs);
        if (through)
            store_cell<false>(out + i, v);
        else
            out[i] = v;
    }
}

// 3D 8^3 patches, one wave (64 lanes) per leaf.  Lane l owns the z-column at
// (y, x) = (l / 8, l % 8) in registers: x- and y-neighbours come from lanes
// l -+ 1 and l -+ 8, z-neighbours from the lane's own registers.  The six
// ghost faces are gathered one face cell per lane; the -+z faces land in the
// lane that needs them, the -+y / -+x faces go through 2 KiB of LDS.  With
// no interior tile in LDS, 32 leaves are in flight per CU.
template <bool NT, int FROM>
__device__ inline void step_leaf_3d8(const double* __restrict__ u, double* __restrict__ un,
                                     const uint64_t* __restrict__ keys, const face_link* __restrict__ links,
                                     const uint32_t* __restrict__ metas, uint32_t leaf, step_params const& prm,
                                     const step_params* __restrict__ table, const uint32_t* __restrict__ inst)
{
    constexpr int NI = 512;
    __shared__ double gface[4][64]; // -y, +y (index z*8+x), -x, +x (index z*8+y)
    const int      lane = threadIdx.x, hi3 = lane >> 3, lo3 = lane & 7;
    const uint32_t who  = leaf_instance<FROM>(inst, leaf);
    const int      lv   = key_level(keys[leaf]);
    uint32_t       m[6];
    int4           nb[6];
    load_faces<3>(links + static_cast<size_t>(leaf) * 6, metas + static_cast<size_t>(leaf) * 6, m, nb);
    const double* up = u + static_cast<size_t>(leaf) * NI;
    double        r[8];
#pragma unroll
    for (int z = 0; z < 8; ++z) r[z] = up[z * 64 + lane];
    const step_consts<3> C = leaf_consts<FROM, 3>(prm, table, who, lv);
    double               g[6];
    gather_ghosts_3d8(u, m, nb, hi3, lo3, true, true, g);
    const double gzm = g[0], gzp = g[1];
#pragma unroll
    for (int k = 0; k < 4; ++k) gface[k][lane] = g[2 + k];
    __syncthreads();
    const int y = hi3, x = lo3;
    double*   out = un + static_cast<size_t>(leaf) * NI;
    // z faces are evaluated once: the +z flux of cell z is the -z flux of z+1
    double fz = upwind_flux(gzm, r[0], C.vel[2], C.hs[2]);
#pragma unroll
    for (int z = 0; z < 8; ++z)
    {
        const double uc = r[z];
        const double xl = lane_minus1(uc);
        const double xr = lane_plus1(uc);
        const double yl = __shfl_up(uc, 8, 64);
        const double yr = __shfl_down(uc, 8, 64);
        const double lx = (x == 0) ? gface[2][z * 8 + y] : xl;
        const double hx = (x == 7) ? gface[3][z * 8 + y] : xr;
        const double ly = (y == 0) ? gface[0][z * 8 + x] : yl;
        const double hy = (y == 7) ? gface[1][z * 8 + x] : yr;
        const double hz = (z == 7) ? gzp : r[z < 7 ? z + 1 : 7];
        const double fzr = upwind_flux(uc, hz, C.vel[2], C.hs[2]);
        const double fL[3] = { upwind_flux(lx, uc, C.vel[0], C.hs[0]), upwind_flux(ly, uc, C.vel[1], C.hs[1]), fz };
        const double fR[3] = { upwind_flux(uc, hx, C.vel[0], C.hs[0]), upwind_flux(uc, hy, C.vel[1], C.hs[1]), fzr };
        store_cell<NT>(out + z * 64 + lane, update_from_fluxes<3>(uc, fL, fR, C.dtdx));
        fz = fzr;
    }
}

template <bool NT, int FROM>
__global__ __launch_bounds__(64) void k_step_3d8(const double* __restrict__ u, double* __restrict__ un,
                                                 const uint64_t* __restrict__ keys,
                                                 const face_link* __restrict__ links,
                                                 const uint32_t* __restrict__ metas, uint32_t nleaves, uint32_t walk, step_params prm,
    const step_params* __restrict__ table, const uint32_t* __restrict__ inst)
{
    const uint32_t leaf = sweep_item(blockIdx.x, walk);
    if (leaf >= nleaves) return;
    step_leaf_3d8<NT, FROM>(u, un, keys, links, metas, leaf, prm, table, inst);
}

// 3D 8^3 patches, one wave per run of same-level leaves along +x (leaf_run).
// The lane layout is k_step_3d8's.  Walking the run front to back, the -x
// ghosts of a leaf are the previous leaf's x = 7 column (left in LDS) and
// its +x ghosts the next leaf's x = 0 column (that leaf's interior is
// loaded before the current leaf is updated, so its loads overlap the
// update); only the run's two end faces are gathered from memory.  An x face
// touches every 64 B row of the neighbour patch, so this removes most of the
// ghost traffic that does not hit in L2.
template <bool NT, int FROM>
__global__ __launch_bounds__(64) void k_step_3d8_run(const double* __restrict__ u, double* __restrict__ un,
                                                     const uint64_t* __restrict__ keys,
                                                     const face_link* __restrict__ links,
                                                     const uint32_t* __restrict__ metas, uint32_t nruns, uint32_t walk, step_params prm,
    const step_params* __restrict__ table, const uint32_t* __restrict__ inst, const leaf_run* __restrict__ runs)
{
    constexpr int NI = 512;
    __shared__ double gface[4][64]; // -y, +y (index z*8+x), -x, +x (index z*8+y)
    const uint32_t r = sweep_item(blockIdx.x, walk);
    if (r >= nruns) return;
    const int      lane = threadIdx.x, hi3 = lane >> 3, lo3 = lane & 7;
    const int      y = hi3, x = lo3;
    const leaf_run run  = runs[r];
    uint32_t       leaf = run.head;
    double         cur[8], nxt[8];
    {
        const double* up = u + static_cast<size_t>(leaf) * NI;
#pragma unroll
        for (int z = 0; z < 8; ++z)
        {
            cur[z] = up[z * 64 + lane];
            nxt[z] = 0.0;
        }
    }
    for (uint32_t i = 0; i < run.len; ++i)
    {
        const face_link* L    = links + static_cast<size_t>(leaf) * 6;
        const uint32_t*  M    = metas + static_cast<size_t>(leaf) * 6;
        const bool       more = i + 1 < run.len;
        // ghosts of this leaf first, then the next leaf's interior, so that
        // the update below waits only for the ghosts
        const uint32_t who = leaf_instance<FROM>(inst, leaf);
        const int      lv  = key_level(keys[leaf]);
        uint32_t       m[6];
        int4           nb[6];
        load_faces<3>(L, M, m, nb);
        const step_consts<3> C = leaf_consts<FROM, 3>(prm, table, who, lv);
        double               g[6];
        gather_ghosts_3d8(u, m, nb, hi3, lo3, i == 0, !more, g);
        const double gzm = g[0], gzp = g[1];
        gface[0][lane]   = g[2];
        gface[1][lane]   = g[3];
        if (i == 0) gface[2][lane] = g[4];
        if (!more) gface[3][lane] = g[5];
        const uint32_t next = more ? static_cast<uint32_t>(L[5].ids[0]) : leaf;
        if (more)
        {
            const double* np = u + static_cast<size_t>(next) * NI;
#pragma unroll
            for (int z = 0; z < 8; ++z) nxt[z] = np[z * 64 + lane];
        }
        __syncthreads();
        double* out = un + static_cast<size_t>(leaf) * NI;
        double  fz  = upwind_flux(gzm, cur[0], C.vel[2], C.hs[2]); // z faces once
#pragma unroll
        for (int z = 0; z < 8; ++z)
        {
            const double uc = cur[z];
            const double xl = lane_minus1(uc);
            const double xr = lane_plus1(uc);
            const double yl = __shfl_up(uc, 8, 64);
            const double yr = __shfl_down(uc, 8, 64);
            const double xn = __shfl(nxt[z], lane & ~7, 64); // next leaf, x = 0, same (z, y)
            const double lx = (x == 0) ? gface[2][z * 8 + y] : xl;
            const double hx = (x == 7) ? (more ? xn : gface[3][z * 8 + y]) : xr;
            const double ly = (y == 0) ? gface[0][z * 8 + x] : yl;
            const double hy = (y == 7) ? gface[1][z * 8 + x] : yr;
            const double hz = (z == 7) ? gzp : cur[z < 7 ? z + 1 : 7];
            const double fzr = upwind_flux(uc, hz, C.vel[2], C.hs[2]);
            const double fL[3] = { upwind_flux(lx, uc, C.vel[0], C.hs[0]), upwind_flux(ly, uc, C.vel[1], C.hs[1]), fz };
            const double fR[3] = { upwind_flux(uc, hx, C.vel[0], C.hs[0]), upwind_flux(uc, hy, C.vel[1], C.hs[1]), fzr };
            store_cell<NT>(out + z * 64 + lane, update_from_fluxes<3>(uc, fL, fR, C.dtdx));
            fz = fzr;
        }
        __syncthreads();
        // this leaf's x = 7 column is the next leaf's -x ghost face
#pragma unroll
        for (int z = 0; z < 8; ++z)
        {
            if (x == 7) gface[2][z * 8 + y] = cur[z];
            cur[z] = nxt[z];
        }
        leaf = next;
        __syncthreads();
    }
}

// 2D 16^2 patches, one wave per leaf.  Lane l owns x = l % 16 of rows
// y = 4 (l / 16) .. 4 (l / 16) + 3; x-neighbours from lanes l -+ 1, the row
// above / below a lane's four from lanes l -+ 16; the four ghost faces are
// gathered one face cell per lane into 512 B of LDS.
template <bool NT, int FROM>
__device__ inline void step_leaf_2d16(const double* __restrict__ u, double* __restrict__ un,
                                      const uint64_t* __restrict__ keys, const face_link* __restrict__ links,
                                      const uint32_t* __restrict__ metas, uint32_t leaf, step_params const& prm,
                                      const step_params* __restrict__ table, const uint32_t* __restrict__ inst)
{
    constexpr int NI = 256;
    __shared__ double gface[4][16]; // -y, +y (index x), -x, +x (index y)
    const int      lane = threadIdx.x, x = lane & 15, q = lane >> 4;
    const uint32_t who  = leaf_instance<FROM>(inst, leaf);
    const int      lv   = key_level(keys[leaf]);
    uint32_t       m[4];
    int4           nb[4];
    load_faces<2>(links + static_cast<size_t>(leaf) * 4, metas + static_cast<size_t>(leaf) * 4, m, nb);
    const double* up = u + static_cast<size_t>(leaf) * NI;
    double        r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = up[(4 * q + j) * 16 + x];
    const step_consts<2> C = leaf_consts<FROM, 2>(prm, table, who, lv);
    // lane (q, x) gathers cell x of face q
    gface[q][x] = gather_ghost_2d16(u, m, nb, q, x);
    __syncthreads();
    const double above   = __shfl_up(r[3], 16, 64);  // row 4q - 1
    const double below   = __shfl_down(r[0], 16, 64); // row 4q + 4
    double*      out     = un + static_cast<size_t>(leaf) * NI;
    // y faces are evaluated once: the +y flux of row j is the -y flux of j+1
    double fy = upwind_flux((q == 0) ? gface[0][x] : above, r[0], C.vel[1], C.hs[1]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const int    y  = 4 * q + j;
        const double uc = r[j];
        const double xl = lane_minus1(uc);
        const double xr = lane_plus1(uc);
        const double lx = (x == 0) ? gface[2][y] : xl;
        const double hx = (x == 15) ? gface[3][y] : xr;
        const double hy = (j < 3) ? r[j < 3 ? j + 1 : 3] : ((q == 3) ? gface[1][x] : below);
        const double fyr   = upwind_flux(uc, hy, C.vel[1], C.hs[1]);
        const double fL[2] = { upwind_flux(lx, uc, C.vel[0], C.hs[0]), fy };
        const double fR[2] = { upwind_flux(uc, hx, C.vel[0], C.hs[0]), fyr };
        store_cell<NT>(out + y * 16 + x, update_from_fluxes<2>(uc, fL, fR, C.dtdx));
        fy = fyr;
    }
}

template <bool NT, int FROM>
__global__ __launch_bounds__(64) void k_step_2d16(const double* __restrict__ u, double* __restrict__ un,
                                                  const uint64_t* __restrict__ keys,
                                                  const face_link* __restrict__ links,
                                                  const uint32_t* __restrict__ metas, uint32_t nleaves, uint32_t walk, step_params prm,
    const step_params* __restrict__ table, const uint32_t* __restrict__ inst)
{
    const uint32_t leaf = sweep_item(blockIdx.x, walk);
    if (leaf >= nleaves) return;
    step_leaf_2d16<NT, FROM>(u, un, keys, links, metas, leaf, prm, table, inst);
}

// 2D 16^2 patches, one wave per run of same-level leaves along +x, the lane
// layout of k_step_2d16 and the hand-over of k_step_3d8_run: the -x ghosts
// of a leaf are the previous leaf's x = 15 column (left in LDS), its +x
// ghosts the next leaf's x = 0 column (registers of the prefetched leaf).
template <bool NT, int FROM>
__global__ __launch_bounds__(64) void k_step_2d16_run(const double* __restrict__ u, double* __restrict__ un,
                                                      const uint64_t* __restrict__ keys,
                                                      const face_link* __restrict__ links,
                                                      const uint32_t* __restrict__ metas, uint32_t nruns, uint32_t walk, step_params prm,
    const step_params* __restrict__ table, const uint32_t* __restrict__ inst, const leaf_run* __restrict__ runs)
{
    constexpr int NI = 256;
    __shared__ double gface[4][16]; // -y, +y (index x), -x, +x (index y)
    const uint32_t r = sweep_item(blockIdx.x, walk);
    if (r >= nruns) return;
    const int      lane = threadIdx.x, x = lane & 15, q = lane >> 4;
    const leaf_run run  = runs[r];
    uint32_t       leaf = run.head;
    double         cur[4], nxt[4];
    {
        const double* up = u + static_cast<size_t>(leaf) * NI;
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            cur[j] = up[(4 * q + j) * 16 + x];
            nxt[j] = 0.0;
        }
    }
    for (uint32_t i = 0; i < run.len; ++i)
    {
        const bool   more = i + 1 < run.len;
        const size_t e0   = static_cast<size_t>(leaf) * 4;
        // lanes of quarter q gather face q (y faces always, the run's end x faces)
        const uint32_t who = leaf_instance<FROM>(inst, leaf);
        const int      lv  = key_level(keys[leaf]);
        uint32_t       m[4];
        int4           nb[4];
        load_faces<2>(links + e0, metas + e0, m, nb);
        const step_consts<2> C = leaf_consts<FROM, 2>(prm, table, who, lv);
        if (q < 2 || (q == 2 && i == 0) || (q == 3 && !more)) gface[q][x] = gather_ghost_2d16(u, m, nb, q, x);
        const uint32_t next = more ? static_cast<uint32_t>(links[e0 + 3].ids[0]) : leaf;
        if (more)
        {
            const double* np = u + static_cast<size_t>(next) * NI;
#pragma unroll
            for (int j = 0; j < 4; ++j) nxt[j] = np[(4 * q + j) * 16 + x];
        }
        __syncthreads();
        const double       above   = __shfl_up(cur[3], 16, 64);  // row 4q - 1
        const double       below   = __shfl_down(cur[0], 16, 64); // row 4q + 4
        double*            out     = un + static_cast<size_t>(leaf) * NI;
        double             fy      = upwind_flux((q == 0) ? gface[0][x] : above, cur[0], C.vel[1], C.hs[1]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const int    y  = 4 * q + j;
            const double uc = cur[j];
            const double xl = lane_minus1(uc);
            const double xr = lane_plus1(uc);
            const double xn = __shfl(nxt[j], lane & ~15, 64); // next leaf, x = 0, same row
            const double lx = (x == 0) ? gface[2][y] : xl;
            const double hx = (x == 15) ? (more ? xn : gface[3][y]) : xr;
            const double hy = (j < 3) ? cur[j < 3 ? j + 1 : 3] : ((q == 3) ? gface[1][x] : below);
            const double fyr   = upwind_flux(uc, hy, C.vel[1], C.hs[1]);
            const double fL[2] = { upwind_flux(lx, uc, C.vel[0], C.hs[0]), fy };
            const double fR[2] = { upwind_flux(uc, hx, C.vel[0], C.hs[0]), fyr };
            store_cell<NT>(out + y * 16 + x, update_from_fluxes<2>(uc, fL, fR, C.dtdx));
            fy = fyr;
        }
        __syncthreads();
        // this leaf's x = 15 column is the next leaf's -x ghost face
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            if (x == 15) gface[2][4 * q + j] = cur[j];
            cur[j] = nxt[j];
        }
        leaf = next;
        __syncthreads();
    }
}

// Padded view with H ghost layers (the reference's patch after
// halo_exchange_update): interior copied, face halos gathered, corners 0.
template <int R, int N, int H, int NT>
__global__ __launch_bounds__(NT) void k_padded_view(const double* __restrict__ u, double* __restrict__ pad,
                                                    const face_link* __restrict__ links,
                                                    const uint32_t* __restrict__ metas, uint32_t nleaves)
{
    constexpr int  P    = N + 2 * H;
    constexpr int  FLAT = (R == 2) ? P * P : P * P * P;
    const uint32_t leaf = blockIdx.x;
    if (leaf >= nleaves) return;
    for (int i = threadIdx.x; i < FLAT; i += NT)
    {
        int kind;
        pad[static_cast<size_t>(leaf) * FLAT + i] = padded_value<R, N, H>(u, leaf, links, metas, i, &kind);
    }
}

template <int NT>
__device__ inline double block_max(double v, double* red)
{
    // each wave by shuffles, then the waves' values: one barrier
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
    for (int w = 1; w < NT / 64; ++w) v = fmax(v, red[w]);
    return v;
}

// Undivided-gradient criterion: one workgroup per leaf.
template <int R, int N, int NT>
__global__ __launch_bounds__(NT) void k_criterion_gradient(const double* __restrict__ u,
                                                           const uint64_t* __restrict__ keys,
                                                           const face_link* __restrict__ links,
                                                           const uint32_t* __restrict__ metas, double rthr,
                                                           double cthr, int min_level, int max_level,
                                                           int8_t* __restrict__ flags, uint32_t nleaves)
{
    using S = patch_shape<R, N>;
    __shared__ double tile[tile_shape<R, N>::TS];
    __shared__ double red[NT / 64];
    const uint32_t leaf = xcd_item(blockIdx.x, gridDim.x);
    if (leaf >= nleaves) return;
    const int lv = key_level(keys[leaf]);
    stage_tile<R, N, NT>(tile, u, leaf, links, metas);
    __syncthreads();
    double g = 0.0;
    for (int i = threadIdx.x; i < S::NI; i += NT) g = fmax(g, gradient_cell<R, N>(tile, i));
    g = block_max<NT>(g, red);
    if (threadIdx.x == 0) flags[leaf] = decide(g, lv, rthr, cthr, min_level, max_level);
}

// Face-halo cells of a patch with h ghost layers: h * face(dim) items per
// direction, direction after direction.
template <int R, class BX>
__host__ __device__ inline int halo_items(BX const& B, int h)
{
    int items = 0;
    for (int dir = 0; dir < box<R>::NDIR; ++dir) items += h * B.face(dir >> 1);
    return items;
}

// Halo item g (0 <= g < halo_items): its direction (returned) and its cell c
// in compact coordinates (layer `layer` beyond the face, tangential cells in
// row-major order).
template <int R, class BX>
__host__ __device__ inline int halo_item(BX const& B, int h, int g, int* c)
{
    int dir = 0, r = g;
    while (r >= h * B.face(dir >> 1))
    {
        r -= h * B.face(dir >> 1);
        ++dir;
    }
    const int dim = dir >> 1, fc = B.face(dim);
    int       layer = 0; // < h <= 8
    while (r >= fc)
    {
        r -= fc;
        ++layer;
    }
    for (int d = R - 1; d >= 0; --d)
    {
        if (d == dim) continue;
        const int q = B.quot(r, d);
        c[d]        = r - q * B.n(d);
        r           = q;
    }
    c[dim] = (dir & 1) ? B.n(dim) + layer : -1 - layer;
    return dir;
}

// Maximum over one leaf's interior and its h-deep face halos, starting from
// 0, reduced over the workgroup (every thread must call it): the interior
// with coalesced loads, then the face halos by the ghost rules (padded_value's
// cells of kind 0 and 1; the maximum is order-free).
template <int R, int NT, class BX>
__device__ inline double leaf_max_value(BX const& B, int h, const double* __restrict__ u, uint32_t leaf,
                                        const face_link* __restrict__ links, const uint32_t* __restrict__ metas,
                                        double* red)
{
    // the first cells of a thread are in flight while it follows its ghost's
    // record (with that, leaves kept to their XCD and a maximum of one barrier
    // instead of nine: 900 leaves of 64^2 on average 10.8 -> 7.4 us, of 32^2
    // 6.5 -> 5.1; the gradient criterion on 200 leaves of 16^2 4.4 -> 3.7)
    constexpr int CH = 16;
    double        m  = 0.0, r[CH];
    const int     ni = B.ni();
    const double* up = u + static_cast<size_t>(leaf) * ni;
#pragma unroll
    for (int k = 0; k < CH; ++k)
    {
        const int i = threadIdx.x + k * NT;
        r[k]        = i < ni ? up[i] : 0.0;
    }
    const int items = halo_items<R>(B, h);
    for (int g = threadIdx.x; g < items; g += NT)
    {
        int            c[R];
        const int      dir = halo_item<R>(B, h, g, c);
        const size_t   e   = static_cast<size_t>(leaf) * box<R>::NDIR + dir;
        m                  = fmax(m, ghost_value<R>(B, u, links[e], metas[e], dir, c));
    }
#pragma unroll
    for (int k = 0; k < CH; ++k) m = fmax(m, r[k]);
    for (int i = threadIdx.x + CH * NT; i < ni; i += NT) m = fmax(m, up[i]);
    return block_max<NT>(m, red);
}

// Maximum-value criterion over the interior and the H-deep face halos,
// starting from 0.
template <int R, int N, int H, int NT>
__global__ __launch_bounds__(NT) void k_criterion_max(const double* __restrict__ u,
                                                      const uint64_t* __restrict__ keys,
                                                      const face_link* __restrict__ links,
                                                      const uint32_t* __restrict__ metas, double rthr, double cthr,
                                                      int min_level, int max_level, int8_t* __restrict__ flags,
                                                      uint32_t nleaves)
{
    constexpr box<R>  B = box<R>::cube(N);
    __shared__ double red[NT / 64];
    const uint32_t    leaf = xcd_item(blockIdx.x, gridDim.x);
    if (leaf >= nleaves) return;
    const int lv = key_level(keys[leaf]);
    const double m = leaf_max_value<R, NT>(B, H, u, leaf, links, metas, red);
    if (threadIdx.x == 0) flags[leaf] = decide(m, lv, rthr, cthr, min_level, max_level);
}

// ---------------------------------------------------------------------------
// Kernels for patches of any shape (the box is a launch argument): one
// workgroup per leaf, neighbour cells read from memory -- the operands and
// expressions of the fixed-shape kernels, so the results are the same bits.
// ---------------------------------------------------------------------------

// One time step of patches of any shape whose tile fits in LDS, one workgroup
// per leaf.  Bound by the latency of its two dependent ghost loads and the
// index arithmetic of runtime extents, hence the column walk (one coordinate
// decomposition per thread) and the divisions by multiplication.  us per step
// against k_step_box on adapted trees: 2200 leaves of 12x10x6 12.9 for 26.6,
// 990 of 16^3 28 for 93, 10000 of 6^3 21 for 54, 2200 of 32^2 12.4 for 20.4.
template <int R, int NT, int CH, int FROM>
__global__ __launch_bounds__(NT) void k_step_box_tile(const double* __restrict__ u,
                                                      double* __restrict__ un, const uint64_t* __restrict__ keys,
                                                      const face_link* __restrict__ links,
                                                      const uint32_t* __restrict__ metas, uint32_t nleaves, uint32_t walk, launch_box<R, true> B, box_walk W, step_params prm,
    const step_params* __restrict__ table, const uint32_t* __restrict__ inst)
{
    HIP_DYNAMIC_SHARED(double, box_lds)
    const uint32_t leaf = sweep_item(blockIdx.x, walk);
    if (leaf >= nleaves) return;
    const uint32_t      who = leaf_instance<FROM>(inst, leaf);
    const int           lv  = key_level(keys[leaf]);
    const box_tile<R>   T(B);
    const box_column<R> col(B, T, W);
    stage_box<R, NT, 1, CH>(B, T, col, W, box_lds, u, 0, leaf, links, metas);
    const step_consts<R> C = leaf_consts<FROM, R>(prm, table, who, lv);
    __syncthreads();
    if (!col.on) return;
    double* out = un + static_cast<size_t>(leaf) * B.ni();
    for (int k = 0; col.z0 + k * col.dz < B.n(0); ++k)
        store_cell<false>(out + col.i0 + k * col.di,
                          upwind_tile_cell<R>(box_lds, T, col.t0 + k * col.dt, C.dtdx, C.vel, C.hs));
}

// Patches whose tile does not fit: neighbours from memory, each through its
// own dim's rule (neighbour_values), the fine cells of a ghost in flight
// together.  Bound by the latency of those loads: us per step on adapted
// trees, with one rule for every side -> by dim, 103 leaves of 90x88 53.2 ->
// 37.9, 155 of 20^3 91.3 -> 59.6, 1387 of 4x24x24 50.0 -> 33.2.
template <int R, int NT, int FROM>
__global__ __launch_bounds__(NT) void k_step_box(const double* __restrict__ u, double* __restrict__ un,
                                                 const uint64_t* __restrict__ keys,
                                                 const face_link* __restrict__ links,
                                                 const uint32_t* __restrict__ metas, uint32_t nleaves, uint32_t walk, launch_box<R> B, step_params prm,
    const step_params* __restrict__ table, const uint32_t* __restrict__ inst)
{
    const uint32_t leaf = sweep_item(blockIdx.x, walk);
    if (leaf >= nleaves) return;
    const step_consts<R> C = leaf_consts<FROM, R>(prm, table, leaf_instance<FROM>(inst, leaf), key_level(keys[leaf]));
    const int ni  = B.ni();
    double*   out = un + static_cast<size_t>(leaf) * ni;
    for (int i = threadIdx.x; i < ni; i += NT)
        out[i] = upwind_cell_direct<R>(B, u, leaf, links, metas, i, C.dtdx, C.vel, C.hs);
}

template <int R, int NT>
__global__ __launch_bounds__(NT) void k_padded_box(launch_box<R> B, int h, const double* __restrict__ u,
                                                   double* __restrict__ pad, const face_link* __restrict__ links,
                                                   const uint32_t* __restrict__ metas, uint32_t nleaves)
{
    const uint32_t leaf = blockIdx.x;
    if (leaf >= nleaves) return;
    const int flat = B.padded(h);
    for (int i = threadIdx.x; i < flat; i += NT)
    {
        int kind;
        pad[static_cast<size_t>(leaf) * flat + i] = padded_value<R>(B, h, u, leaf, links, metas, i, &kind);
    }
}

template <int R, int NT>
__global__ __launch_bounds__(NT) void k_criterion_gradient_box(launch_box<R> B, const double* __restrict__ u,
                                                               const uint64_t* __restrict__ keys,
                                                               const face_link* __restrict__ links,
                                                               const uint32_t* __restrict__ metas, double rthr,
                                                               double cthr, int min_level, int max_level,
                                                               int8_t* __restrict__ flags, uint32_t nleaves)
{
    __shared__ double red[NT / 64];
    const uint32_t    leaf = xcd_item(blockIdx.x, gridDim.x);
    if (leaf >= nleaves) return;
    const int lv = key_level(keys[leaf]);
    double    g  = 0.0;
    const int ni = B.ni();
    for (int i = threadIdx.x; i < ni; i += NT) g = fmax(g, gradient_cell_direct<R>(B, u, leaf, links, metas, i));
    g = block_max<NT>(g, red);
    if (threadIdx.x == 0) flags[leaf] = decide(g, lv, rthr, cthr, min_level, max_level);
}

template <int R, int NT>
__global__ __launch_bounds__(NT) void k_criterion_max_box(launch_box<R> B, int h, const double* __restrict__ u,
                                                          const uint64_t* __restrict__ keys,
                                                          const face_link* __restrict__ links,
                                                          const uint32_t* __restrict__ metas, double rthr, double cthr,
                                                          int min_level, int max_level, int8_t* __restrict__ flags,
                                                          uint32_t nleaves)
{
    __shared__ double red[NT / 64];
    const uint32_t    leaf = xcd_item(blockIdx.x, gridDim.x);
    if (leaf >= nleaves) return;
    const int lv = key_level(keys[leaf]);
    const double m = leaf_max_value<R, NT>(B, h, u, leaf, links, metas, red);
    if (threadIdx.x == 0) flags[leaf] = decide(m, lv, rthr, cthr, min_level, max_level);
}

} // namespace amrhip
