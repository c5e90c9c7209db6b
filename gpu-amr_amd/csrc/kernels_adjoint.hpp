// kernels_adjoint.hpp -- discrete adjoint of the advection step, the halo
// fill and the regrid transfer (their exact transposes), in gather form so
// that every sum has a fixed order and no atomics are needed.
//
// For fixed topology, velocity v and dt, one step is linear:
//   u' = u - sum_d dt/dx_d [ F(u, u_R) - F(u_L, u) ],
//   F(a, b) = 0.5 (a v + b v) - 0.5 |v| (b - a) = vp a + vm b,
//   vp = 0.5 (v + |v|), vm = 0.5 (v - |v|),
// so  du'/du = 1 - sum_d dt/dx_d |v_d|,  du'/du_L = dt/dx vp,
//     du'/du_R = -dt/dx vm,
// and du'/dv_d = -dt/dx_d [ G(u, u_R) - G(u_L, u) ],
//     G(a, b) = 0.5 (a + b) - 0.5 sgn(v_d) (b - a)
// (dt held fixed).  Ghosts are linear in the neighbours' interiors:
// same = copy, coarser = injection, finer = mean of 2^R fine cells.  Their
// transposes: a cell copied into a same-level neighbour's ghost receives that
// ghost's adjoint; a cell injected into finer neighbours' ghosts receives the
// sum of their adjoints; a cell averaged into a coarser neighbour's ghost
// receives 1/2^R of it.  The adjoint of a ghost is the coefficient with
// which the neighbour's boundary cell reads it, times that cell's lambda'.
//
// One adjoint step is one launch over the leaves of the step's topology
// (k_adj_step): lambda = A^T lambda' with the transposed halo gathered from
// the neighbours' boundary layers of lambda', plus the per-leaf partial sums
// of lambda' . du'/dv.  A regrid transfer is transposed by k_adj_regrid.
#pragma once

#include "device_common.hpp"
#include "kernels_step.hpp"

#pragma clang fp contract(off)

namespace amrhip
{

// Per-launch adjoint constants: dt/dx per level and dimension, vp, vm and
// sgn(v) per dimension.
struct adjoint_params
{
    double dtdx[kMaxLevels][3];
    double vp[3];
    double vm[3];
    double sgn[3];
};

// In-patch part of (A^T lambda')_c.
template <int R, class BX>
__host__ __device__ inline double adj_interior(BX const& B, const double* __restrict__ lam, int i,
                                               const double* dtdx, const double* vp, const double* vm)
{
    int c[R];
    B.coords(i, c);
    double diag = 1.0;
    for (int d = 0; d < R; ++d) diag -= dtdx[d] * (vp[d] - vm[d]);
    double acc = diag * lam[i];
    for (int d = 0; d < R; ++d)
    {
        const int j = R - 1 - d; // layout dim of physical axis d
        const int s = B.stride(j);
        if (c[j] + 1 < B.n(j)) acc += (dtdx[d] * vp[d]) * lam[i + s]; // c is u_L of c + e_d
        if (c[j] - 1 >= 0) acc -= (dtdx[d] * vm[d]) * lam[i - s];     // c is u_R of c - e_d
    }
    return acc;
}

template <int R, int N>
__host__ __device__ inline double adj_interior(const double* __restrict__ lam, int i, const double* dtdx,
                                               const double* vp, const double* vm)
{
    constexpr box<R> B = box<R>::cube(N);
    return adj_interior<R>(B, lam, i, dtdx, vp, vm);
}

// Transposed halo term for the leaf's boundary cells facing direction dir at
// tangential layout coordinates c (c[dim] ignored), from the neighbours'
// lambda'.  It is added to the depth-0 cell, and for a coarser neighbour also
// to the depth-1 cell (both are averaged into the same coarse ghost).
//   same    : the neighbour reads our cell as its ghost on side dir^1;
//   finer   : the 2^(R-1) fine ghost cells injected from our cell;
//   coarser : the coarse ghost cell that averages our cell, / 2^R.
// The neighbour's boundary cell reads its ghost on side dir^1 with
// coefficient dt/dx vp (ghost is its u_L, dir positive) or -dt/dx vm (ghost
// is its u_R, dir negative), at the neighbour's own level.
template <int R, class BX>
__host__ __device__ inline double adj_face_term(BX const& B, const double* __restrict__ lam, const face_link& L,
                                                uint32_t meta, int dir, const int* c, int level,
                                                const adjoint_params& prm)
{
    const int  dim = dir >> 1;
    const bool pos = (dir & 1) != 0;
    const int  d   = R - 1 - dim;
    const int  nb  = pos ? 0 : B.n(dim) - 1; // the neighbour's layer that touches us
    switch (rel_of(meta))
    {
        case REL_SAME:
        {
            int cc[R];
            for (int k = 0; k < R; ++k) cc[k] = (k == dim) ? nb : c[k];
            const double coef = pos ? (prm.dtdx[level][d] * prm.vp[d]) : -(prm.dtdx[level][d] * prm.vm[d]);
            return coef * lam[static_cast<size_t>(L.ids[0]) * B.ni() + B.lin(cc)];
        }
        case REL_FINER:
        {
            int kid = 0, bit = 0, base[R];
            for (int k = 0; k < R; ++k)
            {
                if (k == dim)
                {
                    base[k] = nb;
                    continue;
                }
                kid |= B.half_of(c[k], k) << bit;
                ++bit;
                base[k] = B.fine(c[k], k);
            }
            const double* q   = lam + static_cast<size_t>(L.ids[kid]) * B.ni();
            double        sum = 0.0;
            for (int o = 0; o < box<R>::K; ++o)
            {
                int cc[R], b = 0;
                for (int k = 0; k < R; ++k)
                {
                    if (k == dim)
                    {
                        cc[k] = base[k];
                        continue;
                    }
                    cc[k] = base[k] + ((o >> (R - 2 - b)) & 1);
                    ++b;
                }
                sum += q[B.lin(cc)];
            }
            const double coef =
                pos ? (prm.dtdx[level + 1][d] * prm.vp[d]) : -(prm.dtdx[level + 1][d] * prm.vm[d]);
            return coef * sum;
        }
        case REL_COARSER:
        {
            int cc[R];
            for (int k = 0; k < R; ++k)
                cc[k] = (k == dim) ? nb : static_cast<int>(quad_of(meta, k)) * B.half(k) + c[k] / 2;
            const double coef =
                pos ? (prm.dtdx[level - 1][d] * prm.vp[d]) : -(prm.dtdx[level - 1][d] * prm.vm[d]);
            return coef * lam[static_cast<size_t>(L.ids[0]) * B.ni() + B.lin(cc)] / static_cast<double>(box<R>::F);
        }
        default: return 0.0;
    }
}

template <int R, int N>
__host__ __device__ inline double adj_face_term(const double* __restrict__ lam, const face_link& L, uint32_t meta,
                                                int dir, const int* c, int level, const adjoint_params& prm)
{
    constexpr box<R> B = box<R>::cube(N);
    return adj_face_term<R>(B, lam, L, meta, dir, c, level, prm);
}

// G-form contribution of a cell to lambda' . du'/dv along physical axis d,
// from its value and its two neighbours.
__host__ __device__ inline double adj_velocity_term(double uc, double ul, double ur, double lam_c, double dtdx,
                                                    double sgn)
{
    const double gR = 0.5 * (uc + ur) - 0.5 * sgn * (ur - uc);
    const double gL = 0.5 * (ul + uc) - 0.5 * sgn * (uc - ul);
    return lam_c * (-dtdx * (gR - gL));
}

// Contribution of cell i to lambda' . du'/dv, from the staged u tile (with
// the ghost layer).
template <int R, int N>
__host__ __device__ inline void adj_velocity_cell(const double* tile, int i, double lam_c, const double* dtdx,
                                                  const double* sgn, double* acc)
{
    using T = tile_shape<R, N>;
    int c[R];
    patch_shape<R, N>::coords(i, c);
    const int    t  = T::idx(c);
    const double uc = tile[t];
    for (int d = 0; d < R; ++d)
    {
        const int s = T::stride(R - 1 - d);
        acc[d] += adj_velocity_term(uc, tile[t - s], tile[t + s], lam_c, dtdx[d], sgn[d]);
    }
}

// adj_velocity_cell with the neighbours read from memory (any patch shape).
template <int R, class BX>
__host__ __device__ inline void adj_velocity_cell_direct(BX const& B, const double* __restrict__ u, uint32_t leaf,
                                                         const face_link* __restrict__ links,
                                                         const uint32_t* __restrict__ metas, int i, double lam_c,
                                                         const double* dtdx, const double* sgn, double* acc)
{
    int c[R];
    B.coords(i, c);
    const double uc = u[static_cast<size_t>(leaf) * B.ni() + i];
    for (int d = 0; d < R; ++d)
    {
        const int j = R - 1 - d;
        c[j] -= 1;
        const double ul = cell_or_ghost<R>(B, u, leaf, links, metas, c);
        c[j] += 2;
        const double ur = cell_or_ghost<R>(B, u, leaf, links, metas, c);
        c[j] -= 1;
        acc[d] += adj_velocity_term(uc, ul, ur, lam_c, dtdx[d], sgn[d]);
    }
}

// Face index of tangential coordinates c (dims other than dim), row-major.
template <int R, class BX>
__host__ __device__ inline int face_index(BX const& B, const int* c, int dim)
{
    int f = 0;
    for (int k = 0; k < R; ++k)
        if (k != dim) f = f * B.n(k) + c[k];
    return f;
}

template <int R, int N>
__host__ __device__ inline int face_index(const int* c, int dim)
{
    constexpr box<R> B = box<R>::cube(N);
    return face_index<R>(B, c, dim);
}

// Tangential coordinates of face index f of direction dir (c[dim] = 0).
template <int R, class BX>
__host__ __device__ inline void face_coords(BX const& B, int f, int dir, int* c)
{
    const int dim = dir >> 1;
    for (int k = R - 1; k >= 0; --k)
    {
        if (k == dim)
        {
            c[k] = 0;
            continue;
        }
        const int q = B.quot(f, k);
        c[k]        = f - q * B.n(k);
        f           = q;
    }
}

template <int R, int N>
__host__ __device__ inline void face_coords(int f, int dir, int* c)
{
    constexpr box<R> B = box<R>::cube(N);
    face_coords<R>(B, f, dir, c);
}

// lambda_c = (A^T lambda')_c + transposed halo terms h[dir][face] of the
// directions whose boundary band holds c.
template <int R, int N>
__host__ __device__ inline double adj_cell(const double* __restrict__ lam, const double* __restrict__ h,
                                           const uint32_t* __restrict__ M, int i, const double* dtdx,
                                           const double* vp, const double* vm)
{
    using S    = patch_shape<R, N>;
    double acc = adj_interior<R, N>(lam, i, dtdx, vp, vm);
    int    c[R];
    S::coords(i, c);
    for (int dir = 0; dir < S::NDIR; ++dir)
    {
        const int dim   = dir >> 1;
        const int depth = (dir & 1) ? (N - 1 - c[dim]) : c[dim];
        if (depth == 0 || (depth == 1 && rel_of(M[dir]) == REL_COARSER))
            acc += h[dir * S::FACE + face_index<R, N>(c, dim)];
    }
    return acc;
}

// adj_cell with lambda' and the transposed halo terms read from memory (any
// patch shape; the terms are added in adj_cell's order, so the same bits).
template <int R, class BX>
__host__ __device__ inline double adj_cell_direct(BX const& B, const double* __restrict__ lam_next, uint32_t leaf,
                                                  const face_link* __restrict__ L, const uint32_t* __restrict__ M,
                                                  int i, int level, const adjoint_params& prm, const double* dtdx,
                                                  const double* vp, const double* vm)
{
    double acc = adj_interior<R>(B, lam_next + static_cast<size_t>(leaf) * B.ni(), i, dtdx, vp, vm);
    int    c[R];
    B.coords(i, c);
    for (int dir = 0; dir < box<R>::NDIR; ++dir)
    {
        const int dim   = dir >> 1;
        const int depth = (dir & 1) ? (B.n(dim) - 1 - c[dim]) : c[dim];
        if (depth == 0 || (depth == 1 && rel_of(M[dir]) == REL_COARSER))
            acc += adj_face_term<R>(B, lam_next, L[dir], M[dir], dir, c, level, prm);
    }
    return acc;
}

// Transposed regrid transfer, value of cell t of old leaf i.
// Refined leaf: sum of lambda over the 2^R fine cells injected from t.
template <int R, class BX>
__host__ __device__ inline double adj_refine_value(BX const& B, const double* __restrict__ lam_new,
                                                   uint32_t first_child, int t)
{
    int tc[R], base[R], kid = 0;
    B.coords(t, tc);
    for (int d = 0; d < R; ++d)
    {
        kid |= B.half_of(tc[d], d) << (R - 1 - d);
        base[d] = B.fine(tc[d], d);
    }
    const double* q   = lam_new + static_cast<size_t>(first_child + kid) * B.ni();
    double        sum = 0.0;
    for (int off = 0; off < box<R>::F; ++off)
    {
        int cc[R];
        for (int d = 0; d < R; ++d) cc[d] = base[d] + ((off >> (R - 1 - d)) & 1);
        sum += q[B.lin(cc)];
    }
    return sum;
}

// Coarsened family: cell f of child kid receives lambda of the parent cell
// that averaged it, divided by 2^R.
template <int R, class BX>
__host__ __device__ inline double adj_restrict_value(BX const& B, const double* __restrict__ lam_parent, int kid,
                                                     int f)
{
    int fc[R], t[R];
    B.coords(f, fc);
    for (int d = 0; d < R; ++d) t[d] = ((kid >> (R - 1 - d)) & 1) * B.half(d) + fc[d] / 2;
    return lam_parent[B.lin(t)] / static_cast<double>(box<R>::F);
}

template <int R, int N>
__host__ __device__ inline double adj_refine_value(const double* __restrict__ lam_new, uint32_t first_child, int t)
{
    constexpr box<R> B = box<R>::cube(N);
    return adj_refine_value<R>(B, lam_new, first_child, t);
}

template <int R, int N>
__host__ __device__ inline double adj_restrict_value(const double* __restrict__ lam_parent, int kid, int f)
{
    constexpr box<R> B = box<R>::cube(N);
    return adj_restrict_value<R>(B, lam_parent, kid, f);
}

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

// One adjoint step, one workgroup per leaf: lam = transpose(step)(lam_next)
// and vpart[leaf][d] = sum over the leaf's cells of lam_next . du'/dv_d.  u
// is the state the forward step started from; the step's constants are read
// from prm_p (device memory, so a captured launch picks up new values).
template <int R, int N, int NT>
__global__ __launch_bounds__(NT) void k_adj_step(const double* __restrict__ lam_next, const double* __restrict__ u,
                                                 const uint64_t* __restrict__ keys,
                                                 const face_link* __restrict__ links,
                                                 const uint32_t* __restrict__ metas,
                                                 const adjoint_params* __restrict__ prm_p, double* __restrict__ lam,
                                                 double* __restrict__ vpart, uint32_t nleaves)
{
    const adjoint_params& prm = *prm_p;
    using S = patch_shape<R, N>;
    __shared__ double tile[tile_shape<R, N>::TS];
    __shared__ double lt[S::NI];
    __shared__ double h[S::NDIR * S::FACE];
    constexpr int     NW = NT / 64;
    static_assert(NT % 64 == 0, "whole waves");
    __shared__ double red[R][NW];
    const uint32_t leaf = blockIdx.x;
    if (leaf >= nleaves) return;
    const face_link* L  = links + static_cast<size_t>(leaf) * S::NDIR;
    const uint32_t*  M  = metas + static_cast<size_t>(leaf) * S::NDIR;
    const int        lv = key_level(keys[leaf]);
    stage_tile<R, N, NT>(tile, u, leaf, links, metas);
    const double* lp = lam_next + static_cast<size_t>(leaf) * S::NI;
    for (int i = threadIdx.x; i < S::NI; i += NT) lt[i] = lp[i];
    // The face terms start half a workgroup away from the ghost gather of
    // stage_tile (which starts at thread 0), so that their two dependent
    // load chains run on different waves.
    for (int g = (threadIdx.x + NT / 2) % NT; g < S::NDIR * S::FACE; g += NT)
    {
        const int dir = g / S::FACE;
        int       c[R];
        face_coords<R, N>(g % S::FACE, dir, c);
        h[g] = adj_face_term<R, N>(lam_next, L[dir], M[dir], dir, c, lv, prm);
    }
    __syncthreads();
    double dtdx[R], vp[R], vm[R], sgn[R], acc[R];
    for (int d = 0; d < R; ++d)
    {
        dtdx[d] = prm.dtdx[lv][d];
        vp[d]   = prm.vp[d];
        vm[d]   = prm.vm[d];
        sgn[d]  = prm.sgn[d];
        acc[d]  = 0.0;
    }
    double* out = lam + static_cast<size_t>(leaf) * S::NI;
    for (int i = threadIdx.x; i < S::NI; i += NT)
    {
        out[i] = adj_cell<R, N>(lt, h, M, i, dtdx, vp, vm);
        adj_velocity_cell<R, N>(tile, i, lt[i], dtdx, sgn, acc);
    }
    // fixed-order reduction of the velocity partials: a shuffle tree inside
    // each wave, then the waves' sums in wave order
    for (int d = 0; d < R; ++d)
        for (int o = 32; o > 0; o >>= 1) acc[d] += __shfl_down(acc[d], o, 64);
    if ((threadIdx.x & 63) == 0)
        for (int d = 0; d < R; ++d) red[d][threadIdx.x >> 6] = acc[d];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int d = 0; d < 3; ++d)
        {
            double sum = 0.0;
            if (d < R)
            {
                sum = red[d][0];
                for (int w = 1; w < NW; ++w) sum += red[d][w];
            }
            vpart[static_cast<size_t>(leaf) * 3 + d] = sum;
        }
}

// ---------------------------------------------------------------------------
// One wave per leaf for the configurations' patches (3D 8^3, 2D 16^2): the
// step kernels' lane layouts, lambda' and u in registers, lambda's halo terms
// and u's ghosts through LDS.  A ghost of u and the transposed halo term of
// the same face cell come from the same neighbour cell, so one address serves
// both loads.  Operands and sums are k_adj_step's in its order, so the same
// bits.
//
// Bound by the chain face records -> neighbour cells -> store; the LDS-tile
// kernel walked it once per face through a switch on the relation, and spent
// most of its instructions on indexes and on 6 R shuffles per wave of the
// velocity sums.  us a launch, LDS tile -> one wave: 16^2, 214 adapted leaves
// (launch and latency) 5.35 -> 3.94; 8^3, 4096 leaves (three passes over
// 16.8 MB, 7.2 us at the copy rate) 28.8 -> 16.1.
// ---------------------------------------------------------------------------

// The level at whose dt/dx the neighbour across a face reads its ghost.
__device__ inline int face_level(uint32_t meta, int lv)
{
    return lv + (rel_of(meta) == REL_FINER ? 1 : 0) - (rel_of(meta) == REL_COARSER ? 1 : 0);
}

// lambda' summed over the four fine cells across face cell c of direction DIR
// (adj_face_term's finer rule).
template <int DIR>
__device__ inline double fine_sum_3d8(const double* __restrict__ lam, int4 nb, const int* c)
{
    constexpr box<3> B   = box<3>::cube(8);
    constexpr int    dim = DIR >> 1;
    int              k = 0, bit = 0, cc[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        cc[d] = (d == dim) ? ((DIR & 1) ? 0 : 7) : B.fine(c[d], d);
        if (d != dim)
        {
            k |= B.half_of(c[d], d) << bit;
            ++bit;
        }
    }
    const int32_t slot = (k & 2) ? ((k & 1) ? nb.w : nb.z) : ((k & 1) ? nb.y : nb.x);
    const double* q    = lam + static_cast<size_t>(slot) * B.ni() + B.lin(cc);
    constexpr int s1   = dim == 0 ? 8 : 64, s2 = dim == 2 ? 8 : 1; // strides of the two tangential dims
    double        f[4];
#pragma unroll
    for (int o = 0; o < 4; ++o) f[o] = q[(o >> 1) * s1 + (o & 1) * s2];
    double sum = 0.0;
#pragma unroll
    for (int o = 0; o < 4; ++o) sum += f[o];
    return sum;
}

// a + b where the lane adds the value N lanes further within its row of 16
// (rotated): with N = 8, 4, 2, 1 in turn every lane holds the row's sum in
// the order of a shuffle-down tree.
template <int N>
__device__ inline double row_rotate_add(double v)
{
    const uint64_t b  = __builtin_bit_cast(uint64_t, v);
    const int      lo = static_cast<int>(b), hi = static_cast<int>(b >> 32);
    const int      l  = __builtin_amdgcn_update_dpp(0, lo, 0x120 + N, 0xF, 0xF, true); // row_ror:N
    const int      h  = __builtin_amdgcn_update_dpp(0, hi, 0x120 + N, 0xF, 0xF, true);
    return v + __builtin_bit_cast(double, (static_cast<uint64_t>(static_cast<uint32_t>(h)) << 32) |
                                              static_cast<uint32_t>(l));
}

__device__ inline double row_sum(double v)
{
    return row_rotate_add<1>(row_rotate_add<2>(row_rotate_add<4>(row_rotate_add<8>(v))));
}

// One level of a tree sum of two values at once: of a over the lanes without
// the WIDTH bit and of b over those with it, each with its partner WIDTH lanes
// away (WIDTH = 32 or 16).
template <int WIDTH>
__device__ inline double fold_pair(double a, double b)
{
    const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
    uint32_t       p[2], q[2];
#pragma unroll
    for (int w = 0; w < 2; ++w)
    {
        const uint32_t xw = static_cast<uint32_t>(x >> (32 * w)), yw = static_cast<uint32_t>(y >> (32 * w));
        if constexpr (WIDTH == 32)
        {
            const auto r = __builtin_amdgcn_permlane32_swap(xw, yw, false, false);
            p[w] = r[0];
            q[w] = r[1];
        }
        else
        {
            const auto r = __builtin_amdgcn_permlane16_swap(xw, yw, false, false);
            p[w] = r[0];
            q[w] = r[1];
        }
    }
    return __builtin_bit_cast(double, (static_cast<uint64_t>(p[1]) << 32) | p[0]) +
           __builtin_bit_cast(double, (static_cast<uint64_t>(q[1]) << 32) | q[0]);
}

// The sums of the four rows of 16 lanes (uniform in each row), in row order.
__device__ inline double rows_in_order(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    double         r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(b), 16 * k);
        const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(b >> 32), 16 * k);
        r[k]              = __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
    }
    return ((r[0] + r[1]) + r[2]) + r[3];
}

// A leaf's adjoint constants: own-level coefficients of lambda's neighbours
// (ap along +, am along -), of the cell itself (diag), dt/dx and sgn(v).
template <int R>
struct adj_consts
{
    double ap[R], am[R], dtdx[R], sgn[R], diag;

    __device__ adj_consts(adjoint_params const& prm, int lv)
    {
        diag = 1.0;
#pragma unroll
        for (int d = 0; d < R; ++d)
        {
            dtdx[d] = prm.dtdx[lv][d];
            sgn[d]  = prm.sgn[d];
            ap[d]   = dtdx[d] * prm.vp[d];
            am[d]   = dtdx[d] * prm.vm[d];
            diag -= dtdx[d] * (prm.vp[d] - prm.vm[d]);
        }
    }
};

// 3D 8^3: lane l owns the z-column at (y, x) = (l / 8, l % 8).
__device__ inline void adj_leaf_3d8(const double* __restrict__ lam_next, const double* __restrict__ u,
                                    const uint64_t* __restrict__ keys, const face_link* __restrict__ links,
                                    const uint32_t* __restrict__ metas, const adjoint_params* __restrict__ prm_p,
                                    double* __restrict__ lam, double* __restrict__ vpart, uint32_t leaf)
{
    constexpr int     NI = 512;
    __shared__ double gface[4][64]; // ghosts of u: -y, +y (index z*8+x), -x, +x (index z*8+y)
    __shared__ double hface[4][64]; // halo terms of lambda on the same faces
    const int lane = threadIdx.x, hi3 = lane >> 3, lo3 = lane & 7;
    const int lv   = key_level(keys[leaf]);
    uint32_t  m[6];
    int4      nb[6];
    load_faces<3>(links + static_cast<size_t>(leaf) * 6, metas + static_cast<size_t>(leaf) * 6, m, nb);
    const double* lp = lam_next + static_cast<size_t>(leaf) * NI;
    const double* up = u + static_cast<size_t>(leaf) * NI;
    double        l[8], r[8];
#pragma unroll
    for (int z = 0; z < 8; ++z) l[z] = lp[z * 64 + lane];
#pragma unroll
    for (int z = 0; z < 8; ++z) r[z] = up[z * 64 + lane];
    const adjoint_params& prm = *prm_p;
    const adj_consts<3>   C(prm, lv);
    const int cf[6][3] = { { -1, hi3, lo3 }, { 8, hi3, lo3 }, { hi3, -1, lo3 },
                           { hi3, 8, lo3 },  { hi3, lo3, -1 }, { hi3, lo3, 8 } };
    double    g[6], h[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
    {
        const size_t src = ghost_source<3, 8>(nb[k].x, m[k], k, cf[k]);
        g[k]             = u[src];
        h[k]             = lam_next[src];
    }
    if (!single_cell_ghosts<3>(m))
    {
        auto fine = [&](auto dir) {
            constexpr int K = decltype(dir)::value;
            if (rel_of(m[K]) != REL_FINER) return;
            g[K] = fine_mean_3d8<K>(u, nb[K], cf[K]);
            h[K] = fine_sum_3d8<K>(lam_next, nb[K], cf[K]);
        };
        fine(std::integral_constant<int, 0>{});
        fine(std::integral_constant<int, 1>{});
        fine(std::integral_constant<int, 2>{});
        fine(std::integral_constant<int, 3>{});
        fine(std::integral_constant<int, 4>{});
        fine(std::integral_constant<int, 5>{});
    }
    bool coarse[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
    {
        const int    d    = 2 - (k >> 1);
        const double dtdx = prm.dtdx[face_level(m[k], lv)][d];
        coarse[k]         = rel_of(m[k]) == REL_COARSER;
        h[k]              = ((k & 1) ? dtdx * prm.vp[d] : -(dtdx * prm.vm[d])) * h[k] * (coarse[k] ? 0.125 : 1.0);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        gface[k][lane] = g[2 + k];
        hface[k][lane] = h[2 + k];
    }
    __syncthreads();
    const int y = hi3, x = lo3;
    // the cells that a face's halo term reaches: the boundary layer and, next
    // to a coarser neighbour, the one behind it
    const bool ym = y == 0 || (y == 1 && coarse[2]), yp = y == 7 || (y == 6 && coarse[3]);
    const bool xm = x == 0 || (x == 1 && coarse[4]), xp = x == 7 || (x == 6 && coarse[5]);
    double     va[4][3] = {}; // k_adj_step's thread (z % 4, lane) sums its two cells
    double*    out      = lam + static_cast<size_t>(leaf) * NI;
#pragma unroll
    for (int z = 0; z < 8; ++z)
    {
        const double lc = l[z], uc = r[z];
        const double lxp = lane_plus1(lc), lxm = lane_minus1(lc);
        const double lyp = __shfl_down(lc, 8, 64), lym = __shfl_up(lc, 8, 64);
        double       acc = C.diag * lc, t;
        t                = acc + C.ap[0] * lxp;
        acc              = x < 7 ? t : acc;
        t                = acc - C.am[0] * lxm;
        acc              = x > 0 ? t : acc;
        t                = acc + C.ap[1] * lyp;
        acc              = y < 7 ? t : acc;
        t                = acc - C.am[1] * lym;
        acc              = y > 0 ? t : acc;
        if (z < 7) acc += C.ap[2] * l[z < 7 ? z + 1 : 7];
        if (z > 0) acc -= C.am[2] * l[z > 0 ? z - 1 : 0];
        if (z == 0 || (z == 1 && coarse[0])) acc += h[0];
        if (z == 7 || (z == 6 && coarse[1])) acc += h[1];
        t   = acc + hface[0][z * 8 + x];
        acc = ym ? t : acc;
        t   = acc + hface[1][z * 8 + x];
        acc = yp ? t : acc;
        t   = acc + hface[2][z * 8 + y];
        acc = xm ? t : acc;
        t   = acc + hface[3][z * 8 + y];
        acc = xp ? t : acc;
        store_cell<false>(out + z * 64 + lane, acc);
        const double uxm = lane_minus1(uc), uxp = lane_plus1(uc);
        const double uym = __shfl_up(uc, 8, 64), uyp = __shfl_down(uc, 8, 64);
        const double lx = x == 0 ? gface[2][z * 8 + y] : uxm, hx = x == 7 ? gface[3][z * 8 + y] : uxp;
        const double ly = y == 0 ? gface[0][z * 8 + x] : uym, hy = y == 7 ? gface[1][z * 8 + x] : uyp;
        const double lz = z == 0 ? g[0] : r[z > 0 ? z - 1 : 0], hz = z == 7 ? g[1] : r[z < 7 ? z + 1 : 7];
        va[z & 3][0] += adj_velocity_term(uc, lx, hx, lc, C.dtdx[0], C.sgn[0]);
        va[z & 3][1] += adj_velocity_term(uc, ly, hy, lc, C.dtdx[1], C.sgn[1]);
        va[z & 3][2] += adj_velocity_term(uc, lz, hz, lc, C.dtdx[2], C.sgn[2]);
    }
    // the tree of k_adj_step's four waves, all twelve sums at once: lanes 32
    // apart (waves 0, 1 and 2, 3 together), lanes 16 apart (row w then holds
    // wave w), each row, and the rows in order
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        const double s02 = fold_pair<32>(va[0][d], va[2][d]), s13 = fold_pair<32>(va[1][d], va[3][d]);
        const double sum = rows_in_order(row_sum(fold_pair<16>(s02, s13)));
        if (lane == 0) vpart[static_cast<size_t>(leaf) * 3 + d] = sum;
    }
}

// 2D 16^2: lane (q, x) owns x of rows 4q .. 4q + 3 and gathers cell x of
// face q.
__device__ inline void adj_leaf_2d16(const double* __restrict__ lam_next, const double* __restrict__ u,
                                    const uint64_t* __restrict__ keys, const face_link* __restrict__ links,
                                    const uint32_t* __restrict__ metas, const adjoint_params* __restrict__ prm_p,
                                    double* __restrict__ lam, double* __restrict__ vpart, uint32_t leaf)
{
    constexpr int     NI = 256;
    __shared__ double gface[4][16]; // ghosts of u: -y, +y (index x), -x, +x (index y)
    __shared__ double hface[4][16]; // halo terms of lambda
    const int lane = threadIdx.x, x = lane & 15, q = lane >> 4;
    const int lv   = key_level(keys[leaf]);
    uint32_t  m[4];
    int4      nb[4];
    load_faces<2>(links + static_cast<size_t>(leaf) * 4, metas + static_cast<size_t>(leaf) * 4, m, nb);
    const double* lp = lam_next + static_cast<size_t>(leaf) * NI;
    const double* up = u + static_cast<size_t>(leaf) * NI;
    double        l[4], r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) l[j] = lp[(4 * q + j) * 16 + x];
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = up[(4 * q + j) * 16 + x];
    const adjoint_params& prm = *prm_p;
    const adj_consts<2>   C(prm, lv);
    ghost_cells_2d16      cells(m, nb, q, x);
    double                ug, hg;
    if (single_cell_ghosts<2>(m))
    {
        ug = u[cells.first];
        hg = lam_next[cells.first];
    }
    else
    {
        // the two fine cells that touch the face: the layer of the 2 x 2
        // block on our side, along the face
        const bool   along_x = q < 2, far = (q & 1) == 0;
        const size_t t0 = cells.first + (cells.finer && far ? (along_x ? 16 : 1) : 0);
        const size_t t1 = t0 + (cells.finer ? (along_x ? 1 : 16) : 0);
        const double h0 = lam_next[t0], h1 = lam_next[t1];
        ug              = cells.value(u);
        hg              = cells.finer ? (0.0 + h0) + h1 : h0;
    }
    bool   coarse[4];
    double dtf = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        coarse[k]      = rel_of(m[k]) == REL_COARSER;
        const double f = prm.dtdx[face_level(m[k], lv)][1 - (k >> 1)];
        dtf            = q == k ? f : dtf;
    }
    const double vf = q == 0 ? -prm.vm[1] : q == 1 ? prm.vp[1] : q == 2 ? -prm.vm[0] : prm.vp[0];
    const bool   cq = q == 0 ? coarse[0] : q == 1 ? coarse[1] : q == 2 ? coarse[2] : coarse[3];
    gface[q][x]     = ug;
    hface[q][x]     = (dtf * vf) * hg * (cq ? 0.25 : 1.0);
    __syncthreads();
    const double lup = __shfl_up(l[3], 16, 64), ldn = __shfl_down(l[0], 16, 64); // rows 4q - 1, 4q + 4
    const double uup = __shfl_up(r[3], 16, 64), udn = __shfl_down(r[0], 16, 64);
    const bool   xm = x == 0 || (x == 1 && coarse[2]), xp = x == 15 || (x == 14 && coarse[3]);
    double       va[4][2];
    double*      out = lam + static_cast<size_t>(leaf) * NI;
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        const int    y  = 4 * q + j;
        const double lc = l[j], uc = r[j];
        const double lxp = lane_plus1(lc), lxm = lane_minus1(lc);
        const double lyp = j < 3 ? l[j < 3 ? j + 1 : 3] : ldn, lym = j > 0 ? l[j > 0 ? j - 1 : 0] : lup;
        double       acc = C.diag * lc, t;
        t                = acc + C.ap[0] * lxp;
        acc              = x < 15 ? t : acc;
        t                = acc - C.am[0] * lxm;
        acc              = x > 0 ? t : acc;
        t                = acc + C.ap[1] * lyp;
        acc              = y < 15 ? t : acc;
        t                = acc - C.am[1] * lym;
        acc              = y > 0 ? t : acc;
        if (j < 2)
        {
            t   = acc + hface[0][x];
            acc = q == 0 && (j == 0 || coarse[0]) ? t : acc;
        }
        if (j > 1)
        {
            t   = acc + hface[1][x];
            acc = q == 3 && (j == 3 || coarse[1]) ? t : acc;
        }
        t   = acc + hface[2][y];
        acc = xm ? t : acc;
        t   = acc + hface[3][y];
        acc = xp ? t : acc;
        store_cell<false>(out + y * 16 + x, acc);
        const double uxm = lane_minus1(uc), uxp = lane_plus1(uc);
        const double lx = x == 0 ? gface[2][y] : uxm, hx = x == 15 ? gface[3][y] : uxp;
        const double ly = j > 0 ? r[j > 0 ? j - 1 : 0] : (q == 0 ? gface[0][x] : uup);
        const double hy = j < 3 ? r[j < 3 ? j + 1 : 3] : (q == 3 ? gface[1][x] : udn);
        va[j][0]        = 0.0 + adj_velocity_term(uc, lx, hx, lc, C.dtdx[0], C.sgn[0]);
        va[j][1]        = 0.0 + adj_velocity_term(uc, ly, hy, lc, C.dtdx[1], C.sgn[1]);
    }
    // the tree of k_adj_step's four waves (wave q held rows 4q .. 4q + 3):
    // lanes 32 and 16 apart were rows 2 and 1 apart
#pragma unroll
    for (int d = 0; d < 2; ++d)
    {
        const double sum = rows_in_order(row_sum((va[0][d] + va[2][d]) + (va[1][d] + va[3][d])));
        if (lane == 0) vpart[static_cast<size_t>(leaf) * 3 + d] = sum;
    }
    if (lane == 0) vpart[static_cast<size_t>(leaf) * 3 + 2] = 0.0;
}

__global__ __launch_bounds__(64) void k_adj_step_3d8(const double* __restrict__ lam_next, const double* __restrict__ u,
                                                     const uint64_t* __restrict__ keys,
                                                     const face_link* __restrict__ links,
                                                     const uint32_t* __restrict__ metas,
                                                     const adjoint_params* __restrict__ prm_p,
                                                     double* __restrict__ lam, uint32_t nleaves, uint32_t walk,
                                                     double* __restrict__ vpart)
{
    const uint32_t leaf = sweep_item(blockIdx.x, walk);
    if (leaf < nleaves) adj_leaf_3d8(lam_next, u, keys, links, metas, prm_p, lam, vpart, leaf);
}

// A forward step that shares an adjoint step's launch.
struct forward_args
{
    const double*      u;
    double*            un;
    const uint64_t*    keys;
    const face_link*   links;
    const uint32_t*    metas;
    const step_params* table;
    uint32_t           nleaves, walk;
};

// One adjoint step by the first adj_blocks workgroups and, by the others, one
// forward step of another topology: the recomputation of the segment before,
// independent of it.  Alone either leaves most of the GPU idle on the trees of
// a few hundred leaves that a 2D gradient steps on; together they take one
// launch (300 steps with 285 recomputed, levels 3 to 6: 3150 -> 2570 us a
// forward and backward pass; on two branches of the captured graph instead:
// 3110).  For 8^3 patches the pair takes 162 registers and the GPU is busier:
// 4096 leaves 526 -> 597 us, 512 leaves unchanged, so 3D keeps to itself.
__global__ __launch_bounds__(64) void k_adj_step_2d16(const double* __restrict__ lam_next,
                                                      const double* __restrict__ u, const uint64_t* __restrict__ keys,
                                                      const face_link* __restrict__ links,
                                                      const uint32_t* __restrict__ metas,
                                                      const adjoint_params* __restrict__ prm_p,
                                                      double* __restrict__ lam, uint32_t nleaves, uint32_t walk,
                                                      uint32_t adj_blocks, double* __restrict__ vpart, forward_args F)
{
    // both grids are multiples of kXcds, so a workgroup keeps its XCD
    if (blockIdx.x < adj_blocks)
    {
        const uint32_t leaf = sweep_item(blockIdx.x, walk);
        if (leaf < nleaves) adj_leaf_2d16(lam_next, u, keys, links, metas, prm_p, lam, vpart, leaf);
        return;
    }
    const uint32_t leaf = sweep_item(blockIdx.x - adj_blocks, F.walk);
    if (leaf >= F.nleaves) return;
    step_leaf_2d16<false, FROM_TABLE>(F.u, F.un, F.keys, F.links, F.metas, leaf, step_params{}, F.table, nullptr);
}

// Transposed regrid transfer of old leaf i (one workgroup; mark / head /
// counts / pos recorded by the forward regrid).
template <int R, int NT, class BX>
__device__ inline void adj_regrid_leaf(BX const& B, const double* __restrict__ lam_new,
                                       const uint8_t* __restrict__ mark, const uint8_t* __restrict__ head,
                                       const uint32_t* __restrict__ counts, const uint32_t* __restrict__ pos,
                                       double* __restrict__ lam_old, uint32_t i)
{
    if (counts[i] == 0) return;
    const int      ni  = B.ni();
    const uint32_t dst = pos[i];
    double*        out = lam_old + static_cast<size_t>(i) * ni;
    if (mark[i])
    {
        for (int t = threadIdx.x; t < ni; t += NT) out[t] = adj_refine_value<R>(B, lam_new, dst, t);
    }
    else if (head[i])
    {
        const double* par = lam_new + static_cast<size_t>(dst) * ni;
        for (int kid = 0; kid < box<R>::F; ++kid)
            for (int f = threadIdx.x; f < ni; f += NT)
                lam_old[static_cast<size_t>(i + kid) * ni + f] = adj_restrict_value<R>(B, par, kid, f);
    }
    else
    {
        const double* src = lam_new + static_cast<size_t>(dst) * ni;
        for (int t = threadIdx.x; t < ni; t += NT) out[t] = src[t];
    }
}

// Transposed regrid transfer, one workgroup per leaf before the regrid.
template <int R, int N, int NT>
__global__ __launch_bounds__(NT) void k_adj_regrid(const double* __restrict__ lam_new, const uint8_t* __restrict__ mark,
                                                   const uint8_t* __restrict__ head,
                                                   const uint32_t* __restrict__ counts,
                                                   const uint32_t* __restrict__ pos, double* __restrict__ lam_old,
                                                   uint32_t n_old)
{
    constexpr box<R> B = box<R>::cube(N);
    const uint32_t   i = blockIdx.x;
    if (i >= n_old) return;
    adj_regrid_leaf<R, NT>(B, lam_new, mark, head, counts, pos, lam_old, i);
}

// k_adj_regrid for patches of any shape.
template <int R, int NT>
__global__ __launch_bounds__(NT) void k_adj_regrid_box(launch_box<R> B, const double* __restrict__ lam_new,
                                                       const uint8_t* __restrict__ mark,
                                                       const uint8_t* __restrict__ head,
                                                       const uint32_t* __restrict__ counts,
                                                       const uint32_t* __restrict__ pos, double* __restrict__ lam_old,
                                                       uint32_t n_old)
{
    const uint32_t i = blockIdx.x;
    if (i >= n_old) return;
    adj_regrid_leaf<R, NT>(B, lam_new, mark, head, counts, pos, lam_old, i);
}

// k_adj_step for patches of any shape: lambda', u and the transposed halo
// terms read from memory (the operands and sums of k_adj_step).
template <int R, int NT>
__global__ __launch_bounds__(NT) void k_adj_step_box(launch_box<R> B, const double* __restrict__ lam_next,
                                                     const double* __restrict__ u, const uint64_t* __restrict__ keys,
                                                     const face_link* __restrict__ links,
                                                     const uint32_t* __restrict__ metas,
                                                     const adjoint_params* __restrict__ prm_p,
                                                     double* __restrict__ lam, double* __restrict__ vpart,
                                                     uint32_t nleaves)
{
    const adjoint_params& prm = *prm_p;
    constexpr int NW = NT / 64;
    static_assert(NT % 64 == 0, "whole waves");
    __shared__ double red[R][NW];
    const uint32_t    leaf = blockIdx.x;
    if (leaf >= nleaves) return;
    const face_link* L  = links + static_cast<size_t>(leaf) * box<R>::NDIR;
    const uint32_t*  M  = metas + static_cast<size_t>(leaf) * box<R>::NDIR;
    const int        lv = key_level(keys[leaf]);
    double           dtdx[R], vp[R], vm[R], sgn[R], acc[R];
    for (int d = 0; d < R; ++d)
    {
        dtdx[d] = prm.dtdx[lv][d];
        vp[d]   = prm.vp[d];
        vm[d]   = prm.vm[d];
        sgn[d]  = prm.sgn[d];
        acc[d]  = 0.0;
    }
    const int     ni  = B.ni();
    const double* lp  = lam_next + static_cast<size_t>(leaf) * ni;
    double*       out = lam + static_cast<size_t>(leaf) * ni;
    for (int i = threadIdx.x; i < ni; i += NT)
    {
        out[i] = adj_cell_direct<R>(B, lam_next, leaf, L, M, i, lv, prm, dtdx, vp, vm);
        adj_velocity_cell_direct<R>(B, u, leaf, links, metas, i, lp[i], dtdx, sgn, acc);
    }
    // the velocity partials reduced as in k_adj_step
    for (int d = 0; d < R; ++d)
        for (int o = 32; o > 0; o >>= 1) acc[d] += __shfl_down(acc[d], o, 64);
    if ((threadIdx.x & 63) == 0)
        for (int d = 0; d < R; ++d) red[d][threadIdx.x >> 6] = acc[d];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int d = 0; d < 3; ++d)
        {
            double sum = 0.0;
            if (d < R)
            {
                sum = red[d][0];
                for (int w = 1; w < NW; ++w) sum += red[d][w];
            }
            vpart[static_cast<size_t>(leaf) * 3 + d] = sum;
        }
}

// k_adj_step_box for patches whose two tiles fit in LDS: u with its ghosts,
// and lambda' with the transposed halo term of each ghost cell in that cell's
// place.  A cell then reads its neighbours from LDS instead of walking the
// face records of up to 4 R of them.  Cells per thread, sums and their order
// as in k_adj_step_box.  Bound by latency on the trees that a gradient steps
// on.  us of a 60-step forward and backward pass, from memory -> tiles: 67
// leaves of 32^2 1847 -> 1207, 331 of 12x8 1105 -> 877, 435 of 6^3 1664 ->
// 1203.
template <int R, int NT>
__global__ __launch_bounds__(NT) void k_adj_step_box_tile(const double* __restrict__ lam_next,
                                                          const double* __restrict__ u,
                                                          const uint64_t* __restrict__ keys,
                                                          const face_link* __restrict__ links,
                                                          const uint32_t* __restrict__ metas,
                                                          const adjoint_params* __restrict__ prm_p,
                                                          double* __restrict__ lam, uint32_t nleaves, uint32_t walk,
                                                          launch_box<R, true> B, double* __restrict__ vpart)
{
    constexpr int NW = NT / 64;
    __shared__ double red[R][NW];
    HIP_DYNAMIC_SHARED(double, lds)
    const uint32_t leaf = sweep_item(blockIdx.x, walk);
    if (leaf >= nleaves) return;
    const adjoint_params& prm = *prm_p;
    const face_link*  L  = links + static_cast<size_t>(leaf) * box<R>::NDIR;
    const uint32_t*   M  = metas + static_cast<size_t>(leaf) * box<R>::NDIR;
    const int         lv = key_level(keys[leaf]), ni = B.ni(), tid = threadIdx.x;
    const box_tile<R> T(B);
    double *          ut = lds, *lt = lds + box_tile<R>::cells(B);
    const double*     up = u + static_cast<size_t>(leaf) * ni;
    const double*     lp = lam_next + static_cast<size_t>(leaf) * ni;
    for (int i = tid; i < ni; i += NT)
    {
        int c[R];
        B.coords(i, c);
        const int t = T.idx(c);
        ut[t]       = up[i];
        lt[t]       = lp[i];
    }
    // the ghosts of each pair of faces, the pairs starting on different waves
    auto ghosts = [&](auto dim) {
        constexpr int D     = decltype(dim)::value;
        constexpr int shift = (D * NT / R) / 64 * 64;
        for (int q = (tid + NT - shift) % NT; q < 2 * B.face(D); q += NT)
        {
            int       c[R];
            const int side = face_pair_item<R, D>(B, q, c), dir = 2 * D + side;
            const int t    = T.idx(c);
            double    g;
            face_values<R, 1, D>(B, u, 0, link_ids(L + dir), M[dir], side, c, &g);
            ut[t] = g;
            c[D]  = 0;
            lt[t] = adj_face_term<R>(B, lam_next, L[dir], M[dir], dir, c, lv, prm);
        }
    };
    ghosts(std::integral_constant<int, 0>{});
    ghosts(std::integral_constant<int, 1>{});
    if constexpr (R == 3) ghosts(std::integral_constant<int, 2>{});
    const adj_consts<R> C(prm, lv);
    bool                coarse[2 * R];
    for (int k = 0; k < 2 * R; ++k) coarse[k] = rel_of(M[k]) == REL_COARSER;
    double acc_v[R];
    for (int d = 0; d < R; ++d) acc_v[d] = 0.0;
    __syncthreads();
    double* out = lam + static_cast<size_t>(leaf) * ni;
    for (int i = tid; i < ni; i += NT)
    {
        int c[R];
        B.coords(i, c);
        const int    t  = T.idx(c);
        const double lc = lt[t], uc = ut[t];
        double       acc = C.diag * lc;
#pragma unroll
        for (int d = 0; d < R; ++d)
        {
            const int    j = R - 1 - d, s = T.st[j]; // layout dim of physical axis d
            const double hi = lt[t + s], lo = lt[t - s];
            if (c[j] + 1 < B.n(j)) acc += C.ap[d] * hi;
            if (c[j] - 1 >= 0) acc -= C.am[d] * lo;
        }
#pragma unroll
        for (int dir = 0; dir < 2 * R; ++dir)
        {
            const int j = dir >> 1, depth = (dir & 1) ? B.n(j) - 1 - c[j] : c[j];
            if (depth == 0 || (depth == 1 && coarse[dir]))
                acc += lt[t + ((dir & 1) ? T.st[j] : -T.st[j]) * (depth + 1)];
        }
        store_cell<false>(out + i, acc);
#pragma unroll
        for (int d = 0; d < R; ++d)
        {
            const int s = T.st[R - 1 - d];
            acc_v[d] += adj_velocity_term(uc, ut[t - s], ut[t + s], lc, C.dtdx[d], C.sgn[d]);
        }
    }
    for (int d = 0; d < R; ++d)
        for (int o = 32; o > 0; o >>= 1) acc_v[d] += __shfl_down(acc_v[d], o, 64);
    if ((tid & 63) == 0)
        for (int d = 0; d < R; ++d) red[d][tid >> 6] = acc_v[d];
    __syncthreads();
    if (tid == 0)
        for (int d = 0; d < 3; ++d)
        {
            double sum = 0.0;
            if (d < R)
            {
                sum = red[d][0];
                for (int w = 1; w < NW; ++w) sum += red[d][w];
            }
            vpart[static_cast<size_t>(leaf) * 3 + d] = sum;
        }
}

// The velocity partials of a run of adjoint steps, one workgroup per step:
// step first + b wrote its leaves' triples at vpart + b * stride * 3 (leaves[]
// per step); they are summed in one fixed order (leaves t, t + 256, ... per
// thread, a shuffle tree inside each wave, the waves in order) into that
// step's slot of step_sums.
__global__ __launch_bounds__(256) void k_sum3_steps(const double* __restrict__ vpart, uint64_t stride,
                                                    const uint32_t* __restrict__ leaves, uint64_t first,
                                                    double* __restrict__ step_sums)
{
    __shared__ double red[3][4];
    const uint64_t    step = first + blockIdx.x;
    const uint32_t    n    = leaves[step];
    const double*     v    = vpart + blockIdx.x * stride * 3;
    double            s[3] = { 0.0, 0.0, 0.0 };
    for (uint32_t l = threadIdx.x; l < n; l += 256)
        for (int d = 0; d < 3; ++d) s[d] += v[static_cast<size_t>(l) * 3 + d];
    for (int d = 0; d < 3; ++d)
        for (int o = 32; o > 0; o >>= 1) s[d] += __shfl_down(s[d], o, 64);
    if ((threadIdx.x & 63) == 0)
        for (int d = 0; d < 3; ++d) red[d][threadIdx.x >> 6] = s[d];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int d = 0; d < 3; ++d) step_sums[step * 3 + d] = ((red[d][0] + red[d][1]) + red[d][2]) + red[d][3];
}

// Deterministic sum of `count` triples: stage 1 gives each of kReduceBlocks
// workgroups a fixed contiguous chunk, stage 2 adds the chunk sums in order
// into acc.
constexpr int kReduceBlocks = 64;

__device__ inline void block_sum3(double* s, double (*red)[256])
{
    for (int d = 0; d < 3; ++d) red[d][threadIdx.x] = s[d];
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1)
    {
        if (static_cast<int>(threadIdx.x) < k)
            for (int d = 0; d < 3; ++d) red[d][threadIdx.x] += red[d][threadIdx.x + k];
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void k_sum3_chunks(const double* __restrict__ v, uint64_t count,
                                                     double* __restrict__ chunk_sums)
{
    __shared__ double red[3][256];
    const uint64_t    per = (count + kReduceBlocks - 1) / kReduceBlocks;
    const uint64_t    b0  = blockIdx.x * per;
    const uint64_t    b1  = b0 + per < count ? b0 + per : count;
    double            s[3] = { 0.0, 0.0, 0.0 };
    for (uint64_t l = b0 + threadIdx.x; l < b1; l += 256)
        for (int d = 0; d < 3; ++d) s[d] += v[l * 3 + d];
    block_sum3(s, red);
    if (threadIdx.x == 0)
        for (int d = 0; d < 3; ++d) chunk_sums[blockIdx.x * 3 + d] = red[d][0];
}

__global__ __launch_bounds__(256) void k_sum3_final(const double* __restrict__ chunk_sums, double* __restrict__ acc)
{
    __shared__ double red[3][256];
    double            s[3] = { 0.0, 0.0, 0.0 };
    if (threadIdx.x < kReduceBlocks)
        for (int d = 0; d < 3; ++d) s[d] = chunk_sums[threadIdx.x * 3 + d];
    block_sum3(s, red);
    if (threadIdx.x == 0)
        for (int d = 0; d < 3; ++d) acc[d] = red[d][0];
}

} // namespace amrhip
