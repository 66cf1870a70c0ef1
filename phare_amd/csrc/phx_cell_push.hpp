// phx_cell_push.hpp -- the fused push + deposit over cell-ordered segmented storage in 2D and 3D, shared
// by the FP64 and the mixed-precision family: the particles of one cell deposit together on the matrix
// cores (phx_cell_deposit.hpp), E and B are gathered from a stage in LDS.
#pragma once

#include "phx_cell_deposit.hpp"

#include <mutex>

namespace phx
{
namespace pc
{
// the cell-grouped push, per dimension and order: work-items of a workgroup, waves per SIMD the
// register allocation targets (what a workgroup's LDS leaves room for), and whether the next row is
// loaded while a row is worked on. In 3D order 1 runs best on many waves without the prefetch's
// registers (58x47x52 cells, 50 particles per cell: 0.243 ms for mode domain_only, against 0.259 with
// two workgroups of 256 and the prefetch); at order 2 two workgroups of 256 fit a CU (64^3 cells, 64
// per cell: 0.95 ms; 1.09 with one of 512); at order 3 the larger stage leaves room for one
// workgroup, of 512 (36x41x30 cells, 32 per cell: 0.207 ms, 0.260 with 256).
// FP32 in 3D: the stage and the buffers take half the LDS and the row half the registers, 256 fit at every
// order (PPC step, order 3: 0.54 ms against 0.63 with 512; order 1: 0.61 and 0.64; order 2: 1.87 and 1.88)
// In 2D four workgroups of 256 fit a CU (256x128 cells, 100 per cell, order 2: 0.093 ms after a sort,
// growing to 0.17 over 25 steps, as drifted particles make more and smaller groups: LDS instructions 3.9 to
// 7.0 million, conflicts 4 to 13 % of the LDS cycles, LDS and vector units below half busy throughout; one
// particle per lane into the tile, in columns, took 0.137)
constexpr int cellBlock(bool fp32, int dim, int order)
{
    return fp32 || dim == 2 || order == 2 ? 256 : 512;
}
template<class X, int D, int O>
struct CellCfg
{
    static constexpr bool FP32     = sizeof(typename X::Real) == 4;
    static constexpr int BLOCK     = cellBlock(FP32, D, O);
    static constexpr int WAVES     = D == 2 || (O == 1 && !FP32) ? 4 : 2;
    static constexpr bool PREFETCH = FP32 || D == 2 || O != 1;
    static constexpr int NW        = BLOCK / LANES;
    // particles listed for the one-by-one push between two passes over the rows (every wavefront
    // that finds room for a workgroup's particles may add its row)
    static constexpr unsigned int LIST = 2 * BLOCK;
};
// the smallest group of lanes of one cell (of the 32 of a half row) that deposits on the matrix cores (one
// lane deposits by itself), and the smallest that moves the accumulated window to its cell: 4, 8 and 16
// lanes are within 1 % of each other at orders 2 and 3 in 2D and 3D; 16 is slower at order 1 in 2D (190x150
// cells, 16 per cell: 157 us per PPC step, 129 with 8 and with 4; 100 per cell 264, 248 and 258)
constexpr int CELL_GROUP = 2;
constexpr int CELL_MOVE  = 8;
constexpr unsigned long long CUS = 256; // compute units of the GPU
// most LDS of a workgroup's tile, stage and buffers
constexpr unsigned int CELL_LDS_MAX = 131072;
// nodes of a cell's gather stencils: the first, relative to the cell, and how many; the stage holds
// them for the segment's cells and those one cell around it
constexpr int cellGatherLo(int order) { return order == 3 ? -2 : -1; }
constexpr int cellGatherNodes(int order) { return order == 1 ? 3 : (order == 2 ? 4 : 5); }
// pitch of the stage's last direction for segments of at most cellFixed cells along it, odd so that
// stencils of different cells start in different banks
constexpr int cellFixed(int dim) { return dim == 2 ? 32 : 4; }
constexpr int cellExt(int dim, int order) { return cellFixed(dim) + 1 + cellGatherNodes(order); }

// the fields of one particle read from its slot (cell[0] is DEAD_CELL for an empty slot)
template<int D, class R = double>
struct Part
{
    int cell[D];
    R delta[D], v[3], w, q;
};

// LDS view of the tile: moment slab (m, copy)
struct TileView
{
    double* lds;
    int org[3];
    int ext[3];
    int pitch[3];
    int copies, stride;
    // slab of moment m (n, rho, Fx, Fy, Fz); RN: the tile leaves the charge density (m = 1) out
    template<bool RN = false>
    __device__ double* mom(int m, int copy) const
    {
        return lds + ((RN && m > 1 ? m - 1 : m) * copies + copy) * stride;
    }
    __device__ int node(int i, int j, int k) const { return (i * pitch[1] + j) * pitch[2] + k; }
    // the O+1 nodes from start lie in the tile along d
    template<int O>
    __device__ bool holds(int d, int start) const
    {
        return start >= org[d] && start + O < org[d] + ext[d];
    }
};

template<bool RN = false, int TB = BLOCK>
__device__ __forceinline__ void zeroTile(double* lds, TileSpec const& S)
{
    for (int x = threadIdx.x; x < (RN ? 4 : 5) * S.copies * S.stride; x += TB)
        lds[x] = 0.;
}

// flush the tile: the copies of each node summed, one HBM atomic per touched node and moment;
// RN: the charge density is the population's charge times n
template<int D, bool RN = false, int TB = BLOCK>
__device__ __forceinline__ void flushTile(Geom const& G, TileView const& T, int nodes,
                                          double* const* mom, double charge = 0.)
{
    int const e12 = T.pitch[1] * T.pitch[2];
    for (int x = threadIdx.x; x < nodes; x += TB)
    {
        int node = -1;
#pragma unroll
        for (int m = 0; m < 5; ++m)
        {
            double val = 0.;
            if (RN && m == 1)
            {
                for (int c = 0; c < T.copies; ++c)
                    val += T.mom<RN>(0, c)[x];
                val *= charge;
            }
            else
                for (int c = 0; c < T.copies; ++c)
                    val += T.mom<RN>(m, c)[x];
            if (val != 0.)
            {
                if (node < 0)
                {
                    int const ti = x / e12;
                    int const r  = x - ti * e12;
                    int const tj = r / T.pitch[2];
                    int const tk = r - tj * T.pitch[2];
                    node = G.idx(QMOM, T.org[0] + ti, D > 1 ? T.org[1] + tj : 0,
                                 D > 2 ? T.org[2] + tk : 0);
                }
                atomicAdd(mom[m] + node, val);
            }
        }
    }
}

__device__ __forceinline__ void tileView(TileView& T, double* lds, TileSpec const& S)
{
    T.lds    = lds;
    T.copies = S.copies;
    T.stride = S.stride;
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        T.ext[d]   = S.ext[d];
        T.pitch[d] = S.pitch[d];
        T.org[d] = 0;
    }
}

// address of a row of one particle component, kept in scalar registers (the lane is the offset of
// the access; folded into a per-lane base the ten components took 20 vector registers)
template<class R>
using GlobalPtr = __attribute__((address_space(1))) R*;
template<class R>
__device__ __forceinline__ GlobalPtr<R> rowOf(R* p, unsigned long long row)
{
    GlobalPtr<R> q = (GlobalPtr<R>)(p + row);
    asm volatile("" : "+s"(q));
    return q;
}

// one row of the segment: the particles of 64 consecutive slots
template<int D, bool RN, class R>
__device__ __forceinline__ void loadRow(PViewT<R> const& in, unsigned long long row, unsigned int lane, Part<D, R>& p)
{
#pragma unroll
    for (int d = 0; d < D; ++d)
        p.cell[d] = rowOf(in.ic[d], row)[lane];
#pragma unroll
    for (int d = 0; d < D; ++d)
        p.delta[d] = rowOf(in.de[d], row)[lane];
#pragma unroll
    for (int d = 0; d < 3; ++d)
        p.v[d] = rowOf(in.v[d], row)[lane];
    p.w = rowOf(in.w, row)[lane];
    if constexpr (!RN)
        p.q = rowOf(in.q, row)[lane];
}

template<class X>
struct CellArgs
{
    PushArgs A;
    PViewT<typename X::Real> v;
};

// the kernel's arguments, read again from the argument segment: a use after a long stretch of code
// reloads what it needs instead of holding registers over it
template<class X>
__device__ __forceinline__ CellArgs<X> const& cellArgs()
{
    auto* p = (__attribute__((address_space(4))) char const*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(CellArgs<X> const*)p;
}

// E and B of the segment's surroundings in LDS: component f (Ex .. Bz) on `nodes` nodes from `org`,
// row-major, e1 and e2 nodes along the second and third direction (e1 in 2D); nodes beyond a
// component's array repeat its last ones (no stencil inside the domain reaches them)
template<class X, int D, int TB>
__device__ __forceinline__ void stageFields(PushArgs const& A, typename X::Real* em, int const* org, int e1, int e2,
                                            int nodes)
{
    Geom const& G = A.G;
    int const e12 = D == 3 ? e1 * e2 : e1;
    for (int x = threadIdx.x; x < nodes; x += TB)
    {
        int const i = x / e12, r = x - i * e12;
        int const j = D == 3 ? r / e2 : r, k = D == 3 ? r - j * e2 : 0;
#pragma unroll
        for (int f = 0; f < 6; ++f)
        {
            int const q    = f < 3 ? QEX + f : QBX + f - 3;
            int const n[3] = {org[0] + i, org[1] + j, D == 3 ? org[2] + k : 0};
            int c[3]       = {0, 0, 0};
#pragma unroll
            for (int d = 0; d < D; ++d)
                c[d] = min(max(n[d], 0), G.shape[q][d] - 1);
            em[f * nodes + x] = X::field(A, f)[G.idx(q, c[0], c[1], c[2])];
        }
    }
}

// E and B at a particle from the staged fields; rel: its cell less the stage's first node
template<class X, int D, int O, class R>
__device__ __forceinline__ void gatherStaged(R const* em, int e1, int e2, int nodes, int const* rel,
                                             R const* delta, R* E, R* B)
{
    constexpr int S  = O + 1;
    constexpr int SZ = D == 3 ? S : 1;
    R w[2][D][S];
    int st[2][D];
#pragma unroll
    for (int d = 0; d < D; ++d)
    {
        st[CP][d] = rel[d] - splineStencil<O>(CP, delta[d], w[CP][d]);
        st[CD][d] = rel[d] - splineStencil<O>(CD, delta[d], w[CD][d]);
    }
#pragma unroll
    for (int f = 0; f < 6; ++f)
    {
        int const q  = f < 3 ? QEX + f : QBX + f - 3;
        int const cx = centering(q, 0), cy = centering(q, 1), cz = centering(q, 2);
        int const at = st[cx][0] * e1 + st[cy][1];
        R const* const p = em + f * nodes + (D == 3 ? at * e2 + st[cz][D - 1] : at);
        R r = 0;
#pragma unroll
        for (int i = 0; i < S; ++i)
        {
            R y = 0;
#pragma unroll
            for (int j = 0; j < S; ++j)
            {
                if constexpr (D == 3)
                {
                    R z = 0;
#pragma unroll
                    for (int k = 0; k < SZ; ++k)
                        z = X::fma(p[(i * e1 + j) * e2 + k], w[cz][D - 1][k], z);
                    y = X::fma(z, w[cy][1][j], y);
                }
                else
                    y = X::fma(p[i * e1 + j], w[cy][1][j], y);
            }
            r = X::fma(y, w[cx][0][i], r);
        }
        (f < 3 ? E[f] : B[f - 3]) = r;
    }
}
} // namespace pc

// ---------------------------------------------------------------------------------------------
// fused push + deposit over cell-ordered segmented storage, A.split workgroups per segment in 3D, one
// per work item in 2D (segments of 4x4x4 and 2x32 cells): the rows of a segment hold its particles in cell
// order, each wavefront takes a run of them, and the particles of one cell deposit together on the matrix
// cores (phx_cell_deposit.hpp). The gather and the weights use fused multiply-adds: a velocity differs from
// the reference's in its last digits (1e-16 of it), where the one-by-one push below and the linear one
// keep the reference's operations bit for bit. The tile covers the segment with the stencil and one cell of motion on
// each side, and E and B of the segment's surroundings are staged beside it. A particle that leaves
// the domain, the tile or the stage is left as it is and noted in a list in LDS; the listed
// particles of the whole workgroup are pushed 64 to a wavefront, gathering from HBM, and deposit one
// by one, into the tile or straight into HBM (the overflow segment, number nsegs, has no tile). RN:
// the population has one charge: the particles' own is not read, and the tile leaves the charge
// density out, its flush taking the charge times n.
// ---------------------------------------------------------------------------------------------
// X: the particle family (storage type, arithmetic of the move and the gather, the push of one particle
// by itself). FIX: the stage has the pitches of the default segments (the stencils' offsets are then constants).
// PACKED: the segments follow each other without padding, and linear slots behind them. DEP: how
// a row's particles deposit (cellDeposit)
template<class X, int D, int O, bool RN, bool FIX, bool PACKED, int DEP>
__global__ __launch_bounds__((pc::CellCfg<X, D, O>::BLOCK)) __attribute__((amdgpu_waves_per_eu(pc::CellCfg<X, D, O>::WAVES)))
void k_push_cell(pc::CellArgs<X> K)
{
    using namespace pc;
    using R                     = typename X::Real;
    using C                     = pc::CellWin<D, O, RN>;
    constexpr int CB            = CellCfg<X, D, O>::BLOCK;
    constexpr bool NEXT         = CellCfg<X, D, O>::PREFETCH;
    constexpr unsigned int LIST = CellCfg<X, D, O>::LIST;
    // 16-byte aligned: the hand-over buffers are read as pairs of words (a pair read 8 bytes off
    // took 8 times as long)
    extern __shared__ __align__(16) double cellLds[];
    double* const lds = cellLds;
    __shared__ unsigned int list[LIST];
    __shared__ unsigned int listed;
    // 3D and packed storage: split workgroups per segment; 2D: the work items of the sort (captured
    // steps keep their grid while the sorts change the items). slots: the segment's, whole rows but in
    // packed storage, whose segments follow each other without padding (the overflow segment takes what
    // was appended since)
    unsigned int seg, rA, rB, slots, nItems = 0;
    unsigned long long off;
    if (D == 3 || PACKED)
    {
        nItems                  = gridDim.x;
        if constexpr (D == 2)
            ktBegin(K.A.kt);
        unsigned int const nsegs = static_cast<unsigned int>(K.A.sg.nsegs);
        unsigned int const base  = nsegs * K.A.split; // workgroups before the overflow segment's
        unsigned int part = blockIdx.x - base, parts = gridDim.x - base;
        seg = nsegs;
        if (blockIdx.x < base)
        {
            unsigned int const item = xcdItem(blockIdx.x, base);
            seg                     = item / K.A.split;
            part                    = item - seg * K.A.split;
            parts                   = K.A.split;
        }
        off = K.A.st.off[seg];
        if (PACKED)
        {
            unsigned long long const end = seg < nsegs ? K.A.st.off[seg + 1] : K.A.n;
            off   = min(off, K.A.n);
            slots = static_cast<unsigned int>(max(min(end, K.A.n), off) - off);
        }
        else
            slots = K.A.st.rows[seg] * LANES;
        unsigned long long const rows = (static_cast<unsigned long long>(slots) + LANES - 1) / LANES;
        rA = static_cast<unsigned int>(rows * part / parts);
        rB = static_cast<unsigned int>(rows * (part + 1) / parts);
    }
    else
    {
        nItems = *K.A.st.nItems;
        if (blockIdx.x >= nItems)
            return;
        pc::ktBegin(K.A.kt);
        seg = K.A.st.items[2 * blockIdx.x];
        pc::itemRows(K.A.st.items[2 * blockIdx.x + 1], K.A.st.rows[seg],
                     K.A.st.rowsPerItem, rA, rB);
        off   = K.A.st.off[seg];
        slots = rB * LANES;
    }
    // the same in every lane: scalar from here on
    rA    = __builtin_amdgcn_readfirstlane(rA);
    rB    = __builtin_amdgcn_readfirstlane(rB);
    slots = __builtin_amdgcn_readfirstlane(slots);
    off   = static_cast<unsigned int>(__builtin_amdgcn_readfirstlane(static_cast<unsigned int>(off)))
          | static_cast<unsigned long long>(static_cast<unsigned int>(
                __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(off >> 32))))
                << 32;
    if (rB > rA && !K.A.G.stopped())
    {
        unsigned int const rows = rB - rA;
        unsigned int const lane = threadIdx.x & 63u;
        unsigned int const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        constexpr int EX  = cellExt(D, O) | 1;
        int const e1      = D == 2 ? (FIX ? EX : K.A.tile.emExt[1] | 1) : (FIX ? cellExt(3, O) : K.A.tile.emExt[1]);
        int const e2      = D == 2 ? 1 : (FIX ? EX : K.A.tile.emExt[2] | 1);
        int const emNodes = K.A.tile.emExt[0] * e1 * e2;
        R* const em       = reinterpret_cast<R*>(lds + (RN ? 4 : 5) * K.A.tile.stride);
        R* const buf      = reinterpret_cast<R*>(lds + (RN ? 4 : 5) * K.A.tile.stride + K.A.tile.emStride) + wave * C::BUF;
        zeroTile<RN, CB>(lds, K.A.tile);
        if (threadIdx.x == 0)
            listed = 0u;
        TileView T;
        tileView(T, lds, K.A.tile);
        pc::segTileOrigin<D>(K.A.G, K.A.sg, K.A.tile, seg, T.org);
#pragma unroll
        for (int d = 0; d < D; ++d)
            T.org[d] = __builtin_amdgcn_readfirstlane(T.org[d]); // the same in every lane: scalar from here on
        int const p2 = T.pitch[2], p12 = T.pitch[1] * T.pitch[2];
        bool const push   = K.A.pushOn;
        // read at run time where the groups' code is kept beside (orders 2 and 3): without it the constants of
        // the one-by-one push move out of the loop over the rows and spill (190x150 cells, order 2, one particle per
        // cell: 92 us per PPC step, 82 with it; order 1: 88 and 87)
        bool const lanes  = DEP == DEP_LANES && (O == 1 || K.A.deposit);
        bool const writes = push && K.A.mode == MODE_ALL;
        // per direction: AMR cell of the deposit tile's and of the stage's first cell, and the number
        // of cells whose windows (stencils) they hold; the stage's cells are clipped to those whose
        // stencils lie in the arrays
        int tileCell[D], tileCells[D], emCell[D], emLow[D], emCells[D], emOrg[D], dom[D], domCells[D];
        R h[D];
#pragma unroll
        for (int d = 0; d < D; ++d)
        {
            int const shift = K.A.G.lower[d] - K.A.G.g; // AMR cell of local cell 0
            tileCell[d]     = T.org[d] + C::WB + shift;
            tileCells[d]    = max(T.ext[d] - C::W + 1, 0);
            emOrg[d]        = T.org[d] + K.A.tile.emLo[d];
            emCell[d]       = emOrg[d] + shift;
            int const lo    = max(emOrg[d] - cellGatherLo(O), K.A.G.safeLo[d]);
            int const hi    = min(emOrg[d] - cellGatherLo(O) + K.A.tile.emExt[d] - cellGatherNodes(O), K.A.G.safeHi[d]);
            emLow[d]        = lo + shift;
            emCells[d]      = max(hi - lo + 1, 0);
            dom[d]          = K.A.box.dom_lo[d];
            domCells[d]     = K.A.box.dom_hi[d] - dom[d] + 1;
            h[d]            = static_cast<R>(K.A.hdtdx[d]);
        }
        double const dto2m = K.A.dto2m, coef = K.A.coef, charge = K.A.charge;
        if (push)
            stageFields<X, D, CB>(K.A, em, emOrg, e1, e2, emNodes);
        __syncthreads();

        unsigned int r          = rA + rows * wave / CellCfg<X, D, O>::NW;
        unsigned int const rEnd = rA + rows * (wave + 1) / CellCfg<X, D, O>::NW;
        do
        {
            C acc;
            acc.zero();
            int cur = -1; // tile node of the accumulated window's origin
            Part<D, R> next;
            if (NEXT && r < rEnd)
                loadRow<D, RN>(K.v, off + static_cast<unsigned long long>(r) * LANES, PACKED ? min(lane, slots - 1 - r * LANES) : lane, next);
            for (; r < rEnd; ++r)
            {
                // until the list might overflow (each wavefront that still finds room may add 64)
                if (__builtin_amdgcn_readfirstlane(*static_cast<unsigned int volatile*>(&listed)) > LIST - CB)
                    break;
                unsigned long long const row = off + static_cast<unsigned long long>(r) * LANES;
                Part<D, R> P;
                if constexpr (NEXT)
                {
                    P = next;
                    if (r + 1 < rEnd)
                        loadRow<D, RN>(K.v, row + LANES, PACKED ? min(lane, slots - 1 - (r + 1) * LANES) : lane, next); // in flight over this row's work
                }
                else
                    loadRow<D, RN>(K.v, row, PACKED ? min(lane, slots - 1 - r * LANES) : lane, P);
                double const q  = RN ? charge : static_cast<double>(P.q);
                bool const mine = !PACKED || lane < slots - r * LANES;
                bool const live = mine & (P.cell[0] != DEAD_CELL);
                bool ok         = live;
                if (push)
                {
                    ok = X::template halfStep<D>(P.cell, P.delta, P.v, h) & ok;
                    int rel[D];
#pragma unroll
                    for (int d = 0; d < D; ++d)
                    {
                        ok     = ok & (static_cast<unsigned int>(P.cell[d] - emLow[d]) < static_cast<unsigned int>(emCells[d]));
                        rel[d] = P.cell[d] - emCell[d];
                    }
                    R E[3] = {0, 0, 0}, B[3] = {0, 0, 0};
                    if (ok)
                        gatherStaged<X, D, O>(em, e1, e2, emNodes, rel, P.delta, E, B);
                    X::accelerate(P.v, E, B, q, dto2m);
                    ok = X::template halfStep<D>(P.cell, P.delta, P.v, h) & ok;
#pragma unroll
                    for (int d = 0; d < D; ++d)
                        ok = ok & (static_cast<unsigned int>(P.cell[d] - dom[d]) < static_cast<unsigned int>(domCells[d]));
                }
                // the tile node of the window's origin; a value that is not finite (it would reach the
                // whole window) deposits by itself
                ok = ok & __builtin_isfinite(P.w * static_cast<R>(coef)) & (RN || __builtin_isfinite(q * P.w * coef));
                int key = 0;
#pragma unroll
                for (int d = 0; d < D; ++d)
                {
                    int const rel = P.cell[d] - tileCell[d];
                    key += rel * (d == 0 ? p12 : (d == 1 ? p2 : 1));
                    ok = ok & (static_cast<unsigned int>(rel) < static_cast<unsigned int>(tileCells[d]))
                         & (P.delta[d] == P.delta[d]);
                }
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    ok = ok & __builtin_isfinite(P.v[d] * P.w * static_cast<R>(coef));
                key = ok ? key : -1;
                unsigned long long strays = 0; // DEP_FEW: the particles of groups below CELL_MOVE
                // the half rows in turn: first the accumulated window's cell, then every other cell
#pragma unroll
                for (int half = 0; half < 2; ++half)
                {
                    unsigned int rest = lanes ? 0u : static_cast<unsigned int>(__ballot(ok) >> (32 * half));
                    if (rest == 0u)
                        continue;
                    pc::cellStage<D, O, RN>(buf, half, ok, P.delta, P.w, q, P.v, coef);
                    unsigned int m = cur < 0 ? 0u : static_cast<unsigned int>(__ballot(key == cur) >> (32 * half));
                    if (m)
                        pc::cellAdd<D, O, RN>(buf, m, acc);
                    rest &= ~m;
                    unsigned int few = 0, fews = 0; // their lanes in this half, and the groups
                    while (rest)
                    {
                        int const p = __builtin_ctz(rest);
                        int const c = __builtin_amdgcn_readlane(key, p + 32 * half);
                        m           = static_cast<unsigned int>(__ballot(key == c) >> (32 * half)) & rest;
                        rest &= ~m;
                        int const n = __popc(m);
                        if (n >= CELL_MOVE || cur < 0)
                        {
                            if (cur >= 0)
                                pc::cellFlush<D, O, RN>(acc, lds, T.stride, cur, p12, p2);
                            acc.zero();
                            cur = c;
                            pc::cellAdd<D, O, RN>(buf, m, acc);
                        }
                        else if (DEP == DEP_FEW)
                        {
                            few |= m;
                            ++fews;
                        }
                        else if (n >= CELL_GROUP)
                        {
                            C one;
                            one.zero();
                            pc::cellAdd<D, O, RN>(buf, m, one);
                            pc::cellFlush<D, O, RN>(one, lds, T.stride, c, p12, p2);
                        }
                        else
                            pc::cellAddOne<D, O, RN>(buf, p, lds, T.stride, c, p12, p2);
                    }
                    // one such group deposits on the matrix cores, more lane by lane after the halves
                    if (DEP == DEP_FEW && fews > 1)
                        strays |= static_cast<unsigned long long>(few) << (32 * half);
                    else if (DEP == DEP_FEW && few)
                    {
                        C one;
                        one.zero();
                        pc::cellAdd<D, O, RN>(buf, few, one);
                        pc::cellFlush<D, O, RN>(one, lds, T.stride, __builtin_amdgcn_readlane(key, __builtin_ctz(few) + 32 * half), p12, p2);
                    }
                }
                if constexpr (DEP == DEP_LANES)
                    pc::cellAddLanes<O, RN, true>(ok, P.delta, P.w, q, P.v, coef, lds, T.stride, key, p12, p2);
                else if constexpr (DEP == DEP_FEW)
                    if (strays)
                        pc::cellAddLanes<O, RN, false>((strays >> lane) & 1ull, P.delta, P.w, q, P.v, coef, lds, T.stride, key, p12, p2);
                unsigned long long const left = __ballot(live && !ok);
                if (left)
                {
                    unsigned int base = 0;
                    if (lane == 0)
                        base = atomicAdd(&listed, static_cast<unsigned int>(__popcll(left)));
                    base = __builtin_amdgcn_readfirstlane(base);
                    if ((left >> lane) & 1ull)
                        list[base + __popcll(left & ((1ull << lane) - 1ull))] = r * LANES + lane;
                }
                if (writes)
                {
                    if (ok)
                    {
#pragma unroll
                        for (int d = 0; d < D; ++d)
                        {
                            rowOf(K.v.ic[d], row)[lane] = P.cell[d];
                            rowOf(K.v.de[d], row)[lane] = P.delta[d];
                        }
#pragma unroll
                        for (int d = 0; d < 3; ++d)
                            rowOf(K.v.v[d], row)[lane] = P.v[d];
                    }
                    uint8_t* const status = K.A.status;
                    if (status && mine && (ok || !live))
                        rowOf(status, row)[lane] = live ? ST_KEEP : ST_DROP;
                }
            }
            if (cur >= 0)
                pc::cellFlush<D, O, RN>(acc, lds, T.stride, cur, p12, p2);
            __syncthreads();
            unsigned int const n = listed;
            CellArgs<X> const& L = cellArgs<X>();
            for (unsigned int x = threadIdx.x; x < n; x += CB)
                X::template pushOne<D, O, RN>(L.A, L.v, off + list[x], T);
            __syncthreads();
            if (threadIdx.x == 0)
            {
                if (n && cellArgs<X>().A.lone)
                    atomicAdd(cellArgs<X>().A.lone, static_cast<unsigned long long>(n));
                listed = 0u;
            }
        } while (__syncthreads_or(r < rEnd));
        PushArgs const& A = cellArgs<X>().A;
        flushTile<D, RN, CB>(A.G, T, A.tile.nodes, A.mom, A.charge);
    }
    if (D == 2 && K.A.kt)
    {
        __syncthreads();
        pc::ktEnd(K.A.kt, nItems);
    }
}

template<class X, int D, int O, bool RN, bool FIX, bool PACKED = false, int DEP = DEP_GROUPS>
static void launchPushCellT(PushArgs const& A, PViewT<typename X::Real> const& in, hipStream_t s)
{
    if constexpr (D == 2 && DEP == DEP_GROUPS)
        if (A.deposit == DEP_LANES)
        {
            launchPushCellT<X, D, O, RN, FIX, PACKED, DEP_LANES>(A, in, s);
            return;
        }
    if constexpr (D == 2 && O == 1 && DEP == DEP_GROUPS)
        if (A.deposit == DEP_FEW)
        {
            launchPushCellT<X, D, O, RN, FIX, PACKED, DEP_FEW>(A, in, s);
            return;
        }
    // more than 64 KB of dynamic LDS has to be allowed for the kernel (once per device)
    static std::mutex mtx;
    static bool allowed[64] = {};
    int dev                 = 0;
    if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64)
    {
        std::lock_guard<std::mutex> lock(mtx);
        if (!allowed[dev])
            allowed[dev] = hipFuncSetAttribute(reinterpret_cast<void const*>(&k_push_cell<X, D, O, RN, FIX, PACKED, DEP>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, pc::CELL_LDS_MAX)
                           == hipSuccess;
    }
    // packed storage: what was appended behind the segments is spread over the GPU (in the workgroups of
    // one segment, 1.9 million particles in 3D took 1.1 ms per pair of pushes after ten steps, 7.6 after
    // eighty, of appended leavers)
    unsigned int const overflow = PACKED ? static_cast<unsigned int>(pc::CUS) : A.split;
    unsigned int const grid = D == 3 || PACKED ? static_cast<unsigned int>(A.sg.nsegs) * A.split + overflow : A.st.itemsCap;
    k_push_cell<X, D, O, RN, FIX, PACKED, DEP><<<grid, pc::CellCfg<X, D, O>::BLOCK, A.tile.bytes, s>>>(pc::CellArgs<X>{A, in});
}
} // namespace phx
