// phx_cell_deposit.hpp -- moment deposit of particles grouped by cell on the FP64 matrix cores.
//
// The particles of one cell deposit into one window of W nodes per direction (W = 2 at order 1:
// nodes cell, cell + 1; W = 4 at orders 2 and 3: nodes cell - 1 .. cell + 2, a particle's weight
// being zero on the node its order-2 stencil leaves out). Over the particles p of the cell the
// window is the contraction
//     window[(a, b), (c, m)] = sum_p (wx_p[a] wy_p[b]) (wz_p[c] value_p[m])
// with m the moments n, Fx, Fy, Fz (in 2D without c): in 3D at W = 4 one 16x16x4 FP64 MFMA per four
// particles, at W = 2 one 4x4x4 (four-block) MFMA per eight; in 2D one 4x4x4 MFMA per four (W = 4) or
// sixteen (W = 2). The window stays in a wavefront's registers while its
// particles stay in the cell and is then added to the workgroup's LDS tile, 4 (3D, W = 4) or 1
// LDS atomics per wavefront and cell instead of one per particle, node and moment: in 3D a particle cost
// 108 (order 2) or 256 (order 3) lanes of ds_add_f64, about 30 cycles of the CU's LDS per
// wavefront instruction, and costs about a quarter (W = 4) or a sixteenth (W = 2) of an MFMA here.
//
// An instruction takes 64 cycles of its SIMD (16x16x4) or 16 (4x4x4), the same rate, at which independent
// chains reach 75 TFLOP/s: in the 3D push at order 2 the matrix cores are 13 % busy.
//
// The lanes of a wavefront hand their weights over through a small LDS buffer of the wavefront, 32
// particles at a time: array j (the weights along x, y, z, then the values) of particle p at
// j * WSTR + p. WSTR is 36 words: the four arrays and four particle pairs that one read touches lie in
// distinct banks in the FP32 buffer, and in the FP64 one pairs 2 and 3 of an array share the banks of
// pairs 0 and 1 of the next (conflicts of the whole push: 15 % of its LDS cycles at order 2 in 3D).
#pragma once

#include "phx_push_common.hpp"

namespace phx
{
namespace pc
{
typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int WHALF = 32; // particles handed over at a time
constexpr int WSTR  = 36; // words between two arrays of the buffer (even: pairs are read as 16 bytes)

// order of the wavefront's own LDS writes before its later reads of other lanes' words
__device__ __forceinline__ void waveLds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// window of a cell. RN: the charge density is derived from n and has no column
template<int D, int O, bool RN>
struct CellWin
{
    static constexpr int W    = O == 1 ? 2 : 4;
    static constexpr int WB   = O == 1 ? 0 : 1; // window base = local cell - WB
    static constexpr int NVAL = RN ? 4 : 5;
    static constexpr int ARR  = D * W + NVAL;
    static constexpr int BUF  = ARR * WSTR; // words of LDS per wavefront
    static constexpr int NACC = D == 3 && W == 4 ? 4 : 1;

    double a[NACC];            // n, Fx, Fy, Fz columns
    double rho[RN ? 1 : NACC]; // the charge density's column

    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int r = 0; r < NACC; ++r)
            a[r] = 0.;
        if constexpr (!RN)
#pragma unroll
            for (int r = 0; r < NACC; ++r)
                rho[r] = 0.;
    }
};

// B-spline weights (interpolator.hpp:54-125) from the offset of the particle in its cell alone: u is
// the particle's position less the stencil's first node, of the size of the stencil, where the
// absolute position would cost its last digits; w[0 .. O]
template<int O>
__device__ __forceinline__ void splineWeights(double u, double* w)
{
    if constexpr (O == 1)
    {
        w[0] = 1. - u;
        w[1] = u;
    }
    else if constexpr (O == 2)
    {
        double const d = u - 1.;
        double const lo = 0.5 - d, hi = 0.5 + d;
        w[0] = 0.5 * lo * lo;
        w[1] = __builtin_fma(-d, d, 0.75);
        w[2] = 0.5 * hi * hi;
    }
    else
    {
        // u = 1 + t, t in [0, 1): cubic B-spline at t + 1, t, 1 - t, 2 - t
        double const t = u - 1., s = 1. - t;
        double const t2 = t * t, s2 = s * s;
        w[0] = s2 * s * (1. / 6.);
        w[1] = __builtin_fma(t2, __builtin_fma(0.5, t, -1.), 2. / 3.);
        w[2] = __builtin_fma(s2, __builtin_fma(0.5, s, -1.), 2. / 3.);
        w[3] = t2 * t * (1. / 6.);
    }
}

// stencil of one direction: shift of its first node from the particle's cell (interpolator.hpp:
// 519-549) and weights, centering c
template<int O>
__device__ __forceinline__ int splineStencil(int c, double delta, double* w)
{
    int const sh   = startShift<O>(c, delta);
    double const u = delta + (c == CD ? static_cast<double>(sh) - 0.5 : static_cast<double>(sh));
    splineWeights<O>(u, w);
    return sh;
}

// B-spline weights at u = np - start (u in [0, O+1)); the products of interpolator.hpp:54-125
// written in u: order 2 uses 1 - u for (start + 1 - np), order 3 uses -u for (start - np)
template<int O>
__device__ __forceinline__ void bspline32(float u, float* w)
{
    if constexpr (O == 1)
    {
        w[1] = u;
        w[0] = 1.f - u;
    }
    else if constexpr (O == 2)
    {
        float const d  = 1.f - u;
        float const c1 = .5f + d;
        float const c3 = .5f - d;
        w[0]           = .5f * c1 * c1;
        w[1]           = .75f - d * d;
        w[2]           = .5f * c3 * c3;
    }
    else
    {
        float const index = -u;
        float const c1    = 1.f + .5f * index;
        float const c2    = index + 1.f;
        float const c3    = index + 2.f;
        float const c4    = 1.f - .5f * (index + 3.f);
        float const c2s   = c2 * c2;
        float const c3s   = c3 * c3;
        w[0]              = (4.f / 3.f) * c1 * c1 * c1;
        w[1]              = (2.f / 3.f) - c2s - .5f * c2s * c2;
        w[2]              = (2.f / 3.f) - c3s + .5f * c3s * c3;
        w[3]              = (4.f / 3.f) * c4 * c4 * c4;
    }
}

template<int O>
__device__ __forceinline__ int splineStencil(int c, float delta, float* w)
{
    int const sh = startShift<O>(c, static_cast<double>(delta));
    float u      = static_cast<float>(sh) + delta;
    if (c == CD)
        u -= .5f;
    bspline32<O>(u, w);
    return sh;
}

// the primal weights of one direction on the cell's window (zero on the node an order-2 stencil
// leaves out)
template<int O, class R>
__device__ __forceinline__ void windowWeights(R delta, R* out)
{
    if constexpr (O == 2)
    {
        R w[3];
        bool const low = splineStencil<2>(CP, delta, w) == 1;
        out[0]         = low ? w[0] : R(0);
        out[1]         = low ? w[1] : w[0];
        out[2]         = low ? w[2] : w[1];
        out[3]         = low ? R(0) : w[2];
    }
    else
        splineStencil<O>(CP, delta, out);
}

// two neighbouring words of the buffer
__device__ __forceinline__ double2 pairAt(double const* p) { return *reinterpret_cast<double2 const*>(p); }
__device__ __forceinline__ double2 pairAt(float const* p)
{
    float2 const f = *reinterpret_cast<float2 const*>(p);
    return double2{static_cast<double>(f.x), static_cast<double>(f.y)};
}

// the 32 particles of lanes [32 half, 32 half + 32) into the wavefront's buffer: the window weights
// of delta along each direction, then the values n, Fx, Fy, Fz (and rho); lanes without `ok` hand over finite
// weights and zero values
template<int D, int O, bool RN, class R>
__device__ __forceinline__ void cellStage(R* buf, int half, bool ok, R const* delta, R weight, double q,
                                          R const* v, double coef)
{
    using C        = CellWin<D, O, RN>;
    int const lane = static_cast<int>(threadIdx.x & 63u);
    waveLds(); // the reads of the half before are done
    if ((lane >> 5) == half)
    {
        R* const b = buf + (lane & (WHALF - 1));
#pragma unroll
        for (int d = 0; d < D; ++d)
        {
            R ww[C::W];
            windowWeights<O>(ok ? delta[d] : R(0), ww);
#pragma unroll
            for (int a = 0; a < C::W; ++a)
                b[(d * C::W + a) * WSTR] = ww[a];
        }
        // the reference's products: 1. * w * coef, v * w * coef, q * w * coef
        b[D * C::W * WSTR] = ok ? weight * static_cast<R>(coef) : R(0);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            b[(D * C::W + 1 + d) * WSTR] = ok ? v[d] * weight * static_cast<R>(coef) : R(0);
        if constexpr (!RN)
            b[(D * C::W + 4) * WSTR] = ok ? q * weight * coef : 0.;
    }
    waveLds();
}

// the staged particles whose bit of `mask` is set (all of one cell) added to the window. ALL: every
// instruction of the half row is issued, without a branch between them (many particles set)
template<int D, int O, bool RN, bool ALL, class R>
__device__ __forceinline__ void cellAddT(R const* buf, unsigned int mask, CellWin<D, O, RN>& acc)
{
    using C        = CellWin<D, O, RN>;
    int const lane = static_cast<int>(threadIdx.x & 63u);
    int const i    = lane & 15;
    int const k    = lane >> 4;
    if constexpr (D == 2)
    {
        // W = 4: block m, rows a, columns b; four particles per instruction, lane group k taking a
        // pair of particles for two instructions. W = 2: block of particles, rows (a, b), columns m;
        // sixteen particles per instruction
        constexpr bool W4 = C::W == 4;
        constexpr int PP  = W4 ? 8 : 32; // particles of two instructions
        int const l4 = lane & 3, blk = (lane >> 2) & 3;
        int const o  = W4 ? 2 * k : 8 * k + 2 * blk;
        R const* const px = buf + (W4 ? l4 : l4 >> 1) * WSTR + o;
        R const* const py = buf + (C::W + (W4 ? l4 : l4 & 1)) * WSTR + o;
        R const* const pv = buf + (2 * C::W + (W4 ? blk : l4)) * WSTR + o;
        R const* const pr = buf + (2 * C::W + 4) * WSTR + o;
        unsigned int const mk  = mask >> o;
#pragma unroll
        for (int t = 0; t < WHALF / PP; ++t)
        {
            if (!ALL && W4 && ((mask >> (8 * t)) & 0xffu) == 0u)
                continue;
            double2 const x = pairAt(px + PP * t);
            double2 const y = pairAt(py + PP * t);
            double2 const v = pairAt(pv + PP * t);
            double const v0 = (mk >> (PP * t % 32)) & 1u ? v.x : 0.;
            double const v1 = (mk >> (PP * t % 32)) & 2u ? v.y : 0.;
            if constexpr (W4)
            {
                acc.a[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x.x * v0, y.x, acc.a[0], 0, 0, 0);
                acc.a[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x.y * v1, y.y, acc.a[0], 0, 0, 0);
            }
            else
            {
                acc.a[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x.x * y.x, v0, acc.a[0], 0, 0, 0);
                acc.a[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x.y * y.y, v1, acc.a[0], 0, 0, 0);
            }
            if constexpr (!RN)
            {
                double2 const q = pairAt(pr + PP * t);
                bool const on   = W4 ? blk == 0 : l4 == 0;
                double const q0 = on && ((mk >> (PP * t % 32)) & 1u) ? q.x : 0.;
                double const q1 = on && ((mk >> (PP * t % 32)) & 2u) ? q.y : 0.;
                if constexpr (W4)
                {
                    acc.rho[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x.x * q0, y.x, acc.rho[0], 0, 0, 0);
                    acc.rho[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x.y * q1, y.y, acc.rho[0], 0, 0, 0);
                }
                else
                {
                    acc.rho[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x.x * y.x, q0, acc.rho[0], 0, 0, 0);
                    acc.rho[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(x.y * y.y, q1, acc.rho[0], 0, 0, 0);
                }
            }
        }
    }
    else if constexpr (C::W == 4)
    {
        // rows (a, b) = (i / 4, i % 4) of A, columns (c, m) = (i / 4, i % 4) of B; four particles
        // per instruction, lane group k taking a pair of particles for two instructions
        R const* const px = buf + (i >> 2) * WSTR + 2 * k;
        R const* const py = buf + (4 + (i & 3)) * WSTR + 2 * k;
        R const* const pz = buf + (8 + (i >> 2)) * WSTR + 2 * k;
        R const* const pv = buf + (12 + (i & 3)) * WSTR + 2 * k;
        R const* const pr = buf + 16 * WSTR + 2 * k;
        unsigned int const mk  = mask >> (2 * k);
        d4 c  = {acc.a[0], acc.a[1], acc.a[2], acc.a[3]};
        d4 cr = {0., 0., 0., 0.};
        if constexpr (!RN)
            cr = d4{acc.rho[0], acc.rho[1], acc.rho[2], acc.rho[3]};
#pragma unroll
        for (int t = 0; t < WHALF / 8; ++t)
        {
            if (!ALL && ((mask >> (8 * t)) & 0xffu) == 0u)
                continue;
            double2 const x = pairAt(px + 8 * t);
            double2 const y = pairAt(py + 8 * t);
            double2 const z = pairAt(pz + 8 * t);
            double2 const v = pairAt(pv + 8 * t);
            double const a0 = x.x * y.x, a1 = x.y * y.y;
            double const z0 = (mk >> (8 * t)) & 1u ? z.x : 0.;
            double const z1 = (mk >> (8 * t)) & 2u ? z.y : 0.;
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, z0 * v.x, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, z1 * v.y, c, 0, 0, 0);
            if constexpr (!RN)
            {
                double2 const q = pairAt(pr + 8 * t);
                bool const on   = (i & 3) == 0;
                cr = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, on ? z0 * q.x : 0., cr, 0, 0, 0);
                cr = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, on ? z1 * q.y : 0., cr, 0, 0, 0);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            acc.a[r] = c[r];
            if constexpr (!RN)
                acc.rho[r] = cr[r];
        }
    }
    else
    {
        // block beta = (c, s): node c along z and half s of the particles; rows (a, b) = bits of
        // lane % 4, columns m; eight particles per instruction
        int const s = (lane >> 3) & 1, c = (lane >> 2) & 1;
        int const o = 4 * k + 2 * s;
        R const* const px = buf + ((lane >> 1) & 1) * WSTR + o;
        R const* const py = buf + (2 + (lane & 1)) * WSTR + o;
        R const* const pz = buf + (4 + c) * WSTR + o;
        R const* const pv = buf + (6 + (lane & 3)) * WSTR + o;
        R const* const pr = buf + 10 * WSTR + o;
        unsigned int const mk  = mask >> o;
#pragma unroll
        for (int t = 0; t < WHALF / 16; ++t)
        {
            if (!ALL && ((mask >> (16 * t)) & 0xffffu) == 0u)
                continue;
            double2 const x = pairAt(px + 16 * t);
            double2 const y = pairAt(py + 16 * t);
            double2 const z = pairAt(pz + 16 * t);
            double2 const v = pairAt(pv + 16 * t);
            double const a0 = x.x * y.x, a1 = x.y * y.y;
            double const z0 = (mk >> (16 * t)) & 1u ? z.x : 0.;
            double const z1 = (mk >> (16 * t)) & 2u ? z.y : 0.;
            acc.a[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, z0 * v.x, acc.a[0], 0, 0, 0);
            acc.a[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, z1 * v.y, acc.a[0], 0, 0, 0);
            if constexpr (!RN)
            {
                double2 const q = pairAt(pr + 16 * t);
                bool const on   = (lane & 3) == 0;
                acc.rho[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, on ? z0 * q.x : 0., acc.rho[0], 0, 0, 0);
                acc.rho[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, on ? z1 * q.y : 0., acc.rho[0], 0, 0, 0);
            }
        }
    }
}

template<int D, int O, bool RN, class R>
__device__ __forceinline__ void cellAdd(R const* buf, unsigned int mask, CellWin<D, O, RN>& acc)
{
    if (__popc(mask) >= WHALF / 2)
        cellAddT<D, O, RN, true>(buf, mask, acc);
    else
        cellAddT<D, O, RN, false>(buf, mask, acc);
}

// one staged particle (p, in no larger group) added to the LDS tile by itself
template<int D, int O, bool RN, class R>
__device__ __forceinline__ void cellAddOne(R const* buf, int p, double* tile, int stride, int node0,
                                           int p12, int p2)
{
    using C        = CellWin<D, O, RN>;
    int const lane = static_cast<int>(threadIdx.x & 63u);
    int const m    = lane & 3;
    int const slab = RN || m == 0 ? m : m + 1;
    auto const at  = [&](int x) { return static_cast<double>(buf[x]); };
    if constexpr (D == 2)
    {
        int const a = lane / (4 * C::W), b = lane / 4 % C::W;
        if (a < C::W)
        {
            double const xy = at(a * WSTR + p) * at((C::W + b) * WSTR + p);
            int const n     = node0 + a * p12 + b * p2;
            atomicAdd(tile + slab * stride + n, xy * at((2 * C::W + m) * WSTR + p));
            if constexpr (!RN)
                if (m == 0)
                    atomicAdd(tile + stride + n, xy * at((2 * C::W + 4) * WSTR + p));
        }
    }
    else if constexpr (C::W == 4)
    {
        int const b = lane >> 4, c = (lane & 15) >> 2;
        double const yz = at((4 + b) * WSTR + p) * at((8 + c) * WSTR + p);
        double const t  = yz * at((12 + m) * WSTR + p);
        int const n     = node0 + b * p2 + c;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            double const x = at(r * WSTR + p);
            atomicAdd(tile + slab * stride + n + r * p12, x * t);
            if constexpr (!RN)
                if (m == 0)
                    atomicAdd(tile + stride + n + r * p12, x * (yz * at(16 * WSTR + p)));
        }
    }
    else if (lane < 32)
    {
        int const a = lane >> 4, b = (lane >> 3) & 1, c = (lane >> 2) & 1;
        double const xyz = at(a * WSTR + p) * at((2 + b) * WSTR + p) * at((4 + c) * WSTR + p);
        int const n      = node0 + a * p12 + b * p2 + c;
        atomicAdd(tile + slab * stride + n, xyz * at((6 + m) * WSTR + p));
        if constexpr (!RN)
            if (m == 0)
                atomicAdd(tile + stride + n, xyz * at(10 * WSTR + p));
    }
}

// a and b turned left by `by` places (N = 2 or 4)
template<int N, class A>
__device__ __forceinline__ void turn(A* a, int* b, int by)
{
#pragma unroll
    for (int s = 1; s < N; s *= 2)
    {
        bool const on = (by & s) != 0;
        A x[N];
        int y[N];
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
            x[i] = on ? a[(i + s) % N] : a[i];
            y[i] = on ? b[(i + s) % N] : b[i];
        }
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
            a[i] = x[i];
            b[i] = y[i];
        }
    }
}

// the particles with `ok` added to the LDS tile, each by its own lane; node0: the tile node of the
// origin of its cell's window (2D). Neighbouring lanes, which hold particles of one cell, start at
// different moments and nodes of the stencil
template<int O, bool RN, bool TURN, class R>
__device__ __forceinline__ void cellAddLanes(bool ok, R const* delta, R weight, double q, R const* v, double coef,
                                             double* tile, int stride, int node0, int p12, int p2)
{
    if (!ok)
        return;
    int const lane = static_cast<int>(threadIdx.x & 63u);
    R w[2][O + 1];
    double val[4];
    int low[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) // order 2: the stencil leaves the window's first or last node out
        low[d] = splineStencil<O>(CP, delta[d], w[d]) == 0 && O == 2 ? 1 : 0;
    val[0] = weight * static_cast<R>(coef);
#pragma unroll
    for (int m = 0; m < 3; ++m)
        val[1 + m] = v[m] * weight * static_cast<R>(coef);
    double const rho = q * weight * coef;
    node0 += (low[0] ? p12 : 0) + (low[1] ? p2 : 0);
    if constexpr (TURN && O == 1)
    {
        int x[2] = {0, p12}, y[2] = {0, p2}, slab[4] = {0, stride, 2 * stride, 3 * stride};
        if constexpr (!RN)
            for (int m = 1; m < 4; ++m)
                slab[m] += stride;
        turn<4>(val, slab, lane & 3);
        turn<2>(w[0], x, (lane >> 2) & 1);
        turn<2>(w[1], y, (lane >> 3) & 1);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
            {
                double const xy = static_cast<double>(w[0][a]) * static_cast<double>(w[1][b]);
                double* const n = tile + node0 + x[a] + y[b];
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    atomicAdd(n + slab[m], xy * val[m]);
                if constexpr (!RN)
                    atomicAdd(n + stride, xy * rho);
            }
    }
    else
    {
        // the nodes' distances anew for every row: kept over the rows they took the push's registers
        asm volatile("" : "+s"(stride), "+s"(p12), "+s"(p2));
#pragma unroll
        for (int a = 0; a <= O; ++a)
#pragma unroll
            for (int b = 0; b <= O; ++b)
            {
                double const xy = static_cast<double>(w[0][a]) * static_cast<double>(w[1][b]);
                double* const n = tile + node0 + a * p12 + b * p2;
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    atomicAdd(n + (RN || m == 0 ? m : m + 1) * stride, xy * val[m]);
                if constexpr (!RN)
                    atomicAdd(n + stride, xy * rho);
            }
    }
}

// add the window to the LDS tile: node0 is the tile node of the window's origin, p12 and p2 the
// node distances along the first two directions, slab m of the tile the moments in the order n, (rho,) Fx, Fy, Fz
template<int D, int O, bool RN>
__device__ __forceinline__ void cellFlush(CellWin<D, O, RN> const& acc, double* tile, int stride, int node0,
                                          int p12, int p2)
{
    using C        = CellWin<D, O, RN>;
    int const lane = static_cast<int>(threadIdx.x & 63u);
    int const m    = lane & 3;
    int const slab = RN || m == 0 ? m : m + 1;
    if constexpr (D == 2)
    {
        // W = 4: lane (a, m, b) = (lane / 16, lane / 4 % 4, lane % 4); W = 2: rows (a, b) = lane / 16,
        // column lane % 4, the four blocks of particles adding to the same node
        constexpr bool W4 = C::W == 4;
        int const mm = W4 ? (lane >> 2) & 3 : m, sl = RN || mm == 0 ? mm : mm + 1;
        int const n  = W4 ? node0 + (lane >> 4) * p12 + (lane & 3) * p2
                          : node0 + (lane >> 5) * p12 + ((lane >> 4) & 1) * p2;
        atomicAdd(tile + sl * stride + n, acc.a[0]);
        if constexpr (!RN)
            if (mm == 0)
                atomicAdd(tile + stride + n, acc.rho[0]);
    }
    else if constexpr (C::W == 4)
    {
        // result register r of lane (q, i): row 4 r + q = (a, b) = (r, q), column i
        int const n = node0 + (lane >> 4) * p2 + ((lane & 15) >> 2);
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            atomicAdd(tile + slab * stride + n + r * p12, acc.a[r]);
            if constexpr (!RN)
                if (m == 0)
                    atomicAdd(tile + stride + n + r * p12, acc.rho[r]);
        }
    }
    else
    {
        int const i = lane >> 4;
        int const n = node0 + (i >> 1) * p12 + (i & 1) * p2 + ((lane >> 2) & 1);
        atomicAdd(tile + slab * stride + n, acc.a[0]);
        if constexpr (!RN)
            if (m == 0)
                atomicAdd(tile + stride + n, acc.rho[0]);
    }
}

} // namespace pc
} // namespace phx
