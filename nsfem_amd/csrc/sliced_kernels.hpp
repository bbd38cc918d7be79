// Row products on sliced rows (sliced ELLPACK), for systems whose rows are in
// locality order: the PCG solver with the factorized approximate inverse, one
// or two channels.
//
// A slice is 64 rows of one system, lane l of a wavefront on its row l; the
// slice's entries are stored column by column (entry k of all 64 rows side by
// side), so values and columns load as whole lines with no row bounds to wait
// for, a lane's gathers all go out together, and no lane reduction or barrier
// is needed.  Rows are sorted by entry count inside windows of the locality
// order, so a slice's rows have about the same count (padding entries have
// value 0 and the row's own column).  A row's terms are added in entry order
// with fused multiply-adds, as the lane-split rows add them.
//
// Bound by the matrix stream; on the P2 mass matrix with 2M rows, FP64 with the
// FP32 factor, two channels: direction 95 us (420 MB algorithmic, 4.4 TB/s;
// 476 MB of traffic), each of the factor's launches 41 us (156 MB, 3.8 TB/s),
// an iteration 224 us.  The lane-split kernels on colour-major rows took 160,
// 56 and 341 us at their best launch shape, 220, 141 and 585 us at the
// default one: a row's gathers came from up to seven colour regions, and the
// rows of 8 and 18 entries left lanes idle.  Chunks of consecutive entries
// with their products summed through LDS came to 96, 42 and 230 us, and
// 42 instead of 36 us an iteration at 240k rows (three phases and two barriers
// per chunk).
#pragma once

#include "kernels.hpp"

namespace nsfem
{
    // Rows of the locality order that are sorted by entry count together.
    constexpr int kSortWindow = 1024;
    // Workgroups of a kernel at most: every one of the next kernel re-sums all
    // partial sums of this one, and two of eight waves on every CU stream as
    // fast as four (2M rows: 224 and 220 us an iteration; 240k rows: the same).
    constexpr int kSliceGroups = 512;

    template <typename T>
    struct SlicedMatrix
    {
        const int4 * slices; // first row, rows, first entry, entries per row
        const int * column;
        const T * values;
    };

    // acc[c] = sum of the next K entries of the lane's row, from entry e on
    // (stride 64); K a compile-time count: their loads, then their gathers, go
    // out together.
    template <int K, int NCH, typename V, typename X>
    __device__ __forceinline__ void slicedStep(const SlicedMatrix<V> & A, int e, const X * __restrict__ x, V (&acc)[NCH])
    {
        V v[K];
        int col[K];
#pragma unroll
        for (int k = 0; k < K; k++)
        {
            v[k] = A.values[e + 64 * k];
            col[k] = A.column[e + 64 * k];
        }
        X xv[K][NCH];
#pragma unroll
        for (int k = 0; k < K; k++)
        {
#pragma unroll
            for (int c = 0; c < NCH; c++)
            {
                xv[k][c] = x[static_cast<long>(col[k]) * NCH + c];
            }
        }
#pragma unroll
        for (int k = 0; k < K; k++)
        {
#pragma unroll
            for (int c = 0; c < NCH; c++)
            {
                acc[c] = fmaT(v[k], static_cast<V>(xv[k][c]), acc[c]);
            }
        }
    }

    template <int NCH, typename V, typename X>
    __device__ __forceinline__ void slicedDot(const SlicedMatrix<V> & A, const int4 & s, const X * __restrict__ x, V (&acc)[NCH])
    {
#pragma unroll
        for (int c = 0; c < NCH; c++)
        {
            acc[c] = V(0);
        }
        int e = s.z + static_cast<int>(threadIdx.x & 63);
        int k = s.w;
        for (; k >= 8; k -= 8, e += 8 * 64)
        {
            slicedStep<8, NCH>(A, e, x, acc);
        }
        if (k >= 4)
        {
            slicedStep<4, NCH>(A, e, x, acc);
            k -= 4;
            e += 4 * 64;
        }
        if (k >= 2)
        {
            slicedStep<2, NCH>(A, e, x, acc);
            k -= 2;
            e += 2 * 64;
        }
        if (k >= 1)
        {
            slicedStep<1, NCH>(A, e, x, acc);
        }
    }

    // The wave's next slice as scalars (uniform over the wavefront).
    __device__ __forceinline__ int4 uniformSlice(const int4 * slices, int i)
    {
        return slices[__builtin_amdgcn_readfirstlane(i)];
    }

    // As pcgDirectionKernel with fused reductions: p = z + beta p, q = A z +
    // beta q, partial sums of p.q; bm.blocks holds ranges of slices.
    template <typename T, typename P, int W, int NCH>
    __global__ void __launch_bounds__(64 * W) slicedDirectionKernel(SlicedMatrix<T> A, const T * __restrict__ diag, BlockMap bm,
                                                                       SolveState st, const P * __restrict__ z, T * __restrict__ p,
                                                                       T * __restrict__ q)
    {
        constexpr int BLOCK = 64 * W;
        constexpr int PRE = W >= 8 ? 2 : 4; // partial sums per thread that load ahead
        __shared__ double sm[2 * NCH * W];
        __shared__ double shBeta[NCH];
        __shared__ int shAct[NCH];
        const int lb = logicalBlock(blockIdx.x, gridDim.x);
        const int4 range = bm.blocks[lb];
        if (st.flags[0])
        {
            return;
        }
        const FusedSlice sl = fusedSlice(bm, range, lb, 0, 0);
        const bool first = st.flags[1] != 0;
        FusedRhoLoads<NCH, BLOCK, PRE> fl;
        fusedRhoLoad<NCH, BLOCK, PRE>(st, sl, fl);
        bool pending = true;
        T beta[NCH];
        double part[NCH];
#pragma unroll
        for (int c = 0; c < NCH; c++)
        {
            beta[c] = T(0);
            part[c] = 0;
        }
        const int lane = static_cast<int>(threadIdx.x & 63);
        // every wave makes the same number of turns (the first has barriers)
        for (int base = range.x; base < range.y; base += W)
        {
            const int i = base + static_cast<int>(threadIdx.x >> 6);
            const bool has = i < range.y;
            const int4 s = uniformSlice(A.slices, has ? i : base);
            const int row = s.x + (lane < s.y ? lane : 0);
            const T dg = diag[row];
            P zr[NCH];
            T pr[NCH], qr[NCH], acc[NCH];
#pragma unroll
            for (int c = 0; c < NCH; c++)
            {
                const long j = static_cast<long>(row) * NCH + c;
                zr[c] = z[j];
                pr[c] = p[j];
                qr[c] = q[j];
            }
            if (has)
            {
                slicedDot<NCH>(A, s, z, acc);
            }
            if (pending)
            {
                pending = false;
                if (!fusedRhoFinish<NCH, BLOCK, PRE>(st, fl, sl, sm, shBeta, shAct))
                {
                    return;
                }
#pragma unroll
                for (int c = 0; c < NCH; c++)
                {
                    beta[c] = static_cast<T>(shBeta[c]);
                }
            }
            if (has && lane < s.y)
            {
#pragma unroll
                for (int c = 0; c < NCH; c++)
                {
                    const long j = static_cast<long>(row) * NCH + c;
                    const T zi = static_cast<T>(zr[c]);
                    const T az = fmaT(dg, zi, acc[c]);
                    const T pi = first ? zi : fmaT(beta[c], pr[c], zi);
                    const T qi = first ? az : fmaT(beta[c], qr[c], az);
                    p[j] = pi;
                    q[j] = qi;
                    part[c] = fma(static_cast<double>(pi), static_cast<double>(qi), part[c]);
                }
            }
        }
        blockSum<NCH, W>(part, sm);
        storePartial<NCH>(part, st.partials3, range.w);
    }

    // r = b - A x, |b|^2 and |r|^2 (pcgInitKernel with a nonzero guess).
    template <typename T, typename P, int W, int NCH>
    __global__ void __launch_bounds__(64 * W) slicedInitKernel(SlicedMatrix<T> A, const T * __restrict__ diag, BlockMap bm, SolveState st,
                                                                  const T * __restrict__ b, const T * __restrict__ x, T * r, P * rP)
    {
        __shared__ double sm[2 * NCH * W];
        const int4 range = bm.blocks[logicalBlock(blockIdx.x, gridDim.x)];
        double part[2 * NCH];
#pragma unroll
        for (int c = 0; c < 2 * NCH; c++)
        {
            part[c] = 0;
        }
        const int lane = static_cast<int>(threadIdx.x & 63);
        for (int i = range.x + static_cast<int>(threadIdx.x >> 6); i < range.y; i += W)
        {
            const int4 s = uniformSlice(A.slices, i);
            const int row = s.x + (lane < s.y ? lane : 0);
            const T dg = diag[row];
            T xr[NCH], br[NCH], acc[NCH];
#pragma unroll
            for (int c = 0; c < NCH; c++)
            {
                const long j = static_cast<long>(row) * NCH + c;
                xr[c] = x[j];
                br[c] = b[j];
            }
            slicedDot<NCH>(A, s, x, acc);
            if (lane < s.y)
            {
#pragma unroll
                for (int c = 0; c < NCH; c++)
                {
                    const long j = static_cast<long>(row) * NCH + c;
                    const T ri = br[c] - fmaT(dg, xr[c], acc[c]);
                    r[j] = ri;
                    if constexpr (!std::is_same_v<T, P>)
                    {
                        rP[j] = static_cast<P>(ri);
                    }
                    part[c] = fma(static_cast<double>(br[c]), static_cast<double>(br[c]), part[c]);
                    part[NCH + c] = fma(static_cast<double>(ri), static_cast<double>(ri), part[NCH + c]);
                }
            }
        }
        blockSum<2 * NCH, W>(part, sm);
        storePartial<2 * NCH>(part, st.partials, range.w);
    }

    // t = G r over the lower-colour entries.
    template <typename P, int W, int NCH>
    __global__ void __launch_bounds__(64 * W) slicedLowerKernel(SlicedMatrix<P> G, const P * __restrict__ diag, BlockMap bm, SolveState st,
                                                                   const P * __restrict__ r, P * __restrict__ t)
    {
        const int4 range = bm.blocks[logicalBlock(blockIdx.x, gridDim.x)];
        if (st.flags[0] || !systemActive<NCH>(st, range.z))
        {
            return;
        }
        const int lane = static_cast<int>(threadIdx.x & 63);
        for (int i = range.x + static_cast<int>(threadIdx.x >> 6); i < range.y; i += W)
        {
            const int4 s = uniformSlice(G.slices, i);
            const int row = s.x + (lane < s.y ? lane : 0);
            const P dg = diag[row];
            P rv[NCH], acc[NCH];
#pragma unroll
            for (int c = 0; c < NCH; c++)
            {
                rv[c] = r[static_cast<long>(row) * NCH + c];
            }
            slicedDot<NCH>(G, s, r, acc);
            if (lane < s.y)
            {
#pragma unroll
                for (int c = 0; c < NCH; c++)
                {
                    t[static_cast<long>(row) * NCH + c] = fmaT(dg, rv[c], acc[c]);
                }
            }
        }
    }

    // z = G^T t over the higher-colour entries, partial sums of rho = r.z.
    template <typename P, typename T, int W, int NCH>
    __global__ void __launch_bounds__(64 * W) slicedUpperKernel(SlicedMatrix<P> G, const P * __restrict__ diag, BlockMap bm, SolveState st,
                                                                   const P * __restrict__ t, P * __restrict__ z, const T * __restrict__ r)
    {
        __shared__ double sm[NCH * W];
        const int4 range = bm.blocks[logicalBlock(blockIdx.x, gridDim.x)];
        if (st.flags[0])
        {
            return;
        }
        double part[NCH];
#pragma unroll
        for (int c = 0; c < NCH; c++)
        {
            part[c] = 0;
        }
        if (systemActive<NCH>(st, range.z))
        {
            const int lane = static_cast<int>(threadIdx.x & 63);
            for (int i = range.x + static_cast<int>(threadIdx.x >> 6); i < range.y; i += W)
            {
                const int4 s = uniformSlice(G.slices, i);
                const int row = s.x + (lane < s.y ? lane : 0);
                const P dg = diag[row];
                P tv[NCH], acc[NCH];
                T rv[NCH];
#pragma unroll
                for (int c = 0; c < NCH; c++)
                {
                    const long j = static_cast<long>(row) * NCH + c;
                    tv[c] = t[j];
                    rv[c] = r[j];
                }
                slicedDot<NCH>(G, s, t, acc);
                if (lane < s.y)
                {
#pragma unroll
                    for (int c = 0; c < NCH; c++)
                    {
                        const long j = static_cast<long>(row) * NCH + c;
                        const P zi = fmaT(dg, tv[c], acc[c]);
                        z[j] = zi;
                        part[c] = fma(static_cast<double>(rv[c]), static_cast<double>(zi), part[c]);
                    }
                }
            }
        }
        blockSum<NCH, W>(part, sm);
        storePartial<NCH>(part, st.partials, range.w);
    }
} // namespace nsfem
