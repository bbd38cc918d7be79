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
// 486 MB of traffic), each of the factor's launches 41 us (156 MB, 3.8 TB/s),
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
    // Workgroups of a kernel, rounded up per system: every one of the next kernel re-sums all
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

    // ------------------------------------------------------------------
    // Four to 32 channels on the same rows in CSR form: one lane per channel
    // (a gathered column is NCH contiguous values), workgroups of 1,024
    // threads.  bm.blocks holds ranges of rows.
    //
    // Every workgroup of the next kernel re-sums this one's partial sums, NCH
    // for each workgroup, so few and large ones: one on every CU, two where
    // the vectors are so long that the sums do not count.  P2 mass matrix, 16
    // channels, mixed: an iteration at 40k pressure nodes 92 us (128 / 512
    // workgroups 153 / 96), at 500k 1,149 us with 512 (1,372 with 256).  The
    // kernels before, 64 rows to a workgroup in colour order, took 200 and
    // 2,511 us: direction 82 -> 35, each factor launch 47 -> 18 us at 40k.
    // ------------------------------------------------------------------
    constexpr int kWideBlock = 1024;
    constexpr int kWideWaves = kWideBlock / 64;
    constexpr int kWideGroups = 256, kWideGroupsLong = 512;
    constexpr long kWideLong = 8L << 20; // values of a vector from which on two pay

    // Rows range.x + t / NCH, + kWideBlock / NCH, ...: own(row) loads the row's
    // operands, part(row, acc) takes its product.  The next row's bounds load
    // with the current row's entries; U entries go out together.  begin() runs
    // once, behind the first row's loads (every thread; false ends the kernel).
    template <int U, int NCH, typename V, typename X, typename Begin, typename Own, typename Part>
    __device__ __forceinline__ bool wideRows(const int * __restrict__ start, const int * __restrict__ end, const int * __restrict__ column,
                                             const V * __restrict__ values, int4 range, const X * __restrict__ x, Begin begin, Own own,
                                             Part part)
    {
        constexpr int step = kWideBlock / NCH;
        const int c = static_cast<int>(threadIdx.x) % NCH;
        int row = range.x + static_cast<int>(threadIdx.x) / NCH;
        int rs = row < range.y ? row : range.x;
        int j0 = start[rs], j1 = end[rs];
        if (!begin())
        {
            return false;
        }
        for (int base = range.x; base < range.y; base += step, row += step)
        {
            const bool valid = row < range.y;
            own(rs);
            const int next = row + step < range.y ? row + step : range.x;
            const int n0 = start[next], n1 = end[next];
            const V acc = channelRowDot<U, NCH>(j0, valid ? j1 : j0, column, values, x);
            if (valid)
            {
                part(row, acc);
            }
            rs = next;
            j0 = n0;
            j1 = n1;
        }
        return true;
    }

    template <typename T, typename P, int NCH>
    __global__ void __launch_bounds__(kWideBlock, 8) wideDirectionKernel(McgsMatrix<T> A, BlockMap bm, SolveState st,
                                                                         const P * __restrict__ z, T * __restrict__ p, T * __restrict__ q)
    {
        constexpr int PRE = 4; // 256 workgroups' partial sums of 16 channels
        __shared__ double sm[2 * NCH * kWideWaves];
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
        FusedRhoLoads<NCH, kWideBlock, PRE> fl;
        fusedRhoLoad<NCH, kWideBlock, PRE>(st, sl, fl);
        const int c = static_cast<int>(threadIdx.x) % NCH;
        T beta = T(0), dg = T(0), pr = T(0), qr = T(0);
        P zr = P(0);
        double sum = 0;
        const bool go = wideRows<4, NCH>(
            A.rowStart, A.rowStart + 1, A.column, A.values, range, z,
            [&]()
            {
                const bool any = fusedRhoFinish<NCH, kWideBlock, PRE>(st, fl, sl, sm, shBeta, shAct);
                beta = static_cast<T>(shBeta[c]);
                return any;
            },
            [&](int row)
            {
                const long i = static_cast<long>(row) * NCH + c;
                dg = A.diag[row];
                zr = z[i];
                pr = p[i];
                qr = q[i];
            },
            [&](int row, T acc)
            {
                const long i = static_cast<long>(row) * NCH + c;
                const T zi = static_cast<T>(zr);
                const T az = fmaT(dg, zi, acc);
                const T pi = first ? zi : fmaT(beta, pr, zi);
                const T qi = first ? az : fmaT(beta, qr, az);
                p[i] = pi;
                q[i] = qi;
                sum = fma(static_cast<double>(pi), static_cast<double>(qi), sum);
            });
        if (!go)
        {
            return;
        }
        const double total = channelBlockSum<NCH, kWideWaves>(sum, sm);
        storeChannelPartial<NCH, NCH>(total, st.partials3, range.w, 0);
    }

    template <typename T, typename P, int NCH>
    __global__ void __launch_bounds__(kWideBlock, 8) wideInitKernel(McgsMatrix<T> A, BlockMap bm, SolveState st, const T * __restrict__ b,
                                                                    const T * __restrict__ x, T * r, P * rP)
    {
        __shared__ double sm[2 * NCH * kWideWaves];
        const int4 range = bm.blocks[logicalBlock(blockIdx.x, gridDim.x)];
        const int c = static_cast<int>(threadIdx.x) % NCH;
        T dg = T(0), xr = T(0), br = T(0);
        double bb = 0, rr = 0;
        wideRows<4, NCH>(
            A.rowStart, A.rowStart + 1, A.column, A.values, range, x, []() { return true; },
            [&](int row)
            {
                const long i = static_cast<long>(row) * NCH + c;
                dg = A.diag[row];
                xr = x[i];
                br = b[i];
            },
            [&](int row, T acc)
            {
                const long i = static_cast<long>(row) * NCH + c;
                const T ri = br - fmaT(dg, xr, acc);
                r[i] = ri;
                if constexpr (!std::is_same_v<T, P>)
                {
                    rP[i] = static_cast<P>(ri);
                }
                bb = fma(static_cast<double>(br), static_cast<double>(br), bb);
                rr = fma(static_cast<double>(ri), static_cast<double>(ri), rr);
            });
        channelBlockSum2<NCH, kWideWaves>(bb, rr, sm);
        storeChannelPartial<NCH, 2 * NCH>(bb, st.partials, range.w, 0);
        storeChannelPartial<NCH, 2 * NCH>(rr, st.partials, range.w, NCH);
    }

    template <typename P, int NCH>
    __global__ void __launch_bounds__(kWideBlock, 8) wideLowerKernel(McgsMatrix<P> G, BlockMap bm, SolveState st, const P * __restrict__ r,
                                                                     P * __restrict__ t)
    {
        const int4 range = bm.blocks[logicalBlock(blockIdx.x, gridDim.x)];
        if (st.flags[0] || !systemActive<NCH>(st, range.z))
        {
            return;
        }
        const int c = static_cast<int>(threadIdx.x) % NCH;
        P dg = P(0), rv = P(0);
        wideRows<8, NCH>(
            G.rowStart, G.rowSplit, G.column, G.values, range, r, []() { return true; },
            [&](int row)
            {
                dg = G.diag[row];
                rv = r[static_cast<long>(row) * NCH + c];
            },
            [&](int row, P acc) { t[static_cast<long>(row) * NCH + c] = fmaT(dg, rv, acc); });
    }

    template <typename P, typename T, int NCH>
    __global__ void __launch_bounds__(kWideBlock, 8) wideUpperKernel(McgsMatrix<P> G, BlockMap bm, SolveState st, const P * __restrict__ t,
                                                                     P * __restrict__ z, const T * __restrict__ r)
    {
        __shared__ double sm[NCH * kWideWaves];
        const int4 range = bm.blocks[logicalBlock(blockIdx.x, gridDim.x)];
        if (st.flags[0])
        {
            return;
        }
        const int c = static_cast<int>(threadIdx.x) % NCH;
        double sum = 0;
        if (systemActive<NCH>(st, range.z))
        {
            P dg = P(0), tv = P(0);
            T rv = T(0);
            wideRows<8, NCH>(
                G.rowSplit, G.rowStart + 1, G.column, G.values, range, t, []() { return true; },
                [&](int row)
                {
                    const long i = static_cast<long>(row) * NCH + c;
                    dg = G.diag[row];
                    tv = t[i];
                    rv = r[i];
                },
                [&](int row, P acc)
                {
                    const long i = static_cast<long>(row) * NCH + c;
                    const P zi = fmaT(dg, tv, acc);
                    z[i] = zi;
                    sum = fma(static_cast<double>(rv), static_cast<double>(zi), sum);
                });
        }
        const double total = channelBlockSum<NCH, kWideWaves>(sum, sm);
        storeChannelPartial<NCH, NCH>(total, st.partials, range.w, 0);
    }
} // namespace nsfem
