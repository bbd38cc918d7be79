#include "dense_inverse.hpp"

#include <stdexcept>

#include "ops.hpp"

namespace nsfem
{
    namespace
    {
        // Block Gauss-Jordan elimination in place, 32 columns a step (no
        // pivoting: the matrix is SPD).  A step reads and writes the whole
        // matrix once, so the inversion moves n / 32 times 16 n^2 bytes; the
        // 32 x 32 x 32 tile products run from LDS.
        constexpr int kNb = 32;

        // d = inverse of the pivot block (k0, k0); bad is set when a pivot is
        // not above 1e-10 of the original diagonal.
        __global__ void __launch_bounds__(kNb * kNb) gjPivotKernel(int n, int k0, const double * __restrict__ m,
                                                                   const double * __restrict__ diag, double * __restrict__ d, int * bad)
        {
            __shared__ double a[kNb][kNb + 1];
            const int i = threadIdx.x / kNb, j = threadIdx.x % kNb;
            a[i][j] = m[static_cast<size_t>(k0 + i) * n + k0 + j];
            __syncthreads();
            for (int p = 0; p < kNb; p++)
            {
                const double piv = a[p][p], aip = a[i][p], apj = a[p][j], aij = a[i][j];
                __syncthreads();
                if (threadIdx.x == 0 && !(piv > 1e-10 * fabs(diag[k0 + p])))
                {
                    *bad = 1;
                }
                const double r = 1.0 / piv;
                double v;
                if (i == p)
                {
                    v = j == p ? r : apj * r;
                }
                else
                {
                    v = j == p ? -aip * r : fma(-aip * r, apj, aij);
                }
                a[i][j] = v;
                __syncthreads();
            }
            d[i * kNb + j] = a[i][j];
        }

        // One tile column t: row[., t] = d m[k0.., t] and a copy of the tile
        // column's block of the pivot column, col[t, .] = m[t, k0..].
        __global__ void __launch_bounds__(kNb * 8) gjPanelKernel(int n, int k0, const double * __restrict__ m, const double * __restrict__ d,
                                                                 double * __restrict__ row, double * __restrict__ col)
        {
            __shared__ double sd[kNb][kNb + 1], sm[kNb][kNb + 1];
            const int t0 = blockIdx.x * kNb;
            const int x = threadIdx.x % kNb, y = threadIdx.x / kNb;
            for (int i = y; i < kNb; i += 8)
            {
                sd[i][x] = d[i * kNb + x];
                sm[i][x] = m[static_cast<size_t>(k0 + i) * n + t0 + x];
                col[static_cast<size_t>(t0 + i) * kNb + x] = m[static_cast<size_t>(t0 + i) * n + k0 + x];
            }
            __syncthreads();
            for (int i = y; i < kNb; i += 8)
            {
                double v = 0;
#pragma unroll 8
                for (int k = 0; k < kNb; k++)
                {
                    v = fma(sd[i][k], sm[k][x], v);
                }
                row[static_cast<size_t>(i) * n + t0 + x] = v;
            }
        }

        // Tile (r, c): the pivot block becomes d, its row d m, its column
        // -m d, the rest m - col row.
        __global__ void __launch_bounds__(kNb * 8) gjUpdateKernel(int n, int k0, double * __restrict__ m, const double * __restrict__ d,
                                                                  const double * __restrict__ row, const double * __restrict__ col)
        {
            __shared__ double sc[kNb][kNb + 1], sr[kNb][kNb + 1];
            const int c0 = blockIdx.x * kNb, r0 = blockIdx.y * kNb;
            const int x = threadIdx.x % kNb, y = threadIdx.x / kNb;
            const bool pr = r0 == k0, pc = c0 == k0;
            for (int i = y; i < kNb; i += 8)
            {
                sc[i][x] = col[static_cast<size_t>(r0 + i) * kNb + x];
                sr[i][x] = pc ? d[i * kNb + x] : row[static_cast<size_t>(i) * n + c0 + x];
            }
            __syncthreads();
            for (int i = y; i < kNb; i += 8)
            {
                double * to = m + static_cast<size_t>(r0 + i) * n + c0 + x;
                if (pr)
                {
                    *to = sr[i][x];
                    continue;
                }
                double v = pc ? 0.0 : *to;
#pragma unroll 8
                for (int k = 0; k < kNb; k++)
                {
                    v = fma(-sc[i][k], sr[k][x], v);
                }
                *to = v;
            }
        }

        template <typename T>
        __global__ void __launch_bounds__(256) gjStoreKernel(int n, int stride, const double * __restrict__ m, int ld, T * __restrict__ out)
        {
            for (long t = blockIdx.x * 256L + threadIdx.x; t < static_cast<long>(ld) * ld; t += gridDim.x * 256L)
            {
                const int i = static_cast<int>(t / ld), j = static_cast<int>(t % ld);
                out[t] = i < n && j < n ? static_cast<T>(0.5 * (m[static_cast<size_t>(i) * stride + j] + m[static_cast<size_t>(j) * stride + i])) : T(0);
            }
        }
    } // namespace

    template <typename T>
    bool denseInverseGpu(int n, const std::vector<double> & m, int ld, T * out, hipStream_t s)
    {
        if (n < 1 || ld < n || m.size() != static_cast<size_t>(n) * n)
        {
            throw std::invalid_argument("dense inverse: bad sizes");
        }
        // padded to whole tiles with an identity block
        const int N = (n + kNb - 1) / kNb * kNb;
        std::vector<double> padded(static_cast<size_t>(N) * N, 0.0), diag(N, 1.0);
        for (int i = 0; i < N; i++)
        {
            if (i < n)
            {
                std::copy(m.begin() + static_cast<size_t>(i) * n, m.begin() + static_cast<size_t>(i + 1) * n,
                          padded.begin() + static_cast<size_t>(i) * N);
                diag[i] = m[static_cast<size_t>(i) * n + i];
            }
            else
            {
                padded[static_cast<size_t>(i) * N + i] = 1.0;
            }
        }
        DeviceArray<double> a, dg, d(kNb * kNb), row(static_cast<size_t>(N) * kNb), col(static_cast<size_t>(N) * kNb);
        DeviceArray<int> bad(1);
        a.upload(padded);
        dg.upload(diag);
        fillInt(1, 0, bad.get(), s);
        const int tiles = N / kNb;
        for (int k = 0; k < tiles; k++)
        {
            gjPivotKernel<<<1, kNb * kNb, 0, s>>>(N, k * kNb, a.get(), dg.get(), d.get(), bad.get());
            gjPanelKernel<<<tiles, kNb * 8, 0, s>>>(N, k * kNb, a.get(), d.get(), row.get(), col.get());
            gjUpdateKernel<<<dim3(tiles, tiles), kNb * 8, 0, s>>>(N, k * kNb, a.get(), d.get(), row.get(), col.get());
        }
        gjStoreKernel<T><<<elementwiseGrid(static_cast<long>(ld) * ld), 256, 0, s>>>(n, N, a.get(), ld, out);
        NSFEM_HIP(hipGetLastError());
        NSFEM_HIP(hipStreamSynchronize(s));
        return bad.download()[0] == 0;
    }

    template bool denseInverseGpu<double>(int, const std::vector<double> &, int, double *, hipStream_t);
    template bool denseInverseGpu<float>(int, const std::vector<double> &, int, float *, hipStream_t);
} // namespace nsfem
