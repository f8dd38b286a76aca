// Density-fitted (RI) Coulomb and exchange matrices from the dense 3-index and 2-index
// integrals of the library (the natural consumer of eri3()/eri2(), eri3.cpp:7-46,
// eri2.cpp:27-72; the reference has no J/K build).  With B_P(mn) = (mn|P), V = (P|Q) = L L^T
// and the fitted tensor W_P = sum_Q (L^-1)_PQ B_Q (so that sum_P W_P W_P^T = B V^-1 B^T):
//   J = sum_P W_P h_P,   h_P = sum_mn W_P(mn) D_mn
//   K = sum_P W_P D W_P   (also of a D that is not symmetric)
// W depends on the geometry only: the first call builds it (eri3, a transpose to P-major, eri2,
// the Cholesky factorisation, one triangular solve) and the context keeps it, so every later
// call (an SCF iteration) costs one or two passes over W for J and, for K, the products
// T_P = W_P D and K = sum_P T_P W_P^T (k = nbf * naux), on FP64 MFMA kernels of this file.
// Factorisation by rocSOLVER, the triangular solve by rocBLAS.
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include "device_common.hpp"
#include "lbx_internal.hpp"

#include <algorithm>
#include <memory>
#include <string>

namespace lbx
{
    namespace
    {
        // out (cols, rows) = in (rows, cols)^T, both row-major, through 32 x 32 LDS tiles
        __global__ __launch_bounds__(256) void transposeKernel(const double *__restrict__ in,
                                                               double *__restrict__ out, long long rows,
                                                               long long cols)
        {
            __shared__ double tile[32][33];
            const long long tr = (rows + 31) / 32, tc = (cols + 31) / 32;
            for (long long t = blockIdx.x; t < tr * tc; t += gridDim.x)
            {
                const long long r0 = (t / tc) * 32, c0 = (t % tc) * 32;
                const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
                for (int k = y; k < 32; k += 8)
                {
                    const long long r = r0 + k, c = c0 + x;
                    tile[k][x] = (r < rows && c < cols) ? in[r * cols + c] : 0.0;
                }
                __syncthreads();
                for (int k = y; k < 32; k += 8)
                {
                    const long long c = c0 + k, r = r0 + x;
                    if (c < cols && r < rows)
                        out[c * rows + r] = tile[x][k];
                }
                __syncthreads();
            }
        }

        // sum over the workgroup's 256 threads, valid in thread 0
        __device__ __forceinline__ double blockSum256(double x)
        {
            __shared__ double part[4];
            x = waveSum(x);
            if ((threadIdx.x & 63) == 0)
                part[threadIdx.x >> 6] = x;
            __syncthreads();
            return part[0] + part[1] + part[2] + part[3];
        }

        // h_P = sum_mn W_P(mn) D_mn, one workgroup per P
        __global__ __launch_bounds__(256) void fitDotKernel(const double *__restrict__ W, const double *__restrict__ D,
                                                            double *__restrict__ h, long long n2)
        {
            const double *w = W + blockIdx.x * n2;
            double s = 0.0;
            for (long long i = threadIdx.x; i < n2; i += 256)
                s = fma(w[i], D[i], s);
            s = blockSum256(s);
            if (threadIdx.x == 0)
                h[blockIdx.x] = s;
        }

        // out = sum over the P of group blockIdx.y of W_P h_P; each group has an n2-sized output of its own
        __global__ __launch_bounds__(256) void fitCoulombKernel(const double *__restrict__ W, const double *__restrict__ h,
                                                                double *__restrict__ out, long long n2, int naux, int group)
        {
            const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
            if (i >= n2)
                return;
            const int p0 = blockIdx.y * group, p1 = min(naux, p0 + group);
            double s = 0.0;
#pragma unroll 8
            for (int p = p0; p < p1; p++)
                s = fma(W[p * n2 + i], h[p], s);
            out[blockIdx.y * n2 + i] = s;
        }

        // out[i] = sum of the groups' outputs, in order (64 elements a workgroup, its waves a quarter of
        // the groups each)
        __global__ __launch_bounds__(256) void sumGroupsKernel(const double *__restrict__ in, double *__restrict__ out,
                                                               long long n2, int groups)
        {
            __shared__ double quarter[4][64];
            const int j = threadIdx.x & 63, w = threadIdx.x >> 6;
            const long long i = min(blockIdx.x * 64LL + j, n2 - 1);
            double s = 0.0;
#pragma unroll 8
            for (int g = groups * w / 4; g < groups * (w + 1) / 4; g++)
                s += in[g * n2 + i];
            quarter[w][j] = s;
            __syncthreads();
            if (w == 0)
                out[i] = (quarter[0][j] + quarter[1][j]) + (quarter[2][j] + quarter[3][j]);
        }

        // Two things that a K needs, in one launch.  Workgroups below naux: h_P = tr(T_P) where
        // T_P = W_P D is there already.  The kFlagBlocks others: whether D is symmetric to rounding,
        // flags[b] = 1 where it is not; K is then not symmetric either, and its upper triangle is made too.
        constexpr int kFlagBlocks = 256;
        __global__ __launch_bounds__(256) void traceSymmetryKernel(const double *__restrict__ T, const double *__restrict__ D,
                                                                   double *__restrict__ h, int *flags, int n, int naux)
        {
            const long long tot = static_cast<long long>(n) * n;
            if (static_cast<int>(blockIdx.x) < naux)
            {
                const double *t = T + blockIdx.x * tot;
                double s = 0.0;
                for (int i = threadIdx.x; i < n; i += 256)
                    s += t[i * (n + 1LL)];
                s = blockSum256(s);
                if (threadIdx.x == 0)
                    h[blockIdx.x] = s;
                return;
            }
            const int b = static_cast<int>(blockIdx.x) - naux;
            bool differ = false;
            for (long long e = b * 256LL + threadIdx.x; e < tot; e += kFlagBlocks * 256LL)
            {
                const int i = static_cast<int>(e / n), j = static_cast<int>(e % n);
                if (j < i)
                {
                    const double x = D[e], y = D[static_cast<long long>(j) * n + i];
                    differ |= fabs(x - y) > 1e-14 * fmax(fabs(x), fabs(y));
                }
            }
            const int any = __syncthreads_or(differ);
            if (threadIdx.x == 0)
                flags[b] = any;
        }

        // the flags of traceSymmetryKernel (all 256 threads call)
        __device__ __forceinline__ bool asymmetric(const int *flags) { return __syncthreads_or(flags[threadIdx.x]); }

        // tile number -> tile: the tiles with row >= column first, then the others
        __device__ __forceinline__ void tileOf(int tile, int nt, int &tr, int &tc)
        {
            const int lower = nt * (nt + 1) / 2;
            if (tile < lower)
            {
                int t = tile;
                tr = 0;
                while (t > tr)
                    t -= ++tr;
                tc = t;
            }
            else
            {
                int t = tile - lower;
                tc = 1;
                while (t >= tc)
                    t -= tc++;
                tr = t;
            }
        }

        // K from the splits' parts of each 64 x 64 tile, added in order (one workgroup per row of a tile,
        // its waves a quarter of the splits each); the upper triangle from the lower one unless D is not
        // symmetric.
        __global__ __launch_bounds__(256) void sumTilesKernel(const double *__restrict__ parts, double *__restrict__ K, int n,
                                                              int splits, const int *flags)
        {
            const bool full = asymmetric(flags);
            const int nt = (n + 63) / 64, tile = blockIdx.x / 64, r = blockIdx.x % 64;
            if (!full && tile >= nt * (nt + 1) / 2)
                return;
            int tr, tc;
            tileOf(tile, nt, tr, tc);
            __shared__ double quarter[4][64];
            const int j = threadIdx.x & 63, w = threadIdx.x >> 6;
            const int s0 = splits * w / 4, s1 = splits * (w + 1) / 4;
            const double *in = parts + (static_cast<long long>(tile) * splits * 64 + r) * 64 + j;
            double v = 0.0;
#pragma unroll 8
            for (int k = s0; k < s1; k++)
                v += in[k * 4096LL];
            quarter[w][j] = v;
            __syncthreads();
            const int row = tr * 64 + r, col = tc * 64 + j;
            if (w > 0 || row >= n || col >= n || (!full && col > row))
                return;
            v = (quarter[0][j] + quarter[1][j]) + (quarter[2][j] + quarter[3][j]);
            K[static_cast<long long>(row) * n + col] = v;
            if (!full)
                K[static_cast<long long>(col) * n + row] = v;
        }

        // upper triangle from the lower one, unless it has been made (D not symmetric)
        __global__ __launch_bounds__(256) void mirrorKernel(double *K, int n, const int *flags)
        {
            if (asymmetric(flags))
                return;
            const long long tot = static_cast<long long>(n) * n;
            for (long long e = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; e < tot;
                 e += static_cast<long long>(gridDim.x) * blockDim.x)
            {
                const int i = static_cast<int>(e / n), j = static_cast<int>(e % n);
                if (j > i)
                    K[e] = K[static_cast<long long>(j) * n + i];
            }
        }

        // C[m n + c] (+)= sum_k A[m + n k] B[c + n k]: both operands have the row index contiguous, so
        // the A and B fragments of v_mfma_f64_16x16x4f64 load straight from memory in 128-byte
        // segments.  A workgroup of 2 x 2 waves makes a 64 x 64 tile, a wave 32 x 32 of it (four
        // MFMAs per four loads, the next 16 k fetched while 16 are multiplied); the waves' shared
        // fragments meet in L1.
        //   SPLIT = false: T_P = W_P D column by column, A = D, B = W_P (k < n, C stored;
        //     blockIdx.y = P)
        //   SPLIT = true:  K = sum_P T_P W_P^T with k = (P, l) running over n naux: for a small n
        //     the n x n tiles alone leave the chip idle (nine tiles at n = 192), so k is split over
        //     `splits` workgroups per tile, each with a part of its own that sumTilesKernel adds up
        //     (atomics into K took the same time and made its last bits differ from call to call);
        //     one split: C is K itself.  The tiles with row >= column come first (K of a symmetric D
        //     is symmetric), then the others, which return at once unless the flags say that D is not
        //     symmetric.
        // At n = 192, naux = 904 (k = 1.7e5) a J and K call takes 0.68 ms, 38 TFLOP/s over both
        // products (library GEMMs, whose few tiles left the chip idle: 19.5 ms).
        template <bool SPLIT>
        __global__ __launch_bounds__(256) void panelGemm(const double *__restrict__ A, const double *__restrict__ B,
                                                         double *__restrict__ C, int n, long long kTotal, long long kChunk,
                                                         int splits, const int *flags)
        {
            const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
            const int g = lane >> 4, j = lane & 15;
            const int nt = (n + 63) / 64;
            int tr, tc;
            long long k0, k1;
            if constexpr (SPLIT)
            {
                // the tiles of one split are `splits` workgroups apart (a multiple of 8), so one XCD's
                // L2 serves them
                const int tile = blockIdx.x / splits;
                if (tile >= nt * (nt + 1) / 2 && !asymmetric(flags))
                    return;
                tileOf(tile, nt, tr, tc);
                k0 = (blockIdx.x % splits) * kChunk;
                k1 = min(kTotal, k0 + kChunk);
            }
            else
            {
                tr = blockIdx.x / nt;
                tc = blockIdx.x % nt;
                k0 = 0;
                k1 = kTotal;
                B += blockIdx.y * static_cast<long long>(n) * n;
                C += blockIdx.y * static_cast<long long>(n) * n;
            }
            const int r0 = tr * 64 + (wave >> 1) * 32, c0 = tc * 64 + (wave & 1) * 32;
            v4d acc[2][2];
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++)
                    acc[x][y] = v4d{0, 0, 0, 0};
            // rows past n read row n - 1; their results are not stored
            const int ra[2] = {min(r0 + j, n - 1), min(r0 + 16 + j, n - 1)};
            const int cb[2] = {min(c0 + j, n - 1), min(c0 + 16 + j, n - 1)};
            auto load = [&](long long k, double (&a)[4][2], double (&b)[4][2]) {
#pragma unroll
                for (int s = 0; s < 4; s++)
                {
                    const long long kk = k + 4 * s + g;
                    const bool in = kk < k1;
                    const long long off = (in ? kk : k1 - 1) * n;
#pragma unroll
                    for (int x = 0; x < 2; x++)
                    {
                        const double v = A[off + ra[x]];
                        a[s][x] = in ? v : 0.0;
                        b[s][x] = B[off + cb[x]];
                    }
                }
            };
            double a[4][2], b[4][2], an[4][2], bn[4][2];
            if (k0 < k1)
            {
                load(k0, a, b);
                for (long long k = k0; k < k1; k += 16)
                {
                    if (k + 16 < k1)
                        load(k + 16, an, bn);
#pragma unroll
                    for (int s = 0; s < 4; s++)
#pragma unroll
                        for (int x = 0; x < 2; x++)
#pragma unroll
                            for (int y = 0; y < 2; y++)
                                acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s][x], b[s][y], acc[x][y], 0, 0, 0);
#pragma unroll
                    for (int s = 0; s < 4; s++)
#pragma unroll
                        for (int x = 0; x < 2; x++)
                        {
                            a[s][x] = an[s][x];
                            b[s][x] = bn[s][x];
                        }
                }
            }
            // accumulator element r of lane (g, j): row 4 r + g, column j
            const bool parts = SPLIT && splits > 1;
            if (parts)
                C += blockIdx.x * 4096LL;
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                    {
                        const int row = r0 + 16 * x + 4 * r + g, col = c0 + 16 * y + j;
                        if (parts)
                            C[(row & 63) * 64 + (col & 63)] = acc[x][y][r];
                        else if (row < n && col < n)
                            C[static_cast<long long>(row) * n + col] = acc[x][y][r];
                    }
        }

        void rb(rocblas_status s, const char *what)
        {
            if (s != rocblas_status_success)
                throw Error(s == rocblas_status_memory_error ? LBX_ERR_NOMEM : LBX_ERR_HIP,
                            std::string(what) + " failed (rocblas status " + std::to_string(static_cast<int>(s)) + ")");
        }

        struct Handle
        {
            rocblas_handle h = nullptr;
            explicit Handle(hipStream_t s)
            {
                rb(rocblas_create_handle(&h), "rocblas_create_handle");
                rb(rocblas_set_stream(h, s), "rocblas_set_stream");
            }
            ~Handle()
            {
                if (h)
                    (void)rocblas_destroy_handle(h);
            }
        };

        struct Buf
        {
            void *p = nullptr;
            explicit Buf(size_t bytes) { LBX_HIP(hipMalloc(&p, bytes ? bytes : 1)); }
            ~Buf()
            {
                if (p)
                    (void)hipFree(p);
            }
            double *d() const { return static_cast<double *>(p); }
        };
    }

    void riJK(lbx_context *ctx, Context &c, hipStream_t stream, long long n, long long naux, const double *D,
              double *J, double *K)
    {
        std::lock_guard<std::mutex> lk(c.ri_mu);
        const long long n2 = n * n;
        if (K && !c.ri_t)
            c.ri_t = c.alloc<double>(static_cast<size_t>(n2 * naux));
        if (K && !c.ri_flags)
            c.ri_flags = c.alloc<int>(kFlagBlocks);
        if (!c.ri_ready)
        {
            Handle h(stream);
            if (!c.ri_h)
                c.ri_h = c.alloc<double>(static_cast<size_t>(naux));
            if (!c.ri_w)
                c.ri_w = c.alloc<double>(static_cast<size_t>(n2 * naux));
            // dense (mn|P), mn-major as the eri3 entry writes it, then P-major into W's buffer
            std::unique_ptr<Buf> tmp;
            double *raw = c.ri_t;
            if (!raw)
            {
                tmp = std::make_unique<Buf>(sizeof(double) * n2 * naux);
                raw = tmp->d();
            }
            {
                const int rc = lbx_eri3(ctx, raw);
                if (rc != LBX_OK)
                    throw Error(rc, std::string("lbx_ri_jk: ") + lbx_last_error());
            }
            {
                const long long tiles = ((n2 + 31) / 32) * ((naux + 31) / 32);
                const int grid = static_cast<int>(tiles < 65536 ? tiles : 65536);
                hipLaunchKernelGGL(transposeKernel, dim3(grid), dim3(256), 0, stream, raw, c.ri_w, n2, naux);
                LBX_HIP(hipGetLastError());
            }
            Buf V(sizeof(double) * naux * naux);
            {
                const int rc = lbx_eri2(ctx, V.d());
                if (rc != LBX_OK)
                    throw Error(rc, std::string("lbx_ri_jk: ") + lbx_last_error());
            }
            // V = L L^T (V symmetric: its row-major storage is also its column-major storage);
            // the factorisation takes 32-bit sizes, the 3-index products rocBLAS's 64-bit
            // entries (nbf^2 naux exceeds 2^31 elements at a few hundred functions)
            const int NA = static_cast<int>(naux);
            Buf info(sizeof(rocblas_int));
            rb(rocsolver_dpotrf(h.h, rocblas_fill_lower, NA, V.d(), NA, static_cast<rocblas_int *>(info.p)),
               "rocsolver_dpotrf");
            rocblas_int hinfo = 0;
            LBX_HIP(hipMemcpyAsync(&hinfo, info.p, sizeof(hinfo), hipMemcpyDeviceToHost, stream));
            LBX_HIP(hipStreamSynchronize(stream));
            if (hinfo != 0)
                throw Error(LBX_ERR_STATE, "lbx_ri_jk: the auxiliary metric (P|Q) is not positive definite (pivot " +
                                                   std::to_string(hinfo) + ")");
            // W = X L^-T with X column-major n2 x naux (column P = the P-major block B_P)
            const double one = 1.0;
            rb(rocblas_dtrsm_64(h.h, rocblas_side_right, rocblas_fill_lower, rocblas_operation_transpose,
                                rocblas_diagonal_non_unit, n2, naux, &one, V.d(), naux, c.ri_w, n2),
               "rocblas_dtrsm (W = X L^-T)");
            LBX_HIP(hipStreamSynchronize(stream));
            c.ri_ready = true;
        }
        const int ni = static_cast<int>(n);
        // K in splits of k, so that about 1024 workgroups share it, at least 256 k each; J in groups of
        // P, so that about 2048 share the pass over W
        const long long nt2 = (n + 63) / 64 * ((n + 63) / 64), tiles = (nt2 + (n + 63) / 64) / 2;
        long long splits = std::min(std::max<long long>(1, 1024 / tiles), (n * naux + 255) / 256);
        splits = (splits + 7) / 8 * 8;
        long long jGroup = std::max<long long>(8, naux * ((n2 + 255) / 256) / 2048);
        if (!c.ri_part)
        {
            // one buffer for the parts of K, then of J: up to 80 MiB at 1000 functions, 8 nbf^2 values
            // where tiles are many.  Without it K and J are made in one part.
            const long long parts = std::max(nt2 * splits * 4096, (naux + jGroup - 1) / jGroup * n2);
            c.ri_part = static_cast<double *>(c.take(sizeof(double) * parts));
        }
        if (!c.ri_part)
        {
            splits = 1;
            jGroup = naux;
        }
        auto blocks1d = [](long long m) { return dim3(static_cast<int>(std::min<long long>((m + 255) / 256, 65536))); };
        if (K)
        {
            // T_P = D^T W_P as panelGemm reads its operands; blockIdx.y holds at most 65535 auxiliary
            // functions
            const int nt = (ni + 63) / 64;
            for (long long p0 = 0; p0 < naux; p0 += 65535)
            {
                const int np = static_cast<int>(std::min<long long>(65535, naux - p0));
                hipLaunchKernelGGL((panelGemm<false>), dim3(nt * nt, np), dim3(256), 0, stream, D, c.ri_w + p0 * n2,
                                   c.ri_t + p0 * n2, ni, n, n, 1, nullptr);
            }
            hipLaunchKernelGGL(traceSymmetryKernel, dim3(static_cast<int>(naux) + kFlagBlocks), dim3(256), 0, stream,
                               c.ri_t, D, c.ri_h, c.ri_flags, ni, static_cast<int>(naux));
            // K = sum_P T_P^T W_P
            const long long kTotal = n * naux;
            const long long chunk = ((kTotal + splits - 1) / splits + 15) / 16 * 16;
            hipLaunchKernelGGL((panelGemm<true>), dim3(static_cast<unsigned>(splits * nt * nt)), dim3(256), 0, stream,
                               c.ri_t, c.ri_w, splits > 1 ? c.ri_part : K, ni, kTotal, chunk, static_cast<int>(splits),
                               c.ri_flags);
            if (splits > 1)
                hipLaunchKernelGGL(sumTilesKernel, dim3(nt * nt * 64), dim3(256), 0, stream, c.ri_part, K, ni,
                                   static_cast<int>(splits), c.ri_flags);
            else
                hipLaunchKernelGGL(mirrorKernel, blocks1d(n2), dim3(256), 0, stream, K, ni, c.ri_flags);
        }
        else
            hipLaunchKernelGGL(fitDotKernel, dim3(static_cast<int>(naux)), dim3(256), 0, stream, c.ri_w, D, c.ri_h, n2);
        const int bx = static_cast<int>((n2 + 255) / 256), groups = static_cast<int>((naux + jGroup - 1) / jGroup);
        hipLaunchKernelGGL(fitCoulombKernel, dim3(bx, groups), dim3(256), 0, stream, c.ri_w, c.ri_h,
                           groups > 1 ? c.ri_part : J, n2, static_cast<int>(naux), static_cast<int>(jGroup));
        if (groups > 1)
            hipLaunchKernelGGL(sumGroupsKernel, dim3(static_cast<int>((n2 + 63) / 64)), dim3(256), 0, stream, c.ri_part, J,
                               n2, groups);
        LBX_HIP(hipGetLastError());
        LBX_HIP(hipStreamSynchronize(stream));
    }
}
