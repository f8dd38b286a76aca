// Hermite integrals of a batch of primitive quartets by one wave, in LDS: the shared front end of
// the one-wave kernels.
//
// A batch is np <= 64 primitive quartets.  Boys function and R^(n)_000 run with one lane per
// primitive quartet; the recursion R^(n)_h = X_ax R^(n+1)_{h-e} + (c-1) R^(n+1)_{h-2e} runs level by
// level over the whole batch, in place: a round of 64 Hermite indices reads only lower ones, so
// the rounds of a level go from the highest indices down.  A lane keeps its Hermite indices for
// all primitives and levels, so their recursion entries stay in registers; levels with at most 32
// (16) entries take two (four) primitives at a time.  All LDS traffic is the wave's own, in issue
// order, so there is no barrier.
#pragma once

#include "device_common.hpp"

namespace lbx
{
    // LDS ordering inside one wave: a wave's LDS operations execute in issue order, so only the
    // compiler has to be kept from moving loads and stores across this point.
    __device__ __forceinline__ void waveFence()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // The lane number as a value the compiler cannot see through: address arithmetic made from it
    // stays in the loop that uses it instead of being hoisted into registers.
    __device__ __forceinline__ int opaqueLane(int lane)
    {
        asm volatile("" : "+v"(lane));
        return lane;
    }

    // The lane's recursion entries (kRecTab format): its index among 16, 32 and 64 lanes.
    template <int L>
    struct RecLane
    {
        static constexpr int NR = ceilDiv(nHerm(L), 64);
        unsigned r16, r32, r64[NR];

        __device__ __forceinline__ void load(int lane)
        {
            constexpr int HL = nHerm(L);
            r16 = (lane & 15) < HL ? kRecTab.v[lane & 15] : 0;
            r32 = (lane & 31) < HL ? kRecTab.v[lane & 31] : 0;
#pragma unroll
            for (int r = 0; r < NR; r++)
                r64[r] = lane + 64 * r < HL ? kRecTab.v[lane + 64 * r] : 0;
        }
    };

    // A recursion entry unpacked for the primitives of one level.
    template <typename T>
    struct RecEntry
    {
        int s1, s2, ax;
        T c;

        __device__ __forceinline__ explicit RecEntry(unsigned rt)
        {
            asm volatile("" : "+v"(rt));   // unpacked per level, not kept across them
            s1 = rt & 2047;
            s2 = (rt >> 11) & 2047;
            ax = (rt >> 22) & 3;
            c = T(static_cast<int>(rt >> 24));
        }
        __device__ __forceinline__ T eval(const T *R, const T *pq) const { return fma(pq[ax], R[s1], c * R[s2]); }
    };

    template <int L, int LEV, typename T>
    __device__ __forceinline__ void recLevels(T *sR, const T *sInit, const T *sPQ, const RecLane<L> &rec, int np, int lane)
    {
        if constexpr (LEV >= 0)
        {
            constexpr int HL = nHerm(L), nh = nHerm(L - LEV);   // entries of this level, 0 included
            if constexpr (nh <= 32)
            {
                constexpr int W = nh <= 16 ? 16 : 32;
                const int h = lane & (W - 1);
                const RecEntry<T> e(W == 16 ? rec.r16 : rec.r32);
#pragma unroll 1
                for (int p = lane / W; p < np; p += 64 / W)
                    if (h < nh)
                    {
                        T *R = sR + p * HL;
                        const T v = e.eval(R, sPQ + 4 * p);
                        R[h] = h == 0 ? sInit[p * (L + 1) + LEV] : v;
                    }
            }
            else
            {
#pragma unroll
                for (int r = ceilDiv(nh, 64) - 1; r >= 0; r--)
                {
                    const int h = lane + 64 * r;
                    const RecEntry<T> e(rec.r64[r]);
#pragma unroll 1
                    for (int p = 0; p < np; p++)
                    {
                        T *R = sR + p * HL;
                        if (64 * r + 64 <= nh || h < nh)
                        {
                            const T v = e.eval(R, sPQ + 4 * p);
                            R[h] = r == 0 && h == 0 ? sInit[p * (L + 1) + LEV] : v;
                        }
                    }
                    waveFence();
                }
            }
            waveFence();
            recLevels<L, LEV - 1, T>(sR, sInit, sPQ, rec, np, lane);
        }
    }

    // R_tuv (order L) of np primitive quartets into sR[p * nHerm(L) + hermIdx]; pb / pk: the bra
    // and ket primitive of the lane's primitive quartet (read for lane < np).  sInit np (L + 1),
    // sPQ 4 np values.
    template <int L, typename T>
    __device__ __forceinline__ void hermiteBatch(T *sR, T *sInit, T *sPQ, const RecLane<L> &rec, int np, int lane,
                                                 const double4 *pb, const double4 *pk, const double *__restrict__ boys)
    {
        if (lane < np)
        {
            const double4 P = *pb, Q = *pk;
            const double pq = P.x * Q.x, ps = P.x + Q.x;
            const double alpha = pq / ps;
            const double X = P.y - Q.y, Y = P.z - Q.z, Z = P.w - Q.w;
            double F[L + 1];
            boysF<L>(alpha * (X * X + Y * Y + Z * Z), boys, F);
            double sc = kTwoPi52 / (pq * sqrt(ps));
#pragma unroll
            for (int m = 0; m <= L; m++)
            {
                F[m] *= sc;
                if (m < L)
                    sInit[lane * (L + 1) + m] = T(F[m]);
                sc *= -2.0 * alpha;
            }
            sPQ[4 * lane] = T(X);
            sPQ[4 * lane + 1] = T(Y);
            sPQ[4 * lane + 2] = T(Z);
            sR[lane * nHerm(L)] = T(F[L]);
        }
        waveFence();
        recLevels<L, L - 1, T>(sR, sInit, sPQ, rec, np, lane);
    }
}
