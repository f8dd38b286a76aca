// One-wave-per-quartet form of the nuclear-gradient kernel (the quantities of grad.hpp), its
// transforms on MFMA.
//
// Per bra primitive pair i and 16-column tile of cd, with W[ab][cd] the density weights:
//   Y[h][cd] = sum_ab Eb_i[h][ab] W[ab][cd]
//   per ket primitive pair k:
//     S[h'][cd] += sum_g R_ik[h' + g] Ek_k[g][cd]      h' up to order l_a + l_b + 1
//     Q[g][cd]   = sum_h R_ik[g + h] Y[h][cd]
//     T_ik,x = sum_{h,cd} Y[h][cd] S_k[h + e_x][cd]    (S_k: k's contribution to S)
//     V_ik,x = sum_{g,cd} Ek'_k,x[g][cd] Q[g][cd]
//   U_i,x = sum_{ab,cd} W[ab][cd] sum_h Eb'_i,x[h][ab] S[h][cd]
// so a primitive quartet takes two products with R (the shifted R of T is in the extra rows of S,
// the three directions of V share Q) where the form of grad.hpp takes five, and R is built once
// per primitive quartet for all columns.  W is computed in the registers that feed it to MFMA (the
// B operand of Y, and the layout of the U accumulators); Y goes from its accumulators straight
// into the B operand of Q, S into that of U; only T reads Y through LDS, shifted by a row.
#pragma once

#include "grad.hpp"

namespace lbx
{
    template <int LA, int LB, int LC, int LD, typename T>
    struct GWPlan
    {
        static constexpr int L1 = LA + LB + LC + LD + 1, HL1 = nHerm(L1);
        static constexpr int HP = nHerm(LA + LB), HP1 = nHerm(LA + LB + 1), HQ = nHerm(LC + LD);
        static constexpr int SB = nSph(LB), SD = nSph(LD), SP = nSph(LA) * SB, SQ = nSph(LC) * SD;
        static constexpr int NQ = ceilDiv(SQ, 16), KQ = ceilDiv(HQ, 4);
        static constexpr int TP = ceilDiv(HP, 16), TP1 = ceilDiv(HP1, 16), TQ = ceilDiv(HQ, 16), TS = ceilDiv(SP, 16);
        // K steps over accumulator rows: element r of a tile holds rows 4 r .. 4 r + 3
        static constexpr int KP = ceilDiv(HP, 4), KS = ceilDiv(SP, 4);
        // primitive quartets whose R is held at a time: 10 KiB of LDS
        static constexpr int PB0 = 10240 / (HL1 * static_cast<int>(sizeof(T)));
        static constexpr int PB = PB0 < 1 ? 1 : (PB0 > 64 ? 64 : PB0);
        static constexpr int TW = 16 * TQ;   // width of the Hermite-sum table
        static constexpr int YS = 17;        // row stride of Y in LDS
    };

    // T: type of R, the E and the E' matrices (float: the small-bound quartets of a mixed build).
    // Every product and sum is FP64 in both, on the FP64 MFMA: T_ik is the difference of two totals
    // over the ket primitives, and in FP32 accumulators the share of a small primitive was rounded at
    // the size of the ones before it.  7 atoms (s to f), every quartet in the float form: 36.9 ms (FP32
    // accumulators 33.9, the double form 41.9); 19 atoms 1058 ms (1017, 1207).
    template <int LA, int LB, int LC, int LD, typename T>
    __global__ __launch_bounds__(64, 2) void gradWave(const GArgs A)
    {
        using P = GWPlan<LA, LB, LC, LD, T>;
        constexpr int L1 = P::L1, HL1 = P::HL1, HP = P::HP, HP1 = P::HP1, HQ = P::HQ, SP = P::SP, SQ = P::SQ;
        constexpr int SB = P::SB, SD = P::SD, NQ = P::NQ, KQ = P::KQ, TP = P::TP, TP1 = P::TP1, TQ = P::TQ, TS = P::TS;
        constexpr int KP = P::KP, KS = P::KS, PB = P::PB, TW = P::TW, YS = P::YS;
        constexpr bool F32 = sizeof(T) == 4;
        __shared__ T sR[PB * HL1];
        __shared__ T sInit[PB * (L1 + 1)];
        __shared__ T sPQ[4 * PB];
        __shared__ unsigned short sTab[16 * TP1 * TW]; // R index of (h', g); 0 past HP1, HQ
        __shared__ unsigned short sDn[16 * TP1][4];    // Y row of h' - e_x times YS; the zero row when there is none
        __shared__ double sY[(HP + 1) * YS];

        const int lane0 = threadIdx.x;
        const long long t0 = A.ntasks * blockIdx.x / gridDim.x;
        const long long t1 = A.ntasks * (blockIdx.x + 1) / gridDim.x;
        if (t0 >= t1)
            return;
        const DPairs &LP = A.lane, &UP = A.unif;
        const long long n = A.nbf;
        const double *D = A.D;
        double *const grad = A.grad + static_cast<long long>(blockIdx.x % A.ncopy) * A.stride;

        RecLane<L1> rec;
        rec.load(lane0);
        for (int e = lane0; e < 16 * TP1 * TW; e += 64)
        {
            const int h = e / TW, k = e - h * TW;
            int v = 0;
            if (h < HP1 && k < HQ)
            {
                const int a = hermTuv(h), b = hermTuv(k);
                v = hermIdx((a & 255) + (b & 255), ((a >> 8) & 255) + ((b >> 8) & 255), (a >> 16) + (b >> 16));
            }
            sTab[e] = static_cast<unsigned short>(v);
        }
        for (int e = lane0; e < 16 * TP1; e += 64)
        {
            const int a = e < HP1 ? hermTuv(e) : 0;
            const int t = a & 255, u = (a >> 8) & 255, v = a >> 16;
            sDn[e][0] = static_cast<unsigned short>((t > 0 ? hermIdx(t - 1, u, v) : HP) * YS);
            sDn[e][1] = static_cast<unsigned short>((u > 0 ? hermIdx(t, u - 1, v) : HP) * YS);
            sDn[e][2] = static_cast<unsigned short>((v > 0 ? hermIdx(t, u, v - 1) : HP) * YS);
        }
        if (lane0 < YS)
            sY[HP * YS + lane0] = 0.0;
        waveFence();

        int q = uniform(findKet(A.prefix, A.nket, t0));
        long long base = A.prefix[q], next = A.prefix[q + 1];
        for (long long t = t0; t < t1; t++)
        {
            while (t >= next)
            {
                q++;
                base = next;
                next = A.prefix[q + 1];
            }
            const int lane = opaqueLane(lane0);
            const int g4 = lane >> 4, j = lane & 15;
            // accumulator element (K step) kk of this lane holds row 4 kk + g4
            const int p = uniform(A.plo[q] + static_cast<int>(t - base));
            const int u = uniform(UP.order[q]), l = uniform(LP.order[p]);
            const int upoff = uniform(UP.poff[u]), ucnt = uniform(UP.pcnt[u]);
            const int lpoff = uniform(LP.poff[l]), lcnt = uniform(LP.pcnt[l]);
            const int a0 = uniform(LP.ao_a[l]), b0 = uniform(LP.ao_b[l]);
            const int c0 = uniform(UP.ao_a[u]), d0 = uniform(UP.ao_b[u]);
            double f = 1.0;
            if (LP.sh_a[l] == LP.sh_b[l])
                f *= 0.5;
            if (UP.sh_a[u] == UP.sh_b[u])
                f *= 0.5;
            if (A.same_class && p == q)
                f *= 0.5;

            double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0}, gC[3] = {0, 0, 0};
            const int nkMax = min(ucnt, PB), nbMax = min(lcnt, PB / nkMax);
#pragma unroll 1
            for (int i0 = 0; i0 < lcnt; i0 += nbMax)
#pragma unroll 1
                for (int k0 = 0; k0 < ucnt; k0 += nkMax)
                {
                    const int nb = min(nbMax, lcnt - i0), nk = min(nkMax, ucnt - k0);
                    {
                        const int bi = lane / nk, ki = lane - bi * nk;
                        waveFence();
                        hermiteBatch<L1, T>(sR, sInit, sPQ, rec, nb * nk, lane, LP.pp + lpoff + i0 + bi,
                                            UP.pp + upoff + k0 + ki, A.boys);
                    }
#pragma unroll 1
                    for (int pass = 0; pass < NQ; pass++)
                    {
                        const int col = 16 * pass + j;
                        const bool inC = col < SQ;
                        const unsigned ekOff = g4 * SQ + col, e1kOff = g4 * SQ + col;
                        const int yOff = g4 * YS + j;
                        // density weights: this lane's B-operand elements
                        double wB[KS];
                        {
                            const int ga = inC ? col / SD : 0, de = inC ? col % SD : 0;
                            const long long ic = c0 + ga, id = d0 + de;
                            const double dcd = 4.0 * D[ic * n + id];
#pragma unroll
                            for (int kk = 0; kk < KS; kk++)
                            {
                                const int ab = 4 * kk + g4;
                                const bool in = inC && ab < SP;
                                const int al = in ? ab / SB : 0, be = in ? ab % SB : 0;
                                const long long ia = a0 + al, ib = b0 + be;
                                const double w = f * (D[ia * n + ib] * dcd - D[ia * n + ic] * D[ib * n + id] -
                                                      D[ia * n + id] * D[ib * n + ic]);
                                wB[kk] = in ? w : 0.0;
                            }
                        }
#pragma unroll 1
                        for (int i = 0; i < nb; i++)
                        {
                            const int ip = lpoff + i0 + i;
                            const T *eb, *e1b;
                            if constexpr (F32)
                            {
                                eb = LP.eb32 + static_cast<size_t>(ip) * HP * SP;
                                e1b = LP.e1b32 + static_cast<size_t>(ip) * 3 * HP * SP;
                            }
                            else
                            {
                                eb = LP.eb + static_cast<size_t>(ip) * HP * SP;
                                e1b = LP.e1b + static_cast<size_t>(ip) * 3 * HP * SP;
                            }
                            const unsigned ebOff = j * SP + g4, e1bOff = g4 * SP + j;
                            v4d y[TP];
#pragma unroll
                            for (int tp = 0; tp < TP; tp++)
                                y[tp] = v4d{0, 0, 0, 0};
#pragma unroll
                            for (int kk = 0; kk < KS; kk++)
                            {
                                const int ab0 = 4 * kk;
#pragma unroll
                                for (int tp = 0; tp < TP; tp++)
                                {
                                    const bool in = 16 * tp + j < HP && ab0 + g4 < SP;
                                    const double a = in ? (eb + 16 * tp * SP + ab0)[ebOff] : T(0);
                                    y[tp] = mfma16(a, wB[kk], y[tp]);
                                }
                            }
                            waveFence();
#pragma unroll
                            for (int tp = 0; tp < TP; tp++)
#pragma unroll
                                for (int r = 0; r < 4; r++)
                                {
                                    const int row = 4 * (4 * tp + r);
                                    if (row + g4 < HP)
                                        sY[row * YS + yOff] = y[tp][r];
                                }
                            waveFence();

                            v4d s[TP1];
#pragma unroll
                            for (int tp = 0; tp < TP1; tp++)
                                s[tp] = v4d{0, 0, 0, 0};
                            double dsum[3] = {0, 0, 0};   // sum over the k so far of T_ik (this lane's part)
#pragma unroll 1
                            for (int k = 0; k < nk; k++)
                            {
                                const size_t kp = static_cast<size_t>(upoff + k0 + k);
                                const T *R = sR + (i * nk + k) * HL1;
                                // opaque again: nothing in this loop writes LDS, so its table and Y reads
                                // would all move in front of it
                                const int jk = opaqueLane(j), rk = opaqueLane(g4);
                                const int tabS = jk * TW + g4, tabQ = rk * TW + jk;
                                const T *ek, *e1k;
                                if constexpr (F32)
                                {
                                    ek = UP.ek32 + kp * HQ * SQ;
                                    e1k = UP.e1k32 + kp * 3 * HQ * SQ;
                                }
                                else
                                {
                                    ek = UP.ek + kp * HQ * SQ;
                                    e1k = UP.e1k + kp * 3 * HQ * SQ;
                                }
#pragma unroll
                                for (int kt = 0; kt < KQ; kt++)
                                {
                                    const bool in = 4 * kt + g4 < HQ && inC;
                                    const double b = in ? (ek + 4 * kt * SQ)[ekOff] : T(0);
#pragma unroll
                                    for (int tp = 0; tp < TP1; tp++)
                                        s[tp] = mfma16(double(R[sTab[tabS + 16 * tp * TW + 4 * kt]]), b, s[tp]);
                                }
                                // keep the phases apart: left alone the scheduler fetches all their operands
                                // first, and the registers for that cost more than the latency
                                __builtin_amdgcn_sched_barrier(0);
                                v4d qa[TQ];
#pragma unroll
                                for (int tq = 0; tq < TQ; tq++)
                                    qa[tq] = v4d{0, 0, 0, 0};
#pragma unroll
                                for (int kt = 0; kt < KP; kt++)
                                {
#pragma unroll
                                    for (int tq = 0; tq < TQ; tq++)
                                        qa[tq] = mfma16(double(R[sTab[tabQ + 4 * kt * TW + 16 * tq]]), y[kt >> 2][kt & 3], qa[tq]);
                                }
                                // V
#pragma unroll
                                for (int tq = 0; tq < TQ; tq++)
#pragma unroll
                                    for (int r = 0; r < 4; r++)
                                    {
                                        const int gg = 4 * (4 * tq + r);
                                        const bool in = gg + g4 < HQ && inC;
                                        const double qv = qa[tq][r];
#pragma unroll
                                        for (int x = 0; x < 3; x++)
                                        {
                                            const T e = in ? (e1k + (x * HQ + gg) * SQ)[e1kOff] : T(0);
                                            gC[x] = fma(qv, static_cast<double>(e), gC[x]);
                                        }
                                    }
                                // T: S against Y one row down per direction
                                double d[3] = {0, 0, 0};
#pragma unroll
                                for (int tp = 0; tp < TP1; tp++)
                                {
                                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                                    for (int r = 0; r < 4; r++)
                                    {
                                        const unsigned short *dn = sDn[4 * (4 * tp + r) + rk];
                                        const double sv = s[tp][r];
#pragma unroll
                                        for (int x = 0; x < 3; x++)
                                            d[x] = fma(sv, sY[dn[x] + jk], d[x]);
                                    }
                                }
                                const double rc = UP.ra[kp];   // c / q
#pragma unroll
                                for (int x = 0; x < 3; x++)
                                {
                                    gC[x] = fma(-rc, d[x] - dsum[x], gC[x]);
                                    dsum[x] = d[x];
                                }
                            }
                            const double ra = LP.ra[ip];   // a / p
#pragma unroll
                            for (int x = 0; x < 3; x++)
                            {
                                gA[x] = fma(ra, dsum[x], gA[x]);
                                gB[x] = fma(1.0 - ra, dsum[x], gB[x]);
                                // U
                                __builtin_amdgcn_sched_barrier(0);
                                double ux = 0.0;
#pragma unroll
                                for (int ts = 0; ts < TS; ts++)
                                {
                                    v4d gx = v4d{0, 0, 0, 0};
                                    const int ab = 16 * ts + j;
#pragma unroll
                                    for (int kt = 0; kt < KP; kt++)
                                    {
                                        const int h = 4 * kt;
                                        const bool in = h + g4 < HP && ab < SP;
                                        const double a = in ? (e1b + (x * HP + h) * SP + 16 * ts)[e1bOff] : T(0);
                                        gx = mfma16(a, s[kt >> 2][kt & 3], gx);
                                    }
#pragma unroll
                                    for (int r = 0; r < 4; r++)
                                        if (4 * ts + r < KS)
                                            ux = fma(gx[r], wB[4 * ts + r], ux);
                                }
                                gA[x] += ux;
                                gB[x] -= ux;
                            }
                        }
                    }
                }
#pragma unroll
            for (int x = 0; x < 3; x++)
            {
                gA[x] = waveSum(gA[x]);
                gB[x] = waveSum(gB[x]);
                gC[x] = waveSum(gC[x]);
            }
            // lanes 0..11: (centre, direction)
            if (lane < 12)
            {
                const int cen = lane / 3, x = lane - 3 * cen;
                double v = 0.0;
#pragma unroll
                for (int y = 0; y < 3; y++)
                    if (x == y)
                        v = cen == 0 ? gA[y] : cen == 1 ? gB[y] : cen == 2 ? gC[y] : -(gA[y] + gB[y] + gC[y]);
                const int at = cen == 0 ? LP.atom_a[l] : cen == 1 ? LP.atom_b[l] : cen == 2 ? UP.atom_a[u] : UP.atom_b[u];
                unsafeAtomicAdd(&grad[3 * at + x], v);
            }
        }
    }

    template <int LA, int LB, int LC, int LD, typename T>
    void launchGradWave(const GArgs &A, hipStream_t s)
    {
        if (A.ntasks <= 0)
            return;
        const int grid = static_cast<int>(A.ntasks < 16384 ? A.ntasks : 16384);
        hipLaunchKernelGGL((gradWave<LA, LB, LC, LD, T>), dim3(grid), dim3(64), 0, s, A);
    }

    template <int LA, int LB, int LC, int LD>
    void registerGradWave()
    {
        GradSlot &s = gradSlot(LA, LB, LC, LD);
        s.fn = &launchGradWave<LA, LB, LC, LD, double>;
        s.fn32 = &launchGradWave<LA, LB, LC, LD, float>;
        s.width = 1;
    }
}
