// One-wave-per-quartet form of the quartet kernels for gfx950 (variants VAR_MFMA / VAR_MFMA32):
// both transforms on MFMA (v_mfma_f64_16x16x4f64; FP32 form v_mfma_f32_16x16x4f32).
//
// The bra primitive pairs are stacked along M, (prim, tuv) rows, so one GEMM per ket primitive
// covers the batch's bra primitives: X[(i, tuv), kl] += R[(i, tuv), t'u'v'] Ek[t'u'v', kl]; the bra
// transform contracts over the stacked rows, I^T = X^T Eb_stack, reading X^T straight out of the
// accumulator registers: accumulator element c of a 16-row tile holds rows 4c..4c+3 across the
// lane groups, which is exactly the A-operand layout of K-chunk c.
//
// R is built for a batch of primitive quartets at a time (hermite_lds.hpp): as many bra
// primitives with all their ket primitives as fit 9 KiB of LDS, so that the latency of the Boys
// function and of the recursion levels is paid once per batch and several waves stay resident on
// each SIMD.
#pragma once

#include "hermite_lds.hpp"
#include "quartet.hpp"

namespace lbx
{
    template <int N>
    using ic = std::integral_constant<int, N>;

    template <int LA, int LB, int LC, int LD, typename T>
    struct WavePlan
    {
        using C = Cls<LA, LB, LC, LD>;
        static constexpr int L = C::L, HL = C::HL, HP = C::HP, HQ = C::HQ, SP = C::SP, SQ = C::SQ;
        static constexpr int NQ = ceilDiv(SQ, 16), NP = ceilDiv(SP, 16), KQ = ceilDiv(HQ, 4);
        // primitive quartets per batch
        static constexpr int PB0 = 9216 / (HL * static_cast<int>(sizeof(T)));
        static constexpr int PB = PB0 < 1 ? 1 : (PB0 > 64 ? 64 : PB0);
        // row tiles per chunk: accumulators (acc1 + acc2) within ~48 doubles per lane, at least
        // two tiles and at most the rows of four primitive pairs
        static constexpr int mtBudget = (48 - 4 * NQ * NP) / (4 * NQ);
        static constexpr int mtRows = ceilDiv(4 * HP, 16);
        static constexpr int MT0 = mtBudget < 2 ? 2 : (mtBudget > 6 ? 6 : mtBudget);
        static constexpr int MT = MT0 < mtRows ? MT0 : mtRows;
        static constexpr int RC = 16 * MT;   // rows per chunk
        // waves per SIMD asked of the register allocator (accumulators and ~80 registers)
        static constexpr int kRegs = (4 * NQ * NP + 4 * MT * NQ) * 2 + 80;
        static constexpr int WPE = kRegs <= 128 ? 4 : (kRegs <= 168 ? 3 : (kRegs <= 256 ? 2 : 1));
        // R of the batch and I of the epilogue share one buffer
        static constexpr int bytesR = PB * HL * static_cast<int>(sizeof(T)), bytesI = SP * SQ * 8;
        // density blocks of the epilogue: ab, cd, bd, ad, bc, ac
        static constexpr int oD1 = SP, oD2 = oD1 + SQ, oD3 = oD2 + C::SB * C::SD, oD4 = oD3 + C::SA * C::SD,
                             oD5 = oD4 + C::SB * C::SC, nD = oD5 + C::SA * C::SC;
        static constexpr int bufDoubles = ((bytesR > bytesI ? bytesR : bytesI) + 7) / 8;
        static constexpr int ldsBytes = 8 * (bufDoubles + nD) + static_cast<int>(sizeof(T)) * PB * (L + 5) + 8 * HP * KQ;
        // Class pairs with a main g shell (J/K only): those whose Hermite-sum table and block leave
        // at least two workgroups per CU and whose accumulators fit the registers, i.e. all but
        // (gg|gg) and (gg|gf)
        static constexpr bool kFitsG = ldsBytes <= 65536 && NQ * NP <= 18;
        // elements of the epilogue's loops per lane: shell-pair blocks have up to 81
        static constexpr int each(int n) { return ceilDiv(n, 64); }
    };

    // T = double, or float (the small-bound quartets of mixed-precision J/K: R, the E matrices
    // and both transforms in FP32 on the FP32 MFMA; Boys values and the epilogue in FP64).
    //
    // Addresses are a uniform base plus one lane offset per operand, and the lane number is made
    // opaque once per quartet (opaqueLane): otherwise the compiler keeps every unrolled address in
    // registers across quartets, which halves the waves per SIMD.
    template <int LA, int LB, int LC, int LD, int MODE, typename T = double>
    __global__ __launch_bounds__(64, (WavePlan<LA, LB, LC, LD, T>::WPE)) void quartetM(const KArgs A)
    {
        using P = WavePlan<LA, LB, LC, LD, T>;
        using C = typename P::C;
        constexpr int L = P::L, HP = P::HP, HQ = P::HQ, SP = P::SP, SQ = P::SQ, HL = P::HL;
        constexpr int NQ = P::NQ, NP = P::NP, KQ = P::KQ, MT = P::MT, RC = P::RC, PB = P::PB;
        constexpr int SA = C::SA, SB = C::SB, SC = C::SC, SD = C::SD;
        constexpr bool F32 = sizeof(T) == 4;
        using Acc = std::conditional_t<F32, v4f, v4d>;
        static_assert(!F32 || MODE == MODE_JK, "FP32 MFMA form: J/K only");
        __shared__ double sBuf[P::bufDoubles];
        __shared__ T sInit[PB * (L + 1)];
        __shared__ T sPQ[4 * PB];
        __shared__ unsigned short sTab[HP * 4 * KQ];
        __shared__ double sD[MODE == MODE_JK ? P::nD : 1];
        T *const sR = reinterpret_cast<T *>(sBuf);
        double *const sI = sBuf;

        const int lane0 = threadIdx.x;

        // contiguous task range per workgroup
        const long long t0 = A.ntasks * blockIdx.x / gridDim.x;
        const long long t1 = A.ntasks * (blockIdx.x + 1) / gridDim.x;
        if (t0 >= t1)
            return;
        RecLane<L> rec;
        rec.load(lane0);
        // Hermite-sum table: row tuv, column t'u'v' -> index of the summed Hermite function
        for (int e = lane0; e < HP * 4 * KQ; e += 64)
        {
            const int h = e / (4 * KQ), k = e % (4 * KQ);
            int v = 0;
            if (k < HQ)
            {
                const int a = hermTuv(h), b = hermTuv(k);
                v = hermIdx((a & 255) + (b & 255), ((a >> 8) & 255) + ((b >> 8) & 255),
                            (a >> 16) + (b >> 16));
            }
            sTab[e] = static_cast<unsigned short>(v);
        }
        waveFence();

        int mol = -1;   // MODE_SUM: the molecule of the sums
        double sums[2] = {0.0, 0.0};
        int q = 0;
        long long base = 0, next = 0;
        if constexpr (MODE != MODE_BLOCK)
        {
            q = uniform(findKet(A.prefix, A.nket, t0));
            base = A.prefix[q];
            next = A.prefix[q + 1];
        }
        for (long long t = t0; t < t1; t++)
        {
            const int lane = opaqueLane(lane0);
            const int g = lane >> 4, j = lane & 15;
            int p = 0, ab, cd;
            if constexpr (MODE == MODE_BLOCK)
            {
                ab = uniform(A.plo[4 * t]);
                cd = uniform(A.plo[4 * t + 1]);
            }
            else
            {
                while (t >= next)
                {
                    q++;
                    base = next;
                    next = A.prefix[q + 1];
                }
                p = uniform(A.plo[q] + static_cast<int>(t - base));
                // task tables run over the ket pairs of one bra pair when bra_major is set (the
                // larger E matrix is then shared by consecutive tasks and stays in cache)
                cd = uniform(A.ket.order[A.bra_major ? p : q]);
                ab = uniform(A.bra.order[A.bra_major ? q : p]);
            }
            const int kpoff = uniform(A.ket.poff[cd]), kcnt = uniform(A.ket.pcnt[cd]);
            const int bpoff = uniform(A.bra.poff[ab]), bcnt = uniform(A.bra.pcnt[ab]);
            const int a0 = uniform(A.bra.ao_a[ab]), b0 = uniform(A.bra.ao_b[ab]);
            const int c0 = uniform(A.ket.ao_a[cd]), d0 = uniform(A.ket.ao_b[cd]);
            // the epilogue's density blocks, fetched ahead: 0 ab, 1 cd, 2 bd, 3 ad, 4 bc, 5 ac
            double dv[6][2] = {};
            if constexpr (MODE == MODE_JK)
            {
                const long long n = A.nbf;
                const double *D = A.D;
                auto fetch = [&](double (&v)[2], auto size, auto width, int r0, int c0_) {
#pragma unroll
                    for (int r = 0; r < P::each(size); r++)
                        if (lane + 64 * r < size)
                            v[r] = D[(r0 + (lane + 64 * r) / width) * n + c0_ + (lane + 64 * r) % width];
                };
                fetch(dv[0], ic<SP>{}, ic<SB>{}, a0, b0);
                fetch(dv[1], ic<SQ>{}, ic<SD>{}, c0, d0);
                fetch(dv[2], ic<SB * SD>{}, ic<SD>{}, b0, d0);
                fetch(dv[3], ic<SA * SD>{}, ic<SD>{}, a0, d0);
                fetch(dv[4], ic<SB * SC>{}, ic<SC>{}, b0, c0);
                fetch(dv[5], ic<SA * SC>{}, ic<SC>{}, a0, c0);
            }

            Acc acc2[NQ][NP];
#pragma unroll
            for (int a = 0; a < NQ; a++)
#pragma unroll
                for (int b = 0; b < NP; b++)
                    acc2[a][b] = Acc{0, 0, 0, 0};

            const T *ekBase, *ebBase;
            if constexpr (F32)
            {
                ekBase = A.ket.ek32 + static_cast<size_t>(kpoff) * HQ * SQ;
                ebBase = A.bra.eb32 + static_cast<size_t>(bpoff) * HP * SP;
            }
            else
            {
                ekBase = A.ket.ek + static_cast<size_t>(kpoff) * HQ * SQ;
                ebBase = A.bra.eb + static_cast<size_t>(bpoff) * HP * SP;
            }
            // batches: nb bra primitives with their ket primitives, or one bra primitive with PB
            // ket primitives at a time
            const int nkMax = min(kcnt, PB);
            const int nbMax = min(bcnt, PB / nkMax);
            for (int i0 = 0; i0 < bcnt; i0 += nbMax)
            {
                const int nb = min(nbMax, bcnt - i0), nrows = nb * HP;
                for (int rowbase = 0; rowbase < nrows; rowbase += RC)
                {
                    Acc acc1[MT][NQ];
#pragma unroll
                    for (int a = 0; a < MT; a++)
#pragma unroll
                        for (int b = 0; b < NQ; b++)
                            acc1[a][b] = Acc{0, 0, 0, 0};
                    // this lane's row of each tile: its Hermite-table row and bra primitive.  Rows
                    // past the batch repeat row 0: their X meets zeros in the bra transform.
                    int rowH[MT], rowP[MT];
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                    {
                        const int gr = rowbase + 16 * mt + j < nrows ? rowbase + 16 * mt + j : 0;
                        const int pr = gr / HP;
                        rowH[mt] = (gr - pr * HP) * (4 * KQ) + g;
                        rowP[mt] = pr;
                    }
                    for (int k0 = 0; k0 < kcnt; k0 += nkMax)
                    {
                        const int nk = min(nkMax, kcnt - k0);
                        if (rowbase == 0 || nkMax < kcnt)
                        {
                            const int bi = lane / nk, ki = lane - bi * nk;
                            waveFence();
                            hermiteBatch<L, T>(sR, sInit, sPQ, rec, nb * nk, lane, A.bra.pp + bpoff + i0 + bi,
                                               A.ket.pp + kpoff + k0 + ki, A.boys);
                        }
#pragma unroll 1
                        for (int k = 0; k < nk; k++)
                        {
                            // ket transform: acc1[mt][nt] += R[rows, t'u'v'] Ek[t'u'v', cols]
                            const T *ek = ekBase + static_cast<size_t>(k0 + k) * HQ * SQ;
                            const unsigned eOff = g * SQ + j;
                            int rOff[MT];
#pragma unroll
                            for (int mt = 0; mt < MT; mt++)
                                rOff[mt] = (rowP[mt] * nk + k) * HL;
#pragma unroll
                            for (int kt = 0; kt < KQ; kt++)
                            {
                                T b1[NQ];
#pragma unroll
                                for (int nt = 0; nt < NQ; nt++)
                                {
                                    const bool in = (4 * kt + 4 <= HQ || 4 * kt + g < HQ) && (16 * nt + 16 <= SQ || 16 * nt + j < SQ);
                                    b1[nt] = in ? (ek + 4 * kt * SQ + 16 * nt)[eOff] : T(0);
                                }
#pragma unroll
                                for (int mt = 0; mt < MT; mt++)
                                {
                                    if (rowbase + 16 * mt >= nrows)
                                        continue;
                                    const T a = sR[rOff[mt] + sTab[rowH[mt] + 4 * kt]];
#pragma unroll
                                    for (int nt = 0; nt < NQ; nt++)
                                        acc1[mt][nt] = mfma16(a, b1[nt], acc1[mt][nt]);
                                }
                            }
                        }
                    }
                    // bra transform: I^T[kl, mn] += X^T[kl, rows] Eb[rows, mn].  K-chunk c of X^T =
                    // accumulator element c of every lane: rows 16 mt + 4 c + (0..3) in FP64
                    // (element c holds row 4 c + g), rows 16 mt + c + 4 (0..3) in FP32 (row 4 g + c)
                    const T *eb0 = ebBase + (static_cast<size_t>(i0) * HP + rowbase) * SP;
                    const unsigned bOff = (F32 ? 4 * g : g) * SP + j;
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                    {
                        if (rowbase + 16 * mt >= nrows)
                            continue;
#pragma unroll
                        for (int c = 0; c < 4; c++)
                        {
                            const int r0 = 16 * mt + (F32 ? c : 4 * c);
                            const bool rv = rowbase + r0 + (F32 ? 4 * g : g) < nrows;
#pragma unroll
                            for (int np = 0; np < NP; np++)
                            {
                                const bool in = rv && (16 * np + 16 <= SP || 16 * np + j < SP);
                                const T b2 = in ? (eb0 + r0 * SP + 16 * np)[bOff] : T(0);
#pragma unroll
                                for (int nq = 0; nq < NQ; nq++)
                                    acc2[nq][np] = mfma16(acc1[mt][nq][c], b2, acc2[nq][np]);
                            }
                        }
                    }
                }
            }
            waveFence();
            // accumulator element r of lane (g, j) holds D[4 r + g][j] (FP64) or D[4 g + r][j]
            // (FP32); here D = I^T[16 nq + row][16 np + j]
#pragma unroll
            for (int nq = 0; nq < NQ; nq++)
#pragma unroll
                for (int np = 0; np < NP; np++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                    {
                        const int kl = 16 * nq + (F32 ? 4 * g + r : 4 * r + g), mn = 16 * np + j;
                        if (kl < SQ && mn < SP)
                            sI[mn * SQ + kl] = double(acc2[nq][np][r]);
                    }
            if constexpr (MODE == MODE_JK)
            {
                auto store = [&](const double (&v)[2], auto size, int at) {
#pragma unroll
                    for (int r = 0; r < P::each(size); r++)
                        if (lane + 64 * r < size)
                            sD[at + lane + 64 * r] = v[r];
                };
                store(dv[0], ic<SP>{}, 0);
                store(dv[1], ic<SQ>{}, P::oD1);
                store(dv[2], ic<SB * SD>{}, P::oD2);
                store(dv[3], ic<SA * SD>{}, P::oD3);
                store(dv[4], ic<SB * SC>{}, P::oD4);
                store(dv[5], ic<SA * SC>{}, P::oD5);
            }
            waveFence();

            if constexpr (MODE == MODE_JK)
            {
                double f = 1.0;
                if (A.bra.sh_a[ab] == A.bra.sh_b[ab])
                    f *= 0.5;
                if (A.ket.sh_a[cd] == A.ket.sh_b[cd])
                    f *= 0.5;
                if (A.same_class && p == q)
                    f *= 0.5;
                const long long n = A.nbf;
                for (int e = lane; e < SP; e += 64)
                {
                    double s = 0.0;
#pragma unroll
                    for (int kl = 0; kl < SQ; kl++)
                        s = fma(sI[e * SQ + kl], sD[P::oD1 + kl], s);
                    unsafeAtomicAdd(&A.J[(a0 + e / SB) * n + b0 + e % SB], 2.0 * f * s);
                }
                for (int e = lane; e < SQ; e += 64)
                {
                    double s = 0.0;
#pragma unroll
                    for (int mn = 0; mn < SP; mn++)
                        s = fma(sI[mn * SQ + e], sD[mn], s);
                    unsafeAtomicAdd(&A.J[(c0 + e / SD) * n + d0 + e % SD], 2.0 * f * s);
                }
                // The K blocks go to whichever triangle has the longer block rows: adjacent lanes
                // then add to adjacent addresses, and one 64-byte line takes one request (FP64
                // atomics run at 23 G lines/s whatever the line holds).
                // K_ac[mu,ka] += f sum_{nu,la} I D_bd[nu,la]
                for (int e = lane; e < SA * SC; e += 64)
                {
                    const int mu = e % SA, ka = e / SA;
                    double s = 0.0;
#pragma unroll
                    for (int nu = 0; nu < SB; nu++)
#pragma unroll
                        for (int la = 0; la < SD; la++)
                            s = fma(sI[(mu * SB + nu) * SQ + ka * SD + la], sD[P::oD2 + nu * SD + la], s);
                    unsafeAtomicAdd(&A.K[(c0 + ka) * n + a0 + mu], f * s);
                }
                // K_bc[nu,ka] += f sum_{mu,la} I D_ad[mu,la]
                for (int e = lane; e < SB * SC; e += 64)
                {
                    const int nu = SB >= SC ? e % SB : e / SC, ka = SB >= SC ? e / SB : e % SC;
                    double s = 0.0;
#pragma unroll
                    for (int mu = 0; mu < SA; mu++)
#pragma unroll
                        for (int la = 0; la < SD; la++)
                            s = fma(sI[(mu * SB + nu) * SQ + ka * SD + la], sD[P::oD3 + mu * SD + la], s);
                    unsafeAtomicAdd(&A.K[SB >= SC ? (c0 + ka) * n + b0 + nu : (b0 + nu) * n + c0 + ka], f * s);
                }
                // K_ad[mu,la] += f sum_{nu,ka} I D_bc[nu,ka]
                for (int e = lane; e < SA * SD; e += 64)
                {
                    const int mu = e % SA, la = e / SA;
                    double s = 0.0;
#pragma unroll
                    for (int nu = 0; nu < SB; nu++)
#pragma unroll
                        for (int ka = 0; ka < SC; ka++)
                            s = fma(sI[(mu * SB + nu) * SQ + ka * SD + la], sD[P::oD4 + nu * SC + ka], s);
                    unsafeAtomicAdd(&A.K[(d0 + la) * n + a0 + mu], f * s);
                }
                // K_bd[nu,la] += f sum_{mu,ka} I D_ac[mu,ka]
                for (int e = lane; e < SB * SD; e += 64)
                {
                    const int nu = SB >= SD ? e % SB : e / SD, la = SB >= SD ? e / SB : e % SD;
                    double s = 0.0;
#pragma unroll
                    for (int mu = 0; mu < SA; mu++)
#pragma unroll
                        for (int ka = 0; ka < SC; ka++)
                            s = fma(sI[(mu * SB + nu) * SQ + ka * SD + la], sD[P::oD5 + mu * SC + ka], s);
                    unsafeAtomicAdd(&A.K[SB >= SD ? (d0 + la) * n + b0 + nu : (b0 + nu) * n + d0 + la], f * s);
                }
            }
            else if constexpr (MODE == MODE_DENSE)
            {
                for (int e = lane; e < SP * SQ; e += 64)
                    denseStore<C>(A, sI[e], e / SQ, e % SQ, a0, b0, c0, d0);
            }
            else if constexpr (MODE == MODE_BLOCK)
            {
                const int flags = uniform(A.plo[4 * t + 2]);
                double *o = A.out + static_cast<long long>(uniform(A.plo[4 * t + 3])) * (SP * SQ);
                for (int e = lane; e < SP * SQ; e += 64)
                {
                    const int mn = e / SQ, kl = e - mn * SQ;
                    const int ib = (flags & 1) ? (mn % SB) * SA + mn / SB : mn;
                    const int ik = (flags & 2) ? (kl % SD) * SC + kl / SD : kl;
                    o[(flags & 4) ? ik * SP + ib : ib * SQ + ik] = sI[e];
                }
            }
            else if constexpr (MODE == MODE_SUM)
            {
                double sa = 0.0, ss = 0.0;
                for (int e = lane; e < SP * SQ; e += 64)
                {
                    sa += fabs(sI[e]);
                    ss += sI[e];
                }
                const bool one = A.kind == 3 ? A.bra.sh_a[ab] == A.bra.sh_b[ab] : (A.same_class && p == q);
                const double w = one ? 1.0 : 2.0;
                const int m = uniform(A.ket.mol[cd]);
                if (m != mol)
                {
                    if (mol >= 0)
                        flushSums(A, mol, lane, sums[0], sums[1]);
                    mol = m;
                    sums[0] = sums[1] = 0.0;
                }
                sums[0] = fma(w, sa, sums[0]);
                sums[1] = fma(w, ss, sums[1]);
            }
            else
            {
                if (lane == 0)
                {
                    double m = 0.0;
                    for (int mn = 0; mn < SP; mn++)
                        m = fmax(m, fabs(sI[mn * SQ + mn]));
                    A.qout[ab] = sqrt(m);
                }
                if (A.dout)
                    for (int mn = lane; mn < SP; mn += 64)
                    {
                        const int mu = mn / SB, nu = mn % SB;
                        const double v = sI[mn * SQ + mn];
                        if (A.kind == 2)
                            A.dout[a0 + mu] = v;
                        else
                        {
                            A.dout[(a0 + mu) * A.nbf + b0 + nu] = v;
                            A.dout[(b0 + nu) * A.nbf + a0 + mu] = v;
                        }
                    }
            }
            waveFence();
        }
        if constexpr (MODE == MODE_SUM)
            if (mol >= 0)
                flushSums(A, mol, lane0, sums[0], sums[1]);
    }

    template <int LA, int LB, int LC, int LD, int MODE, typename T = double>
    void launchMfma(const KArgs &A, hipStream_t s)
    {
        if (A.ntasks <= 0)
            return;
        const int grid = static_cast<int>(A.ntasks < 16384 ? A.ntasks : 16384);
        hipLaunchKernelGGL((quartetM<LA, LB, LC, LD, MODE, T>), dim3(grid), dim3(64), 0, s, A);
    }

    // The one-wave forms of a class pair: FP64 in every mode, FP32 for J/K (FORMS as in
    // registerQuartet).  For J/K they also stand in for the one-lane forms that would fit the
    // registers but are not built (Cls::laneBuilt; main shells to f only).
    template <int LA, int LB, int LC, int LD, int MODE, int FORMS = 3>
    void registerWave()
    {
        using C = Cls<LA, LB, LC, LD>;
        constexpr bool same = LA == LC && LB == LD;
        auto put = [](int variant, Launcher fn) {
            KernelSlot &s = kernelSlot(MODE, LA, LB, LC, LD, variant);
            s.fn = fn;
            s.width = 1;
            s.swap = false;
            s.kind = KIND_WAVE;
        };
        if constexpr (FORMS & 1)
        {
            put(VAR_MFMA, &launchMfma<LA, LB, LC, LD, MODE>);
            if constexpr (MODE == MODE_JK && LA <= 3 && C::NC0 > 0 && !C::kLane0)
                put(VAR_VALU_BRA, &launchMfma<LA, LB, LC, LD, MODE>);
            if constexpr (MODE == MODE_JK && LA <= 3 && C::NC1 > 0 && !C::kLane1 && !same)
                put(VAR_VALU_KET, &launchMfma<LA, LB, LC, LD, MODE>);
        }
        if constexpr ((FORMS & 2) && MODE == MODE_JK)
        {
            put(VAR_MFMA32, &launchMfma<LA, LB, LC, LD, MODE, float>);
            if constexpr (C::NC0f > 0 && !C::kLane0f)
                put(VAR_VALU_BRA32, &launchMfma<LA, LB, LC, LD, MODE, float>);
            if constexpr (C::NC1f > 0 && !C::kLane1f && !same)
                put(VAR_VALU_KET32, &launchMfma<LA, LB, LC, LD, MODE, float>);
        }
    }
}
