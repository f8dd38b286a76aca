// Nuclear gradient of the two-electron energy E = 1/2 tr(DJ) - 1/4 tr(DK), contracted on the
// fly (adjoint form): no derivative integral is stored.
//
// For a shell quartet (ab|cd) with weight W[ab][cd] = f (4 D_ab D_cd - D_ac D_bd - D_ad D_bc)
// (f the permutational weight of the unique quartet) the gradient is sum W d(ab|cd)/dX.  With
// the Hermite form (ab|cd) = sum_{ij} Eb_i[ab][h] Ek_j[cd][g] R_{h+g} (prim pairs i, j) and
// E a function of the relative coordinate A - B only (P = (aA + bB)/p moves the Hermite
// Gaussian, d/dP_x raises its x index by one):
//   dA = sum_ij [ (a/p) T_ij + U_ij ],   dB = sum_ij [ (b/p) T_ij - U_ij ],
//   dC = sum_ij [ V_ij - (c/q) T_ij ],   dD = -(dA + dB + dC)
// with, per Cartesian direction x,
//   T_ij = sum W Eb_i Ek_j R_{h+g+e_x},  U_ij = sum W Eb'_i,x Ek_j R_{h+g},
//   V_ij = sum W Eb_i Ek'_j,x R_{h+g}   (E' = dE/d(A-B)_x; the ket's (-1)^{t'+u'+v'} in Ek, Ek').
// This is the quantity of the reference's ERI4D1 kernel (eri_kernel_funs.cpp:582-748) contracted
// with the density weights.
//
// Two kernels: the slot form here for class pairs of low total angular momentum, the one-wave MFMA
// form (grad_wave.hpp) for the others.
//
// Slot form: one wave per task, a task is G lane-side pairs against one uniform-side pair; each
// pair (slot) has LPS = 64/G lanes that split its Hermite index h.  R of LPS primitive quartets per
// slot is made at a time, one lane per primitive quartet with the recursion in registers, and goes
// to LDS; then per primitive pair i of the lane side and column pass of cd
//   Y[h][cd] = sum_ab Eb_i[ab][h] W[ab][cd]
//   per ket primitive j:  T += sum_{h,g} (sum_cd Y Ek_j) R_{h+g+e_x},  V += sum_{h,g} R_{h+g}
//                         (sum_cd Y Ek'_j,x),   X[h][cd] += sum_g R_{h+g} Ek_j[cd][g]
//   U = sum_{ab,cd} W[ab][cd] sum_h Eb'_i,x[ab][h] X[h][cd].
#pragma once

#include "hermite_lds.hpp"
#include "dpairs.hpp"

namespace lbx
{
    struct GArgs
    {
        DPairs lane, unif;           // lane-side class (the "bra" of the formulas), uniform side
        const long long *prefix;     // per uniform-side position: first task
        const int *plo, *phi;        // lane-side sorted-position range per uniform position
        int nket;
        long long ntasks;
        int same_class;
        const double *boys;
        const double *D;
        long long nbf;
        // ncopy gradients of 3 natoms values, `stride` apart, which the caller adds up: a workgroup
        // adds to copy blockIdx % ncopy (the few lines of a small molecule's gradient would
        // serialise the atomics: about 60 M additions per second and line)
        double *grad;
        int ncopy;
        long long stride;
    };

    using GradLauncher = void (*)(const GArgs &, hipStream_t);
    struct GradSlot
    {
        GradLauncher fn = nullptr;     // FP64
        GradLauncher fn32 = nullptr;   // R, E, E' and the transforms in FP32, sums in FP64
        int width = 0;   // lane-side pairs per task
    };
    // (la lb) lane side, (lc ld) uniform side
    GradSlot &gradSlot(int la, int lb, int lc, int ld);

    constexpr LBX_HD int pow2Ceil(int x)
    {
        int p = 1;
        while (p < x)
            p *= 2;
        return p;
    }

    // Class pairs whose R of order L + 1 stays in a lane's registers and 64 of them in 32 KiB of
    // LDS take the slot form.
    constexpr int kGradSlotL1 = 5;
    constexpr LBX_HD bool gradUsesSlots(int la, int lb, int lc, int ld) { return la + lb + lc + ld + 1 <= kGradSlotL1; }

    // Work of a quartet of the one-wave form when (la lb) takes the rows, in quarters of an MFMA
    // (64 cycles): per primitive quartet the products S and Q, the sums T (about 7 MFMAs' time per
    // four row tiles of S) and V (3 per two of Q) and the loop; per row-side primitive Y, U and the
    // turn of the accumulators; per column tile the weights.  The depths are the synthetic shells' (4, 3,
    // 1, 1 primitives for s, p, d, f), not the basis at hand's: the choice is made when the kernels are
    // compiled.  It moves 7 atoms of those shells by 4%; other contractions were not measured.
    constexpr LBX_HD int gradWaveCost(int la, int lb, int lc, int ld)
    {
        const int depth[5] = {4, 3, 1, 1, 1};
        const int kb = depth[la] * depth[lb], kk = depth[lc] * depth[ld];
        const int hp = nHerm(la + lb), hp1 = nHerm(la + lb + 1), hq = nHerm(lc + ld);
        const int sp = nSph(la) * nSph(lb), sq = nSph(lc) * nSph(ld);
        const int tp1 = ceilDiv(hp1, 16), tq = ceilDiv(hq, 16);
        const int prim = 4 * (tp1 * ceilDiv(hq, 4) + tq * ceilDiv(hp, 4)) + 7 * tp1 + 6 * tq + 12;
        const int row = 4 * (ceilDiv(hp, 16) * ceilDiv(sp, 4) + 3 * ceilDiv(sp, 16) * ceilDiv(hp, 4)) + 32;
        return ceilDiv(sq, 16) * (kb * kk * prim + kb * row + 8 * ceilDiv(sp, 4));
    }

    // lane side ("bra") chosen for an unordered class pair: in the one-wave form (main shells to f)
    // the assignment with less work, else the larger Hermite dimension (more lanes in use); ties
    // to the larger class index
    constexpr LBX_HD bool gradLaneFirst(int la, int lb, int lc, int ld)
    {
        const bool tie = pairClassIdx(la, lb) >= pairClassIdx(lc, ld);
        if (!gradUsesSlots(la, lb, lc, ld) && la <= 3 && lc <= 3)
        {
            const int x = gradWaveCost(la, lb, lc, ld), y = gradWaveCost(lc, ld, la, lb);
            return x != y ? x < y : tie;
        }
        return nHerm(la + lb) > nHerm(lc + ld) || (nHerm(la + lb) == nHerm(lc + ld) && tie);
    }

    template <int LA, int LB, int LC, int LD>
    struct GCls
    {
        static constexpr int L = LA + LB + LC + LD, L1 = L + 1;
        static constexpr int HP = nHerm(LA + LB), HQ = nHerm(LC + LD), HL1 = nHerm(L1);
        static constexpr int SA = nSph(LA), SB = nSph(LB), SC = nSph(LC), SD = nSph(LD);
        static constexpr int SP = SA * SB, SQ = SC * SD;
        // lanes per slot: the Hermite rows (HR) times REP, REP groups of them taking the ket
        // primitives of a lane-side primitive in turn (few rows would leave the long primitive loops
        // of contracted s and p shells to one or four lanes)
        static constexpr int HR = HP >= 64 ? 64 : pow2Ceil(HP);
        static constexpr int REP = HP == 1 ? 4 : (HP == 4 ? 2 : 1);
        static constexpr int LPS = HR * REP;
        static constexpr int G = 64 / LPS;
        static constexpr int NH = ceilDiv(HP, HR);         // h values per lane
        static constexpr int NPASS = ceilDiv(SQ, 9);
        static constexpr int NC = ceilDiv(SQ, NPASS);      // cd columns per pass, at most 9
        static constexpr int RS = HL1 | 1;                 // LDS stride of one primitive quartet's R (odd)
    };

    template <bool UNIFORM, typename T>
    __device__ __forceinline__ auto uniformView(const T *p)
    {
        if constexpr (UNIFORM)
            return constView(p);
        else
            return p;
    }

    // sum over the LPS lanes of one slot (contiguous lane groups)
    template <int LPS>
    __device__ __forceinline__ double slotSum(double x)
    {
#pragma unroll
        for (int o = LPS / 2; o >= 1; o >>= 1)
            x += __shfl_xor(x, o, 64);
        return x;
    }

    __device__ __forceinline__ int waveMaxInt(int x)
    {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1)
            x = max(x, __shfl_xor(x, o, 64));
        return x;
    }

    // T: type of R, the E and E' matrices and the transforms (double, or float for the
    // small-bound quartets of the mixed-precision gradient); Boys values, density weights and the
    // gradient sums stay double.
    template <int LA, int LB, int LC, int LD, typename T>
    __global__ __launch_bounds__(64, 2) void gradKernel(const GArgs A)
    {
        using C = GCls<LA, LB, LC, LD>;
        constexpr int L1 = C::L1, HP = C::HP, HQ = C::HQ, HL1 = C::HL1, SP = C::SP, SQ = C::SQ, SB = C::SB, SD = C::SD,
                      G = C::G, LPS = C::LPS, HR = C::HR, REP = C::REP, NH = C::NH, NC = C::NC, RS = C::RS;
        constexpr bool F32 = sizeof(T) == 4;
        __shared__ T sR[64 * RS];
        __shared__ double sW[G * SP * SQ];
        __shared__ unsigned short sTab[HP * HQ][4];   // R index of h + g, and of h + g + e_x
        const int lane0 = threadIdx.x;
        const DPairs &LP = A.lane, &UP = A.unif;
        const long long n = A.nbf;
        const double *D = A.D;
        double *const grad = A.grad + static_cast<long long>(blockIdx.x % A.ncopy) * A.stride;

        const long long t0 = A.ntasks * blockIdx.x / gridDim.x;
        const long long t1 = A.ntasks * (blockIdx.x + 1) / gridDim.x;
        if (t0 >= t1)
            return;
        for (int e = lane0; e < HP * HQ; e += 64)
        {
            const int a = hermTuv(e / HQ), b = hermTuv(e % HQ);
            const int t = (a & 255) + (b & 255), u = ((a >> 8) & 255) + ((b >> 8) & 255), v = (a >> 16) + (b >> 16);
            sTab[e][0] = static_cast<unsigned short>(hermIdx(t, u, v));
            sTab[e][1] = static_cast<unsigned short>(hermIdx(t + 1, u, v));
            sTab[e][2] = static_cast<unsigned short>(hermIdx(t, u + 1, v));
            sTab[e][3] = static_cast<unsigned short>(hermIdx(t, u, v + 1));
        }
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
            const int slot = lane / LPS, jl = lane % LPS, jh = jl % HR, rep = jl / HR;
            const int local = static_cast<int>(t - base);
            const int plo = uniform(A.plo[q]), phi = uniform(A.phi[q]);
            const int p = plo + local * G + slot;
            const bool active = p < phi;
            const int u = uniform(UP.order[q]);
            const int l = LP.order[active ? p : plo];
            const int upoff = uniform(UP.poff[u]), ucnt = uniform(UP.pcnt[u]);
            const int lpoff = LP.poff[l], lcnt = active ? LP.pcnt[l] : 0;
            const int imax = uniform(waveMaxInt(lcnt));
            const int a0 = LP.ao_a[l], b0 = LP.ao_b[l];
            const int c0 = uniform(UP.ao_a[u]), d0 = uniform(UP.ao_b[u]);
            double f = active ? 1.0 : 0.0;
            if (LP.sh_a[l] == LP.sh_b[l])
                f *= 0.5;
            if (UP.sh_a[u] == UP.sh_b[u])
                f *= 0.5;
            if (A.same_class && p == q)
                f *= 0.5;

            // density weights of this slot's quartet
            double *const w0 = sW + slot * (SP * SQ);
            for (int e = jl; e < SP * SQ; e += LPS)
            {
                const int ab = e / SQ, cd = e - ab * SQ;
                const int al = ab / SB, be = ab - al * SB, ga = cd / SD, de = cd - ga * SD;
                const long long ia = a0 + al, ib = b0 + be, ic = c0 + ga, id = d0 + de;
                w0[e] = active ? f * (4.0 * D[ia * n + ib] * D[ic * n + id] - D[ia * n + ic] * D[ib * n + id] -
                                      D[ia * n + id] * D[ib * n + ic])
                               : 0.0;
            }
            waveFence();

            double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0}, gC[3] = {0, 0, 0};
            // primitive quartets e = i ucnt + k of every slot, LPS of them at a time
            const int emax = imax * ucnt;
#pragma unroll 1
            for (int e0 = 0; e0 < emax; e0 += LPS)
            {
                {
                    const int e = e0 + jl, i = e / ucnt, k = e - i * ucnt;
                    waveFence();
                    if (i < lcnt)
                    {
                        const double4 Pl = LP.pp[lpoff + i], Pu = UP.pp[upoff + k];
                        const double pq = Pl.x * Pu.x, ps = Pl.x + Pu.x, alpha = pq / ps;
                        const double X = Pl.y - Pu.y, Y = Pl.z - Pu.z, Z = Pl.w - Pu.w;
                        double F[L1 + 1];
                        boysF<L1>(alpha * (X * X + Y * Y + Z * Z), A.boys, F);
                        T R[HL1 + L1];
                        double sc = kTwoPi52 / (pq * sqrt(ps));
#pragma unroll
                        for (int m = 0; m <= L1; m++)
                        {
                            R[m] = T(F[m] * sc);
                            sc *= -2.0 * alpha;
                        }
                        hermiteR<L1, T>(R, T(X), T(Y), T(Z));
                        T *const out = sR + lane * RS;
                        out[0] = R[0];
#pragma unroll
                        for (int h = 1; h < HL1; h++)
                            out[h] = R[L1 + h];
                    }
                    waveFence();
                }
                const int e1 = min(e0 + LPS, emax);
#pragma unroll 1
                for (int pass = 0; pass < C::NPASS; pass++)
                {
                    const int cd0 = pass * NC;
                    int e = e0;
#pragma unroll 1
                    while (e < e1)
                    {
                        // the run of one lane-side primitive pair in this batch
                        const int i = e / ucnt, kBeg = e - i * ucnt, kEnd = min(ucnt, kBeg + e1 - e);
                        const bool valid = i < lcnt;
                        const int ip = lpoff + (valid ? i : 0);
                        // Y[h][c] = sum_ab Eb_i[h][ab] W[ab][cd0 + c]
                        T Y[NH][NC], X[NH][NC];
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
#pragma unroll
                        for (int r = 0; r < NH; r++)
#pragma unroll
                            for (int c = 0; c < NC; c++)
                            {
                                Y[r][c] = T(0);
                                X[r][c] = T(0);
                            }
#pragma unroll 3
                        for (int ab = 0; ab < SP; ab++)
                        {
                            T w[NC];
#pragma unroll
                            for (int c = 0; c < NC; c++)
                                w[c] = cd0 + c < SQ ? T(w0[ab * SQ + cd0 + c]) : T(0);
#pragma unroll
                            for (int r = 0; r < NH; r++)
                            {
                                const int h = jh + r * HR;
                                const T ev = h < HP ? eb[h * SP + ab] : T(0);
#pragma unroll
                                for (int c = 0; c < NC; c++)
                                    Y[r][c] = fma(ev, w[c], Y[r][c]);
                            }
                        }
                        double Ts[3] = {0, 0, 0};
#pragma unroll 1
                        for (int kr = kBeg; kr < kEnd; kr += REP)
                        {
                            const int k = min(kr + rep, kEnd - 1);   // past the end: not used
                            const bool use = valid && kr + rep < kEnd;
                            const T *R = sR + (slot * LPS + e - e0 + k - kBeg) * RS;
                            const size_t kk = static_cast<size_t>(upoff + k);
                            const T *ekb, *e1kb;
                            if constexpr (F32)
                            {
                                ekb = UP.ek32;
                                e1kb = UP.e1k32;
                            }
                            else
                            {
                                ekb = UP.ek;
                                e1kb = UP.e1k;
                            }
                            // wave-uniform (scalar loads) unless the groups are at different k
                            const auto ek = uniformView<REP == 1>(ekb + kk * HQ * SQ + cd0);
                            const auto e1 = uniformView<REP == 1>(e1kb + kk * 3 * HQ * SQ + cd0);
                            double tk[3] = {0, 0, 0};
                            if (use)
#pragma unroll
                                for (int g = 0; g < HQ; g++)
                                {
                                    T ekv[NC], e1v[3][NC];
#pragma unroll
                                    for (int c = 0; c < NC; c++)
                                    {
                                        const bool in = cd0 + c < SQ;
                                        ekv[c] = in ? ek[g * SQ + c] : T(0);
#pragma unroll
                                        for (int x = 0; x < 3; x++)
                                            e1v[x][c] = in ? e1[(x * HQ + g) * SQ + c] : T(0);
                                    }
#pragma unroll
                                    for (int r = 0; r < NH; r++)
                                    {
                                        const int h = jh + r * HR;
                                        if (h >= HP)
                                            continue;
                                        const unsigned short *tab = sTab[h * HQ + g];
                                        const T r0 = R[tab[0]], rx = R[tab[1]], ry = R[tab[2]], rz = R[tab[3]];
                                        T z = T(0), zx = T(0), zy = T(0), zz = T(0);
#pragma unroll
                                        for (int c = 0; c < NC; c++)
                                        {
                                            z = fma(Y[r][c], ekv[c], z);
                                            zx = fma(Y[r][c], e1v[0][c], zx);
                                            zy = fma(Y[r][c], e1v[1][c], zy);
                                            zz = fma(Y[r][c], e1v[2][c], zz);
                                            X[r][c] = fma(r0, ekv[c], X[r][c]);
                                        }
                                        tk[0] = fma(double(z), double(rx), tk[0]);
                                        tk[1] = fma(double(z), double(ry), tk[1]);
                                        tk[2] = fma(double(z), double(rz), tk[2]);
                                        gC[0] = fma(double(r0), double(zx), gC[0]);
                                        gC[1] = fma(double(r0), double(zy), gC[1]);
                                        gC[2] = fma(double(r0), double(zz), gC[2]);
                                    }
                                }
                            const double rc = uniformView<REP == 1>(UP.ra)[upoff + k];   // c / q
#pragma unroll
                            for (int x = 0; x < 3; x++)
                            {
                                Ts[x] += tk[x];
                                gC[x] = fma(-rc, tk[x], gC[x]);
                            }
                        }
                        if (valid)
                        {
                            const double ra = LP.ra[ip];   // a / p
#pragma unroll
                            for (int x = 0; x < 3; x++)
                            {
                                gA[x] = fma(ra, Ts[x], gA[x]);
                                gB[x] = fma(1.0 - ra, Ts[x], gB[x]);
                            }
                            // U_x = sum_ab sum_c W[ab][cd0 + c] sum_h Eb'_x[h][ab] X[h][c]
                            double ux[3] = {0, 0, 0};
#pragma unroll 3
                            for (int ab = 0; ab < SP; ab++)
                            {
                                T w[NC];
#pragma unroll
                                for (int c = 0; c < NC; c++)
                                    w[c] = cd0 + c < SQ ? T(w0[ab * SQ + cd0 + c]) : T(0);
#pragma unroll
                                for (int r = 0; r < NH; r++)
                                {
                                    const int h = jh + r * HR;
                                    if (h >= HP)
                                        continue;
                                    T s = T(0);
#pragma unroll
                                    for (int c = 0; c < NC; c++)
                                        s = fma(w[c], X[r][c], s);
#pragma unroll
                                    for (int x = 0; x < 3; x++)
                                        ux[x] = fma(double(e1b[(x * HP + h) * SP + ab]), double(s), ux[x]);
                                }
                            }
#pragma unroll
                            for (int x = 0; x < 3; x++)
                            {
                                gA[x] += ux[x];
                                gB[x] -= ux[x];
                            }
                        }
                        e += kEnd - kBeg;
                    }
                }
            }
#pragma unroll
            for (int x = 0; x < 3; x++)
            {
                gA[x] = slotSum<LPS>(gA[x]);
                gB[x] = slotSum<LPS>(gB[x]);
                gC[x] = slotSum<LPS>(gC[x]);
            }
            if (active && jl == 0)
            {
                const int at[4] = {LP.atom_a[l], LP.atom_b[l], UP.atom_a[u], UP.atom_b[u]};
#pragma unroll
                for (int x = 0; x < 3; x++)
                {
                    unsafeAtomicAdd(&grad[3 * at[0] + x], gA[x]);
                    unsafeAtomicAdd(&grad[3 * at[1] + x], gB[x]);
                    unsafeAtomicAdd(&grad[3 * at[2] + x], gC[x]);
                    unsafeAtomicAdd(&grad[3 * at[3] + x], -(gA[x] + gB[x] + gC[x]));
                }
            }
            waveFence();   // sW of the next task
        }
    }

    template <int LA, int LB, int LC, int LD, typename T>
    void launchGrad(const GArgs &A, hipStream_t s)
    {
        if (A.ntasks <= 0)
            return;
        const int grid = static_cast<int>(A.ntasks < 16384 ? A.ntasks : 16384);
        hipLaunchKernelGGL((gradKernel<LA, LB, LC, LD, T>), dim3(grid), dim3(64), 0, s, A);
    }

    template <int LA, int LB, int LC, int LD>
    void registerGrad()
    {
        GradSlot &s = gradSlot(LA, LB, LC, LD);
        s.fn = &launchGrad<LA, LB, LC, LD, double>;
        s.fn32 = &launchGrad<LA, LB, LC, LD, float>;
        s.width = GCls<LA, LB, LC, LD>::G;
    }
}
