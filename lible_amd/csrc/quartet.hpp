// SHARK shell-quartet kernels for gfx950.
//
// Per shell quartet (ab|cd) of class (LA LB | LC LD), following the reference's SHARK scheme
// (eri_kernel_funs.hpp:104-193, after doi:10.1002/jcc.26942 eqs. 25-26):
//   for each bra primitive pair i:  X_i = sum_k R_{ik} . Ek_k          (ket transform)
//   I = sum_i Eb_i^T X_i                                               (bra transform)
// with R_{ik}(tuv, t'u'v') = fac R_{t+t',u+u',v+v'} (Hermite integrals; the ket's sign
// (-1)^{t'+u'+v'} folded into Ek) and Eb, Ek the spherical Hermite-expansion matrices of the
// primitive pairs.
//
// quartetV: one lane per quartet, everything in registers.  A wave holds 64 pairs of one side (the
// "lane" side) against one pair of the other (the "uniform" side), so every uniform-side operand is
// a scalar load and the transforms are VALU FMAs with an SGPR operand.  Registers are bounded by
// splitting the uniform side's spherical components into column passes (Boys + R recomputed per
// pass); which side runs on the lanes is chosen per class pair (variant_cost.hpp).
//
// What bounds it: the loads of the lane side's E, one element per FMA of a column.  As stored, each
// is a line per lane (about 100 cycles against 4 for the FMA), and the compiler waits for it before
// it issues the next; interleaved over the lanes (512 contiguous bytes) and loaded a group ahead
// they cost J/K of 19 atoms (570 functions): (dp|ps) 5.1 -> 2.7 ms, (dp|ds) 5.4 -> 2.7, (fp|ps)
// 9.4 -> 8.4, FP32 (fd|ps) 11.6 -> 1.2, (dd|dp) 4.8 -> 1.6.  At low angular momentum the K atomics
// (16 updates per (ps|ps) quartet at 23 G lines/s): K rows in LDS take J/K of (H2O)10 def2-TZVP
// from (pp|ps) 2.4 -> 1.1 ms, (ps|ps) 2.3 -> 1.1, (ds|ps) 2.2 -> 0.95.  (ss|ss) is left at its Boys
// functions: 4.5e8 in 2.8 ms.
// The other forms: quartet_wave.hpp (one wave per quartet on MFMA), quartet_block.hpp.
// Epilogues: J/K contraction with atomics, dense tensor scatter, per-molecule sums, or (one-wave
// form) the (ab|ab) diagonal and listed blocks.
#pragma once

#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "dpairs.hpp"
#include "registry.hpp"

namespace lbx
{
    enum Mode
    {
        MODE_JK = 0,
        MODE_DENSE = 1,
        MODE_DIAG = 2,
        MODE_SUM = 3,   // per-molecule sums of |value| and value of the dense eri3 / eri2 tensors
        MODE_BLOCK = 4, // blocks of listed pair combinations (one-wave form only): plo = ntasks x
                        // (bra pair, ket pair, flags, slot), block at out + slot * its size; flags
                        // bit 0 / 1: the caller's bra / ket shells are the pair's in reverse,
                        // bit 2: the caller's first side is the ket
        N_MODES = 5
    };

    struct KArgs
    {
        DPairs bra, ket;
        const long long *prefix;   // per uniform-side position q: first task (nket + 1 entries)
        const int *plo, *phi;      // lane-side sorted-position range [plo, phi) for each q
        int nket;
        long long ntasks;
        int same_class;            // bra class == ket class: quartet p == q is its own image
        int bra_major;             // one-wave form: q indexes bra pairs, p ket pairs (classes differ)
        // quartetV lane-block-major order: lane block b = lane positions 64b .. 64b+63; group g =
        // blocks g G .. g G + G - 1 (G = 2^gshift).  Group g's tasks pair its uniform positions
        // q = bq0[g], bq0[g] + 1, ... with its G blocks in turn (bprefix[g+1] - bprefix[g] = G x
        // the count of those q).
        int block_major, nblk, gshift;
        const long long *bprefix;
        const int *bq0;
        // lane-block-major J/K: lane position -> Schwarz-order position (within Schwarz-factor
        // buckets by primitive count when kcols > 0, else by shell, so lanes sharing a shell are
        // adjacent), and per lane block the range [bqlo, bqhi) of Schwarz-order positions it holds;
        // null otherwise
        const int *lperm, *bqlo, *bqhi;
        const double *boys;
        // MODE_JK
        const double *D;
        double *J, *K;
        long long nbf;
        // MODE_DENSE: kind 4 eri4 (nbf^4), 3 eri3 (nbf, nbf, naux), 2 eri2 (naux, naux)
        // MODE_SUM: out = (nmol, 4) sums |eri3|, eri3, |eri2|, eri2 by the ket's molecule
        double *out;
        int kind;
        long long naux;
        // MODE_DIAG
        double *qout;   // sqrt(max |(ab|ab)|) per pair (pair order)
        double *dout;   // (mn|mn) matrix (pair classes) or vector (single classes), may be null
        // quartetV: the lane side's E matrices interleaved over the 64 lanes of a block, so that the
        // lanes' loads of one element are one contiguous run (a pair's own matrix is contiguous: 64
        // lanes would touch 64 lines per element, ~100 cycles a load against 4 an FMA): element e of
        // primitive i of lane position pos at lbase[pos / 64] + (i H S + e) 64 + pos % 64
        const double *le;
        const float *le32;
        const long long *lbase;
        // J/K of quartetV with K rows in LDS (kcols > 0): column of the first function of each
        // lane-side pair's shells a and b among the functions of their angular momenta, the AO of
        // each column, and the number of columns
        const int *kcol_a, *kcol_b, *kao;
        int kcols;
    };

    template <int LA, int LB, int LC, int LD>
    struct Cls
    {
        static constexpr int L = LA + LB + LC + LD;
        static constexpr int HP = nHerm(LA + LB), HQ = nHerm(LC + LD), HL = nHerm(L);
        static constexpr int SA = nSph(LA), SB = nSph(LB), SC = nSph(LC), SD = nSph(LD);
        static constexpr int SP = SA * SB, SQ = SC * SD;

        // ---- one-lane-per-quartet plan: per-lane doubles of I (S_lane x NC) + X (H_lane x NC)
        // + R stay within kBudget (the region where the compiler keeps them in registers)
        static constexpr int kBudget = 160;
        // Pinned: at 192 the ket-on-lanes (ff|ss) form (one static pass of all 49 columns
        // instead of two of 35) gives a wrong lane-side J on the GPU (a few hundred elements off
        // by up to 5%; its K and uniform-side J are right; cause not found).  Raise only with
        // every changed form checked element-wise against the oracle.
        static_assert(kBudget == 160, "one-lane register budget: see the comment above");
        static constexpr int ncFor(int sl, int hl, int su)
        {
            const int nc = (kBudget - (HL + L)) / (sl + hl);
            return nc < 1 ? 0 : (nc > su ? su : nc);
        }
        static constexpr int NC0 = ncFor(SP, HP, SQ);   // lanes = bra, uniform = ket
        static constexpr int NC1 = ncFor(SQ, HQ, SP);   // lanes = ket, uniform = bra
        // FP32 form: the same register budget holds twice as many values
        static constexpr int ncFor32(int sl, int hl, int su)
        {
            const int nc = (2 * kBudget - (HL + L)) / (sl + hl);
            return nc < 1 ? 0 : (nc > su ? su : nc);
        }
        static constexpr int NC0f = ncFor32(SP, HP, SQ);
        static constexpr int NC1f = ncFor32(SQ, HQ, SP);
        // Whether the one-lane form is built: at most three column passes (each its own instance) or
        // up to seven of at least three columns, and at most 5500 FMAs in the unrolled transforms.
        // Past that most run 2-28 times slower than the one-wave form (spilled registers,
        // code beyond the instruction cache: (ff|ps) FP32 28x, (fd|ps) FP32 27x, (dp|dp) FP64 1.2 ms
        // for one wave), which then serves the class pair under this variant too.  Not all: (fp|ds) at 40
        // atoms took 95 ms with the bra on the lanes and takes 102 in the one-wave form.
        static constexpr bool laneBuilt(int nc, int sl, int hl, int su, int hu)
        {
            if (nc < 1)
                return false;
            const int passes = ceilDiv(su, nc);
            return (passes <= 3 || (passes <= 7 && nc >= 3)) && nc * (hl * hu + sl * hl) <= 5500;
        }
        static constexpr bool kLane0 = laneBuilt(NC0, SP, HP, SQ, HQ), kLane1 = laneBuilt(NC1, SQ, HQ, SP, HP);
        static constexpr bool kLane0f = laneBuilt(NC0f, SP, HP, SQ, HQ), kLane1f = laneBuilt(NC1f, SQ, HQ, SP, HP);
        template <typename T, bool SWAP>
        static constexpr int nc() { return sizeof(T) == 4 ? (SWAP ? NC1f : NC0f) : (SWAP ? NC1 : NC0); }
    };

    // ------------------------------------------------------------------------------- dense out
    template <class C>
    __device__ __forceinline__ void denseStore(const KArgs &A, double v, int mn, int kl, int a0,
                                               int b0, int c0, int d0)
    {
        const long long n = A.nbf;
        const int mu = mn / C::SB, nu = mn - mu * C::SB;
        const int ka = kl / C::SD, la = kl - ka * C::SD;
        const long long i = a0 + mu, j = b0 + nu, k = c0 + ka, l = d0 + la;
        if (A.kind == 4)
        {
            double *o = A.out;
            o[((i * n + j) * n + k) * n + l] = v;
            o[((i * n + j) * n + l) * n + k] = v;
            o[((j * n + i) * n + k) * n + l] = v;
            o[((j * n + i) * n + l) * n + k] = v;
            o[((k * n + l) * n + i) * n + j] = v;
            o[((k * n + l) * n + j) * n + i] = v;
            o[((l * n + k) * n + i) * n + j] = v;
            o[((l * n + k) * n + j) * n + i] = v;
        }
        else if (A.kind == 3)
        {
            A.out[(i * n + j) * A.naux + k] = v;
            A.out[(j * n + i) * A.naux + k] = v;
        }
        else
        {
            A.out[i * A.naux + k] = v;
            A.out[k * A.naux + i] = v;
        }
    }

    // Runs of adjacent lanes with equal key (a shell of the lane-side pair): per-lane masks of a
    // segmented suffix sum (step i adds the lane 2^i above when it is in the same run), the run
    // head, and whether any lane of the run holds a quartet.
    struct LaneRuns
    {
        unsigned ok;    // bit i: lane + 2^i is in this lane's run
        bool head;      // first lane of its run
        bool any;       // (head lanes) some lane of the run is active
    };

    __device__ __forceinline__ LaneRuns laneRuns(int key, bool active, int lane)
    {
        LaneRuns r;
        const int prev = __shfl_up(key, 1, 64);
        r.head = lane == 0 || prev != key;
        // run id = lane index of the run head (prefix max of head ? lane : 0)
        int id = r.head ? lane : 0;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1)
        {
            const int x = __shfl_up(id, o, 64);
            if (lane >= o)
                id = max(id, x);
        }
        r.ok = 0;
        int act = active ? 1 : 0;
#pragma unroll
        for (int i = 0; i < 6; i++)
        {
            const int o = 1 << i;
            const int xid = __shfl_down(id, o, 64);
            const int xa = __shfl_down(act, o, 64);
            const bool same = lane + o < 64 && xid == id;
            if (same)
            {
                r.ok |= 1u << i;
                act |= xa;
            }
        }
        r.any = act != 0;
        return r;
    }

    __device__ __forceinline__ void ldsAdd(double *p, double v)
    {
        __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    // Adds v of every lane of a run into one address, by the run's head lane (all lanes call).
    __device__ __forceinline__ void runAtomicAdd(const LaneRuns &r, double *addr, double v)
    {
#pragma unroll
        for (int i = 0; i < 6; i++)
        {
            const double x = __shfl_down(v, 1 << i, 64);
            if (r.ok & (1u << i))
                v += x;
        }
        if (r.head && r.any)
            unsafeAtomicAdd(addr, v);
    }

    // MODE_SUM: a wave's sums (per lane) to its molecule's.  Once per run of tasks of a molecule:
    // additions to one line run at about 60 M/s, which a flush per task would exhaust.
    __device__ __forceinline__ void flushSums(const KArgs &A, int mol, int lane, double sabs, double ssum)
    {
        sabs = waveSum(sabs);
        ssum = waveSum(ssum);
        if (lane == 0)
        {
            double *o = A.out + 4 * static_cast<long long>(mol) + (A.kind == 3 ? 0 : 2);
            unsafeAtomicAdd(o, sabs);
            unsafeAtomicAdd(o + 1, ssum);
        }
    }

    // Elements h * S + s of a pair's E matrix, without the structural zeros when SKIP
    template <int La, int Lb, bool SKIP>
    struct EList
    {
        static constexpr int S = nSph(La) * nSph(Lb), N = nHerm(La + Lb) * S;
        int n = 0;
        int e[N]{};
        constexpr EList()
        {
            constexpr EPattern<La, Lb> P{};
            for (int i = 0; i < N; i++)
                if (!SKIP || P.nz[i / S][i % S])
                    e[n++] = i;
        }
    };

    template <int N, typename F, int... I>
    __device__ __forceinline__ void forEachIntImpl(F &&f, std::integer_sequence<int, I...>)
    {
        (f(std::integral_constant<int, I>{}), ...);
    }
    template <int N, typename F>
    __device__ __forceinline__ void forEachInt(F &&f)
    {
        forEachIntImpl<N>(f, std::make_integer_sequence<int, N>{});
    }

    // ------------------------------------------------------------------------------- quartetV
    // One quartet per lane: lane-side pair l (64 consecutive sorted positions) against the
    // wave-uniform pair u.  SWAP = false: lanes = bra, u = ket; SWAP = true: lanes = ket, u = bra.
    // T: type of R, the E matrices and both transforms (double; float for the reduced-precision
    // J/K quartets, whose Boys values, epilogue and accumulation stay double).
    // jl (J/K only, SL entries per lane): this lane's J contributions to its lane-side pair,
    // scaled by 2f, accumulated over a run of tasks that share the lane-side pairs and added to J
    // by the caller at its end.
    // MODE_SUM: the lane's weighted sums of |value| and value are added to jl[0] and jl[1], which
    // the caller adds to the molecule's sums once for a run of tasks of one molecule.
    template <int LA, int LB, int LC, int LD, int MODE, bool SWAP, typename T>
    __device__ __forceinline__ void quartetVTask(const KArgs &A, int q, int local, int lane, double *jl,
                                                 double *sK = nullptr)
    {
        using C = Cls<LA, LB, LC, LD>;
        constexpr int L = C::L, HL = C::HL;
        // lane side (La, Lb), uniform side (Ua, Ub)
        constexpr int La = SWAP ? LC : LA, Lb = SWAP ? LD : LB;
        constexpr int Ua = SWAP ? LA : LC, Ub = SWAP ? LB : LD;
        constexpr int SLa = nSph(La), SLb = nSph(Lb), SUa = nSph(Ua), SUb = nSph(Ub);
        constexpr int SL = SLa * SLb, SU = SUa * SUb;
        constexpr int HLn = nHerm(La + Lb), HU = nHerm(Ua + Ub);
        constexpr int NC = C::template nc<T, SWAP>();
        constexpr int NPASS = ceilDiv(SU, NC);
        constexpr bool F32 = sizeof(T) == 4;
        // Skipping structural zeros scatters the loads of E (no wide contiguous loads); it pays
        // where each loaded value feeds several FMAs: lane side with >= 2 columns per pass,
        // uniform side with >= 4 Hermite rows of X.
        // The lane side's E interleaved over the block's lanes (wave-uniform base + lane); dense
        // tensors, whose lanes are not aligned to the blocks, read it as stored.
        constexpr bool kInter = MODE != MODE_DENSE;
        constexpr int ES = kInter ? 64 : 1;
        constexpr bool kSkipL = NC >= 2;
        constexpr bool kSkipU = HLn >= 4;
        static_assert(!F32 || MODE == MODE_JK || MODE == MODE_SUM, "FP32 forms: J/K and RI sums");
        const DPairs &LP = SWAP ? A.ket : A.bra;
        const DPairs &UP = SWAP ? A.bra : A.ket;

        // lanes cover lane positions local .. local + 63; p is the lane's Schwarz-order position
        // (through A.lperm for J/K)
        const int plo = uniform(A.plo[q]), phi = uniform(A.phi[q]);
        const bool permuted = A.lperm != nullptr;
        // the last group of a lane-block-major table runs G blocks, some past the lane side
        if (local >= LP.n)
            return;
        if (permuted ? (plo >= A.bqhi[local >> 6] || phi <= A.bqlo[local >> 6])
                     : (plo >= local + 64 || phi <= local))
            return;   // no lane has a quartet
        const int pl = local + lane;
        const bool inside = !permuted || pl < LP.n;
        const int p = permuted ? A.lperm[inside ? pl : local] : pl;
        const bool active = inside && p >= plo && p < phi;
        const int u = uniform(UP.order[q]);
        const int l = LP.order[active || permuted ? p : local];
        const int upoff = uniform(UP.poff[u]), ucnt = uniform(UP.pcnt[u]);
        const int lpoff = LP.poff[l], lcnt = active ? LP.pcnt[l] : 0;
        // the ket's E carries the sign (-1)^{t'+u'+v'}
        const T *eUb, *eLb;
        if constexpr (F32)
        {
            eUb = SWAP ? UP.eb32 : UP.ek32;
            eLb = A.le32;
        }
        else
        {
            eUb = SWAP ? UP.eb : UP.ek;
            eLb = kInter ? A.le : LP.eb;
        }
        const cptr<T> eU = constView(eUb + static_cast<size_t>(upoff) * HU * SU);
        const cptr<double> ppU = constView(reinterpret_cast<const double *>(UP.pp + upoff));
        const T *__restrict__ eL;
        if constexpr (kInter)
            eL = eLb + uniform(A.lbase[local >> 6]);
        else
            eL = eLb + static_cast<size_t>(lpoff) * HLn * SL;

        const int l0 = active ? LP.ao_a[l] : 0, l1 = active ? LP.ao_b[l] : 0;
        const int u0 = uniform(UP.ao_a[u]), u1 = uniform(UP.ao_b[u]);
        double f = 1.0;
        if constexpr (MODE == MODE_JK)
        {
            if (LP.sh_a[l] == LP.sh_b[l])
                f *= 0.5;
            if (UP.sh_a[u] == UP.sh_b[u])
                f *= 0.5;
            if (A.same_class && p == q)
                f *= 0.5;
            if (!active)
                f = 0.0;
        }
        const long long n = A.nbf;
        const double *D = A.D;
        // K rows of the uniform pair's functions (r: first shell 0 .. SUa - 1, then the second) on the
        // columns of the lane pair's shells: summed in LDS over the workgroup's lanes (kcols > 0),
        // else added to K, where with a shell-ordered lane side the lanes of one first shell add
        // their sum once (runs of adjacent lanes)
        LaneRuns runs{};
        int la0 = l0, ca = 0, cb = 0;
        if constexpr (MODE == MODE_JK)
        {
            if (A.kcols > 0)
            {
                ca = A.kcol_a[l];
                cb = A.kcol_b[l];
            }
            else if (permuted)
            {
                la0 = LP.ao_a[l];
                runs = laneRuns(la0, active, lane);
            }
        }
        auto addA = [&](int r, long long row, int al, double v) {
            if (A.kcols > 0)
            {
                if (active)
                    ldsAdd(&sK[r * A.kcols + ca + al], v);
            }
            else if (permuted)
                runAtomicAdd(runs, &A.K[row * n + la0 + al], v);
            else if (active)
                unsafeAtomicAdd(&A.K[row * n + l0 + al], v);
        };
        auto addB = [&](int r, long long row, int be, double v) {
            if (!active)
                return;
            if (A.kcols > 0)
                ldsAdd(&sK[r * A.kcols + cb + be], v);
            else
                unsafeAtomicAdd(&A.K[row * n + l1 + be], v);
        };
        double sabs = 0.0, ssum = 0.0;   // MODE_SUM

        // Passes stay a runtime loop (unrolling them lets the compiler overlap the live ranges of
        // successive passes and spill), but each pass runs its own instance of the body with a
        // compile-time pass index, so the column tests fold away and the uniform side's
        // structural zeros are skipped per column.
        auto passBody = [&](auto passC) {
            // a compile-time constant for the instanced passes, a runtime index otherwise
            const int pass = static_cast<int>(passC);
            constexpr bool kStaticPass = !std::is_same_v<decltype(passC), int>;
            T I[SL * NC];
#pragma unroll
            for (int e = 0; e < SL * NC; e++)
                I[e] = T(0);

            for (int i = 0; i < lcnt; i++)
            {
                const double4 Pl = LP.pp[lpoff + i];
                T X[HLn * NC];
#pragma unroll
                for (int e = 0; e < HLn * NC; e++)
                    X[e] = T(0);
                for (int k = 0; k < ucnt; k++)
                {
                    const double4 Pu{ppU[4 * k], ppU[4 * k + 1], ppU[4 * k + 2], ppU[4 * k + 3]};
                    const double4 &Pb = SWAP ? Pu : Pl;
                    const double4 &Pk = SWAP ? Pl : Pu;
                    const double pq = Pb.x * Pk.x, ps = Pb.x + Pk.x;
                    const double alpha = pq / ps;
                    const double X_ = Pb.y - Pk.y, Y_ = Pb.z - Pk.z, Z_ = Pb.w - Pk.w;
                    const double Tb = alpha * (X_ * X_ + Y_ * Y_ + Z_ * Z_);
                    double F[L + 1];
                    boysF<L>(Tb, A.boys, F);
                    T R[HL + L];
                    double sc = kTwoPi52 / (pq * sqrt(ps));
#pragma unroll
                    for (int m = 0; m <= L; m++)
                    {
                        R[m] = T(F[m] * sc);
                        sc *= -2.0 * alpha;
                    }
                    hermiteR<L, T>(R, T(X_), T(Y_), T(Z_));
                    const cptr<T> ek = eU + static_cast<size_t>(k) * HU * SU;
                    constexpr RSumTab<L, HLn, HU> RS{};
                    constexpr EPattern<Ua, Ub> PU{};   // the uniform side's structural zeros
#pragma unroll
                    for (int h = 0; h < HLn; h++)
#pragma unroll
                        for (int g = 0; g < HU; g++)
                        {
                            const T r = R[RS.v[h * HU + g]];
#pragma unroll
                            for (int c = 0; c < NC; c++)
                                if (pass * NC + c < SU &&
                                    (!kSkipU || !kStaticPass || PU.nz[g][pass * NC + c]))
                                    X[h * NC + c] = fma(r, ek[g * SU + pass * NC + c], X[h * NC + c]);
                        }
                }
                // Elements of the lane side's E (about half are structural zeros, skipped) in groups,
                // the next group's loads in flight over this one's FMAs: left to itself the compiler
                // waits for each load before it issues the next.  The two groups take the registers
                // that R held.
                typedef const T __attribute__((address_space(1))) *Row;
                constexpr EList<La, Lb, kSkipL> EL{};
                constexpr int G = (HL + L) / 2 < 2 ? 2 : ((HL + L) / 2 > 16 ? 16 : (HL + L) / 2);
                constexpr int NG = ceilDiv(EL.n, G);
                T eb[2][G];
                auto load = [&](auto gC) {
                    constexpr int g = decltype(gC)::value;
                    // the group's (uniform) address anew, else all of them are formed ahead
                    Row er = (Row)(eL + (static_cast<size_t>(i) * (HLn * SL) + EL.e[g * G]) * ES);
                    if constexpr (kInter)
                        asm("" : "+s"(er));
#pragma unroll
                    for (int j = 0; j < G; j++)
                        if (g * G + j < EL.n)
                            eb[g & 1][j] = er[(EL.e[g * G + j] - EL.e[g * G]) * ES + (kInter ? lane : 0)];
                };
                load(std::integral_constant<int, 0>{});
                forEachInt<NG>([&](auto gC) {
                    constexpr int g = decltype(gC)::value;
                    if constexpr (g + 1 < NG)
                        load(std::integral_constant<int, g + 1>{});
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < G; j++)
                        if (g * G + j < EL.n)
                        {
                            const int h = EL.e[g * G + j] / SL, s = EL.e[g * G + j] % SL;
#pragma unroll
                            for (int c = 0; c < NC; c++)
                                I[s * NC + c] = fma(eb[g & 1][j], X[h * NC + c], I[s * NC + c]);
                        }
                    __builtin_amdgcn_sched_barrier(0);
                });
            }

            // ---- epilogue for the columns of this pass: I[s][c] = (l s | u pass*NC + c)
            if constexpr (MODE == MODE_JK)
            {
                // The lanes' density blocks once per pass, into the registers that X and R held: read
                // where they are used they are read again for every component of the other shells
                // (the additions in between may alias them), a line per lane each time.
                auto readD = [&](auto &d, auto rows, auto cols, auto &&at, auto &&wanted) {
#pragma unroll
                    for (int r = 0; r < decltype(rows)::value; r++)
#pragma unroll
                        for (int c = 0; c < decltype(cols)::value; c++)
                            if (wanted(r))
                                d[r * decltype(cols)::value + c] = at(r, c);
                    __builtin_amdgcn_sched_barrier(0);
                };
                using ia = std::integral_constant<int, SLa>;
                using ib = std::integral_constant<int, SLb>;
                using ua = std::integral_constant<int, SUa>;
                using ub = std::integral_constant<int, SUb>;
                auto every = [](int) { return true; };
                // first index ga of some column of this pass
                auto inPass = [&](int ga) {
                    bool any = false;
#pragma unroll
                    for (int de = 0; de < SUb; de++)
                        any |= (ga * SUb + de) / NC == pass;
                    return any;
                };
                // J_l += 2f I D_u (accumulated over passes); J_u += 2f I^T D_l (wave sum)
                double dl[SL];
                readD(dl, ia{}, ib{}, [&](int al, int be) { return active ? D[(l0 + al) * n + l1 + be] : 0.0; }, every);
#pragma unroll
                for (int c = 0; c < NC; c++)
                {
                    const int su = pass * NC + c;
                    if (su >= SU)
                        continue;
                    const int ga = su / SUb, de = su % SUb;
                    const double du = 2.0 * f * D[(u0 + ga) * n + u1 + de];
                    double ju = 0.0;
#pragma unroll
                    for (int s = 0; s < SL; s++)
                    {
                        const double iv = I[s * NC + c];
                        jl[s] = fma(iv, du, jl[s]);
                        ju = fma(iv, dl[s], ju);
                    }
                    ju = waveSum(2.0 * f * ju);
                    if (lane == 0)
                        unsafeAtomicAdd(&A.J[(u0 + ga) * n + u1 + de], ju);
                }
                {
                    // K[u0+ga][l0+al] += f sum_{be, de} I D[u1+de][l1+be]
                    // K[u0+ga][l1+be] += f sum_{al, de} I D[u1+de][l0+al]
                    // K[u1+de][l0+al] += f sum_{be, ga} I D[u0+ga][l1+be]
                    // K[u1+de][l1+be] += f sum_{al, ga} I D[u0+ga][l0+al]
                    // The wave-uniform shell indexes the row of K (and of the symmetric D): the
                    // unique-quartet contributions are symmetrised at the end (K + K^T), so
                    // either triangle may receive them, and with the row fixed across the wave
                    // its atomics and loads stay on a few rows that remain in L2.
                    double dbb[SUb * SLb], dba[SUb * SLa];   // D[u1 + de][l1 + be], D[u1 + de][l0 + al]
                    readD(dbb, ub{}, ib{}, [&](int de, int be) { return D[(u1 + de) * n + l1 + be]; }, every);
                    readD(dba, ub{}, ia{}, [&](int de, int al) { return D[(u1 + de) * n + l0 + al]; }, every);
#pragma unroll
                    for (int ga = 0; ga < SUa; ga++)
                    {
                        if (!inPass(ga))
                            continue;
#pragma unroll
                        for (int al = 0; al < SLa; al++)
                        {
                            double s = 0.0;
#pragma unroll
                            for (int be = 0; be < SLb; be++)
#pragma unroll
                                for (int de = 0; de < SUb; de++)
                                {
                                    const int su = ga * SUb + de;
                                    if (su / NC != pass)
                                        continue;
                                    s = fma(double(I[(al * SLb + be) * NC + su % NC]),
                                            dbb[de * SLb + be], s);
                                }
                            addA(ga, u0 + ga, al, f * s);
                        }
#pragma unroll
                        for (int be = 0; be < SLb; be++)
                        {
                            double s = 0.0;
#pragma unroll
                            for (int al = 0; al < SLa; al++)
#pragma unroll
                                for (int de = 0; de < SUb; de++)
                                {
                                    const int su = ga * SUb + de;
                                    if (su / NC != pass)
                                        continue;
                                    s = fma(double(I[(al * SLb + be) * NC + su % NC]),
                                            dba[de * SLa + al], s);
                                }
                            addB(ga, u0 + ga, be, f * s);
                        }
                    }
                    double dab[SUa * SLb], daa[SUa * SLa];   // D[u0 + ga][l1 + be], D[u0 + ga][l0 + al]
                    readD(dab, ua{}, ib{}, [&](int ga, int be) { return D[(u0 + ga) * n + l1 + be]; }, inPass);
                    readD(daa, ua{}, ia{}, [&](int ga, int al) { return D[(u0 + ga) * n + l0 + al]; }, inPass);
#pragma unroll
                    for (int de = 0; de < SUb; de++)
                    {
                        bool any = false;
#pragma unroll
                        for (int ga = 0; ga < SUa; ga++)
                            any |= (ga * SUb + de) / NC == pass;
                        if (!any)
                            continue;
#pragma unroll
                        for (int al = 0; al < SLa; al++)
                        {
                            double s = 0.0;
#pragma unroll
                            for (int be = 0; be < SLb; be++)
#pragma unroll
                                for (int ga = 0; ga < SUa; ga++)
                                {
                                    const int su = ga * SUb + de;
                                    if (su / NC != pass)
                                        continue;
                                    s = fma(double(I[(al * SLb + be) * NC + su % NC]),
                                            dab[ga * SLb + be], s);
                                }
                            addA(SUa + de, u1 + de, al, f * s);
                        }
#pragma unroll
                        for (int be = 0; be < SLb; be++)
                        {
                            double s = 0.0;
#pragma unroll
                            for (int al = 0; al < SLa; al++)
#pragma unroll
                                for (int ga = 0; ga < SUa; ga++)
                                {
                                    const int su = ga * SUb + de;
                                    if (su / NC != pass)
                                        continue;
                                    s = fma(double(I[(al * SLb + be) * NC + su % NC]),
                                            daa[ga * SLa + al], s);
                                }
                            addB(SUa + de, u1 + de, be, f * s);
                        }
                    }
                }
            }
            else if constexpr (MODE == MODE_DENSE)
            {
                static_assert(!SWAP, "dense output keeps the bra on the lanes");
                if (active)
#pragma unroll
                    for (int s = 0; s < SL; s++)
#pragma unroll
                        for (int c = 0; c < NC; c++)
                            if (pass * NC + c < SU)
                                denseStore<C>(A, I[s * NC + c], s, pass * NC + c, l0, l1, u0, u1);
            }
            else
            {
                static_assert(MODE == MODE_SUM && !SWAP, "sums keep the bra on the lanes");
                if (active)
#pragma unroll
                    for (int s = 0; s < SL; s++)
#pragma unroll
                        for (int c = 0; c < NC; c++)
                            if (pass * NC + c < SU)
                            {
                                const double v = I[s * NC + c];
                                sabs += fabs(v);
                                ssum += v;
                            }
            }
        };
        forEachPass<NPASS>(passBody);

        if constexpr (MODE == MODE_SUM)
        {
            // images in the dense tensor: (ab|P) and (ba|P) for distinct shells; (P|Q), (Q|P)
            const bool one = A.kind == 3 ? LP.sh_a[l] == LP.sh_b[l] : (A.same_class && p == q);
            const double w = active ? (one ? 1.0 : 2.0) : 0.0;
            jl[0] = fma(w, sabs, jl[0]);
            jl[1] = fma(w, ssum, jl[1]);
        }
    }

    // Uniform-major tables: each wave takes a contiguous range of tasks, which share the uniform
    // pair q and step through its 64-lane blocks (the task -> q search runs once per wave).
    // Lane-block-major tables (A.block_major): a task is one uniform pair q against one lane
    // block of a group of G blocks; a group's tasks are consecutive (q outer, block inner) and
    // wave w takes tasks w, w + nw, ... with nw the resident waves, so the waves in flight share
    // one group of lane-side pairs, whose E matrices (the larger per-task traffic) stay in L2,
    // and each uniform pair's E is read once per group.  With G dividing nw a wave stays on one
    // lane block within a group, so its J contributions to the lane-side pairs are summed in
    // registers and added to J once per block.
    template <int LA, int LB, int LC, int LD, int MODE, bool SWAP, typename T>
    __global__ __launch_bounds__(256) void quartetV(const KArgs A)
    {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        const long long nw = static_cast<long long>(gridDim.x) * 4;
        const long long w = static_cast<long long>(blockIdx.x) * 4 + wave;
        constexpr int SLb = nSph(SWAP ? LD : LB);
        constexpr int SL = nSph(SWAP ? LC : LA) * SLb;
        double jl[MODE == MODE_SUM ? 2 : SL];
        if constexpr (MODE == MODE_JK)
        {
            const DPairs &LP = SWAP ? A.ket : A.bra;
            auto flushJ = [&](int b) {
                const int p = 64 * b + lane;
                if (p < LP.n)
                {
                    const int l = LP.order[A.lperm ? A.lperm[p] : p];
                    const long long r0 = LP.ao_a[l], r1 = LP.ao_b[l];
#pragma unroll
                    for (int s = 0; s < SL; s++)
                        unsafeAtomicAdd(&A.J[(r0 + s / SLb) * A.nbf + r1 + s % SLb], jl[s]);
                }
            };
            const int gs = A.gshift;
            const int ng = (A.nblk + (1 << gs) - 1) >> gs;
            int g = 0, q0 = 0, b = -1;
            long long base = 0, next = 0;
            // K rows in LDS: the workgroup's four waves take four blocks of one uniform pair
            // (G >= 4), so after each round of tasks its rows are complete and go to K
            extern __shared__ double sKrows[];
            constexpr int SUa = nSph(SWAP ? LA : LC), SUb = nSph(SWAP ? LB : LD);
            const int nK = (SUa + SUb) * A.kcols;
            if (A.kcols > 0)
            {
                for (int e = threadIdx.x; e < nK; e += 256)
                    sKrows[e] = 0.0;
                __syncthreads();
            }
            for (long long t = w; t < A.ntasks; t += nw)
            {
                if (t >= next)
                {
                    g = uniform(findKet(A.bprefix, ng, t));
                    base = A.bprefix[g];
                    next = A.bprefix[g + 1];
                    q0 = uniform(A.bq0[g]);
                }
                const long long local = t - base;
                const int bt = (g << gs) + static_cast<int>(local & ((1LL << gs) - 1));
                const int q = q0 + static_cast<int>(local >> gs);
                if (bt != b)
                {
                    if (b >= 0)
                        flushJ(b);
#pragma unroll
                    for (int s = 0; s < SL; s++)
                        jl[s] = 0.0;
                    b = bt;
                }
                quartetVTask<LA, LB, LC, LD, MODE, SWAP, T>(A, q, 64 * b, lane, jl, sKrows);
                if (A.kcols > 0)
                {
                    __syncthreads();
                    const DPairs &UP = SWAP ? A.bra : A.ket;
                    const int u = uniform(UP.order[q]);
                    const long long u0 = uniform(UP.ao_a[u]), u1 = uniform(UP.ao_b[u]);
                    for (int r = 0; r < SUa + SUb; r++)
                    {
                        double *row = A.K + (r < SUa ? u0 + r : u1 + r - SUa) * A.nbf;
                        for (int e = threadIdx.x; e < A.kcols; e += 256)
                        {
                            const double v = sKrows[r * A.kcols + e];
                            if (v != 0.0)
                            {
                                sKrows[r * A.kcols + e] = 0.0;
                                unsafeAtomicAdd(row + A.kao[e], v);
                            }
                        }
                    }
                    __syncthreads();
                }
            }
            if (b >= 0)
                flushJ(b);
            return;
        }
        else
        {
            const long long t0 = A.ntasks * w / nw, t1 = A.ntasks * (w + 1) / nw;
            if (t0 >= t1)
                return;
            int q = uniform(findKet(A.prefix, A.nket, t0));
            long long base = A.prefix[q], next = A.prefix[q + 1];
            int mol = -1;   // MODE_SUM: the molecule of the sums in jl
            for (long long t = t0; t < t1; t++)
            {
                while (t >= next)
                {
                    q++;
                    base = next;
                    next = A.prefix[q + 1];
                }
                if constexpr (MODE == MODE_SUM)
                {
                    const int m = uniform(A.ket.mol[A.ket.order[q]]);
                    if (m != mol)
                    {
                        if (mol >= 0)
                            flushSums(A, mol, lane, jl[0], jl[1]);
                        mol = m;
                        jl[0] = jl[1] = 0.0;
                    }
                }
                // sums: aligned blocks of 64 positions (the interleaved E's)
                const int first = MODE == MODE_SUM ? uniform(A.plo[q]) & ~63 : uniform(A.plo[q]);
                quartetVTask<LA, LB, LC, LD, MODE, SWAP, T>(A, q, first + 64 * static_cast<int>(t - base),
                                                            lane, jl);
            }
            if constexpr (MODE == MODE_SUM)
                flushSums(A, mol, lane, jl[0], jl[1]);
        }
    }

    template <int LA, int LB, int LC, int LD, int MODE, bool SWAP, typename T>
    void launchValu(const KArgs &A, hipStream_t s)
    {
        if (A.ntasks <= 0)
            return;
        // uniform-major: contiguous task ranges per wave, up to 8192 workgroups of 4 waves;
        // lane-block-major: as many workgroups as are resident at once, so that one sweep of the
        // waves over the task order keeps them all on the same few lane blocks
        struct Residency
        {
            int blocks, cus;
        };
        static const Residency resident = [] {
            int per_cu = 0, dev = 0, ncu = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                        &per_cu, reinterpret_cast<const void *>(&quartetV<LA, LB, LC, LD, MODE, SWAP, T>), 256, 0) !=
                        hipSuccess ||
                hipGetDevice(&dev) != hipSuccess ||
                hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
                return Residency{8192, 256};
            return Residency{std::max(1, per_cu) * std::max(1, ncu), std::max(1, ncu)};
        }();
        // K rows of the uniform pair in LDS
        constexpr int SUa = nSph(SWAP ? LA : LC), SUb = nSph(SWAP ? LB : LD);
        const size_t lds = MODE == MODE_JK ? sizeof(double) * (SUa + SUb) * A.kcols : 0;
        long long cap = 8192;
        if (A.block_major)
            cap = std::min<long long>({resident.blocks, cap, lds ? resident.cus * static_cast<long long>(163840 / lds) : cap});
        else if (MODE == MODE_SUM)
            cap = std::min<long long>(4 * resident.blocks, cap);   // each wave ends in one addition per molecule
        long long wg = (A.ntasks + 3) / 4;
        int grid = static_cast<int>(wg < cap ? wg : cap);
        hipLaunchKernelGGL((quartetV<LA, LB, LC, LD, MODE, SWAP, T>), dim3(grid), dim3(256), lds, s, A);
    }

    // The FP32 forms (J/K and RI sums).
    template <int LA, int LB, int LC, int LD, int MODE>
    void registerQuartet32()
    {
        using C = Cls<LA, LB, LC, LD>;
        constexpr bool same = LA == LC && LB == LD;
        if constexpr ((MODE == MODE_JK || MODE == MODE_SUM) && C::kLane0f)
        {
            KernelSlot &s = kernelSlot(MODE, LA, LB, LC, LD, VAR_VALU_BRA32);
            s.fn = &launchValu<LA, LB, LC, LD, MODE, false, float>;
            s.width = 64;
            s.swap = false;
            s.nc = C::NC0f;
        }
        if constexpr (MODE == MODE_JK && C::kLane1f && !same)
        {
            KernelSlot &s = kernelSlot(MODE, LA, LB, LC, LD, VAR_VALU_KET32);
            s.fn = &launchValu<LA, LB, LC, LD, MODE, true, float>;
            s.width = 64;
            s.swap = true;
            s.nc = C::NC1f;
        }
    }

    // Registers the one-lane variants the class supports in this mode.  The ket-on-lanes form
    // only serves J/K between different classes (dense outputs and sums keep the bra on
    // the lanes; for one class both forms coincide).
    // FORMS: 1 the FP64 forms, 2 the FP32 forms, 3 both (lets the build compile them apart).
    template <int LA, int LB, int LC, int LD, int MODE, int FORMS = 3>
    void registerQuartet()
    {
        using C = Cls<LA, LB, LC, LD>;
        if constexpr (FORMS & 2)
            registerQuartet32<LA, LB, LC, LD, MODE>();
        if constexpr (!(FORMS & 1))
            return;
        if constexpr (C::kLane0)
        {
            KernelSlot &s = kernelSlot(MODE, LA, LB, LC, LD, VAR_VALU_BRA);
            s.fn = &launchValu<LA, LB, LC, LD, MODE, false, double>;
            s.width = 64;
            s.swap = false;
            s.nc = C::NC0;
        }
        constexpr bool same = LA == LC && LB == LD;
        if constexpr (MODE == MODE_JK && C::kLane1 && !same)
        {
            KernelSlot &s = kernelSlot(MODE, LA, LB, LC, LD, VAR_VALU_KET);
            s.fn = &launchValu<LA, LB, LC, LD, MODE, true, double>;
            s.width = 64;
            s.swap = true;
            s.nc = C::NC1;
        }
    }
}
