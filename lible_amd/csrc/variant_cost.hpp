// Time estimates of the quartet kernels' forms, from which a class pair's form is chosen when the
// autotuner has not timed them.  Plain C++.
//
// The terms are the counts that the forms' inner loops make (transform FMAs, Hermite-recursion
// steps, MFMAs, E elements loaded, epilogue sums) summed over the waves, one term for the longest
// serial chain of a single wave (which is the time of a small molecule, where every wave runs at
// once), and a constant for the launch.  The coefficients (milliseconds per 10^6 of a count, on
// the MI355X) are a non-negative fit of the logarithm of 2900 timed launches: every form of every class
// pair to (ff|ff) on water clusters of 1 to 10 molecules in def2-SVP, -TZVP and -QZVP and on 2 to
// 19 atoms of the synthetic s to f shells, 0.03 to 200 ms each; the typical residual is a factor of
// 1.45, and single class pairs are further off: (pp|pp) of (H2O)10 def2-TZVP stays on the one-wave form
// at 3.8 ms where the one-lane form takes 1.0, RI sums of two molecules take 3.5 ms (tuned 1.2).  J/K
// time summed over the class pairs, ms, by this rule / by the fastest form of each:
//   H2O SVP 0.77 / 0.74, (H2O)8 SVP 5.5 / 4.9, (H2O)10 TZVP 40 / 35, 7 atoms s-f 9.8 / 8.3,
//   19 atoms s-f 155 / 154;
//   FP32 forms: 0.67 / 0.64, 5.2 / 4.9, 30 / 28, 8.6 / 7.4, 89 / 88
// (the estimate from the mean contraction alone that it replaced, with the one-lane kernels of that
// time: 1.7, 12.2, 72, 19 and 233; FP32 2.3, 11.6, 74, 14 and 149).
#pragma once

#include <algorithm>
#include <cmath>

#include "lbx_common.hpp"

namespace lbx
{
    namespace cost
    {
        // One side of a class pair: angular momenta and primitive pairs per shell pair: the mean,
        // the mean over 64-pair blocks of the largest (what a wave of a one-lane form runs), the
        // largest.
        struct Side
        {
            int la, lb;
            double kmean, klane, kmax;
            int H() const { return nHerm(la + lb); }
            int S() const { return nSph(la) * nSph(lb); }
            int L() const { return la + lb; }
        };

        inline double recursionSteps(int L)
        {
            double r = 0;
            for (int n = 0; n < L; n++)
                for (int m = 1; m <= L - n; m++)
                    r += (m + 1) * (m + 2) / 2;
            return r;
        }

        // One lane per quartet: `waves` tasks of 64 lane-side pairs against one uniform pair, in
        // column passes of nc (R and Boys again in each).  inter: E interleaved over the lanes (J/K and
        // sums; the other modes read it a line per lane); jk: K rows and wave sums in the epilogue.
        inline double laneForm(const Side &lane, const Side &unif, int nc, bool f32, double waves, bool inter, bool jk)
        {
            const int L = lane.L() + unif.L(), su = unif.S(), sl = lane.S();
            const double passes = ceilDiv(su, nc), step = passes * (recursionSteps(L) + 100);
            const double hlsl = double(lane.H()) * sl, hlhu = double(lane.H()) * unif.H();
            const double fma = lane.klane * (unif.kmean * hlhu * su + hlsl * su);
            const double rec = lane.klane * unif.kmean * step;
            const double eLane = lane.klane * hlsl * passes;   // lane-side E elements (a load per lane)
            const double chain = lane.kmax * (unif.kmax * (hlhu * su + step) + hlsl * su);
            // more than three passes share one instance of the pass body, which then spills (in the
            // interleaved forms those with a long body)
            const double shared = passes > 3 && (!inter || nc * (hlhu + hlsl) > (f32 ? 4500 : 1400)) ? 1.0 : 0.0;
            const double big = hlsl > 700 ? 1.0 : 0.0;
            const double rows = nSph(unif.la) + nSph(unif.lb);
            double t;
            // an (ss) lane side: each FMA takes a new scalar load of the uniform side's E
            const double steps = lane.H() == 1 ? lane.klane * unif.kmean : 0.0, uLoads = steps * unif.H() * su;
            if (inter && f32)
                t = waves * (0.0022 * rec + (0.0119 + 0.013 * big) * eLane + 0.0039 * shared * (fma + rec) +
                             0.0036 * uLoads + 0.328 * passes * steps + (jk ? 1.37 * rows + 0.197 * su * su + 10.3 : 0.0)) +
                    (2.41 + 1.74 * shared) * chain;
            else if (inter)
                t = waves * (0.0021 * rec + (0.0212 + 0.0248 * big) * eLane + 0.0179 * shared * (fma + rec) +
                             0.013 * uLoads + 0.207 * passes * steps + (jk ? 0.5 * rows + 0.353 * su * su + 7.27 : 0.0)) +
                    (3.40 + 15.7 * shared) * chain;
            else if (f32)
                t = waves * (0.0033 * rec + (0.0177 + 0.0388 * big) * eLane + 0.0027 * shared * (fma + rec)) +
                    (2.68 + 2.60 * shared) * chain;
            else
                t = waves * (0.0024 * rec + (0.0422 + 0.0176 * big) * eLane + 0.0122 * shared * (fma + rec)) +
                    (3.91 + 9.28 * shared) * chain;
            return 1e-6 * t + (inter && !f32 ? 0.05 : 0.06);
        }

        // One wave per quartet (MFMA).
        inline double waveForm(const Side &bra, const Side &ket, bool f32, double quartets)
        {
            const int L = bra.L() + ket.L(), NQ = ceilDiv(ket.S(), 16), NP = ceilDiv(bra.S(), 16), KQ = ceilDiv(ket.H(), 4);
            const double rows = bra.kmean * bra.H(), kk = bra.kmean * ket.kmean;
            const double mfma = std::ceil(rows / 16) * ket.kmean * KQ * NQ + std::ceil(rows / 4) * NP * NQ;
            const double epilogue = bra.S() * ket.S() * 6 / 64.0 + 20;
            const double batch = std::max(1, std::min(64, 9216 / (8 * nHerm(L))));
            const double kmax = bra.kmax * ket.kmax, steps = recursionSteps(L) / 64;
            const double chain = std::ceil(kmax / batch) * (L + 4) + kmax * (steps + KQ);
            if (f32)
                return 1e-6 * quartets * (0.0379 * mfma + 0.0942 * epilogue) + 1.23e-4 * chain + 0.031;
            return 1e-6 * quartets * (0.0532 * mfma + 0.0016 * kk * steps + 0.107 * epilogue) + 1.97e-4 * chain + 0.029;
        }

        // One workgroup per bra pair and block of ket pairs.
        inline double blockForm(const Side &bra, const Side &ket, bool f32, double quartets)
        {
            const int L = bra.L() + ket.L(), nb = ket.S() >= 48 ? 1 : 48 / ket.S();
            const double groups = std::max(quartets / nb, 1.0);
            const double perWave = std::ceil(std::min<double>(nb, quartets) / 4);   // ket pairs of one wave
            const double batch = std::max(1, std::min(16, 8192 / (8 * nHerm(L))));
            const double rowSets = ceilDiv(bra.H(), 64), steps = recursionSteps(L) / 64;
            const double ket1 = perWave * bra.kmean, prim = ket1 * ket.kmean;
            const double gather = prim * rowSets * ket.H() * ceilDiv(ket.S(), 16);
            const double mfma = ceilDiv(ceilDiv(bra.S(), 16) * ceilDiv(nb * ket.S(), 16), 4) * ceilDiv(bra.H(), 4) * bra.kmean;
            const double levels = ket1 * std::ceil(ket.kmean / batch) * (L + 4);
            const double epilogue = nb * bra.S() * ket.S() * 6 / 256.0;
            const double chain = bra.kmax * perWave *
                                 (std::ceil(ket.kmax / batch) * (L + 4) + ket.kmax * (steps + ket.H() * ket.S() / 8.0));
            if (f32)
                return 1e-6 * groups * (0.0087 * gather + 1.26 * mfma + 0.213 * levels + 0.0388 * prim * steps + 0.425 * epilogue) +
                       4.5e-5 * chain + 0.032;
            return 1e-6 * groups * (0.0215 * gather + 2.09 * mfma + 0.183 * levels + 0.0094 * prim * steps + 0.166 * epilogue) +
                   5.0e-5 * chain + 0.037;
        }
    }
}
