// Instantiation unit of the one-wave MFMA quartet kernels (quartet_wave.hpp), compiled once per
// LBX_UNIT with the classes of instances.hip: 0..9 bra = main pair class (J/K, dense, blocks,
// sums, diagonal), 10, 11 bra = auxiliary shell l = 4, 5; 12..21 the FP32 J/K forms of units 0..9;
// 22..26 J/K (FP64) of bra = (g, LBX_UNIT - 22) for the class pairs this form covers
// (WavePlan::kFitsG; generic.hip runs the others).
#include "quartet_wave.hpp"

#ifndef LBX_UNIT
#error "LBX_UNIT must be defined"
#endif

namespace lbx
{
    namespace
    {
        constexpr bool kGUnit = LBX_UNIT >= 22;
        constexpr bool kF32Unit = LBX_UNIT >= 12 && !kGUnit;
        constexpr int kPairUnit = kF32Unit ? LBX_UNIT - 12 : kGUnit ? LBX_UNIT - 12 : LBX_UNIT;

        constexpr int unitLa()
        {
            constexpr int u = kPairUnit;
            if (kGUnit)
                return 4;
            if (u >= 10)
                return u - 6;   // 10 -> 4, 11 -> 5
            int la = 0;
            while (pairClassIdx(la + 1, 0) <= u)
                la++;
            return la;
        }
        constexpr int unitLb() { return kGUnit ? LBX_UNIT - 22 : kPairUnit >= 10 ? 0 : kPairUnit - pairClassIdx(unitLa(), 0); }

        constexpr int PA = unitLa(), PB = unitLb();
        constexpr int CI = pairClassIdx(PA, PB);

        template <int LC, int LD>
        void regEri4()
        {
            if constexpr (kGUnit && pairClassIdx(LC, LD) <= CI)
                if constexpr (WavePlan<PA, PB, LC, LD, double>::kFitsG)
                    registerWave<PA, PB, LC, LD, MODE_JK, 1>();
            if constexpr (kPairUnit < 10 && pairClassIdx(LC, LD) <= CI)
            {
                if constexpr (kF32Unit)
                    registerWave<PA, PB, LC, LD, MODE_JK, 2>();
                else
                {
                    registerWave<PA, PB, LC, LD, MODE_JK, 1>();
                    registerWave<PA, PB, LC, LD, MODE_DENSE, 1>();
                    registerWave<PA, PB, LC, LD, MODE_BLOCK, 1>();
                }
            }
        }

        template <int LC>
        void regEri3()
        {
            if constexpr (!kF32Unit && kPairUnit < 10 && !(LC <= 3 && pairClassIdx(LC, 0) <= CI))
            {
                registerWave<PA, PB, LC, 0, MODE_DENSE, 1>();
                registerWave<PA, PB, LC, 0, MODE_BLOCK, 1>();
            }
            // batched RI sums: eri3 (PA PB | LC), and eri2 (PA | LC) when PB = 0
            if constexpr (kPairUnit < 10)
                registerWave<PA, PB, LC, 0, MODE_SUM, kF32Unit ? 0 : 1>();
        }

        template <int LC>
        void regEri2()
        {
            if constexpr (!kF32Unit && !kGUnit && kPairUnit >= 10 && LC <= PA)
            {
                registerWave<PA, 0, LC, 0, MODE_DENSE, 1>();
                registerWave<PA, 0, LC, 0, MODE_BLOCK, 1>();
                registerWave<PA, 0, LC, 0, MODE_SUM, 1>();
            }
        }

        struct Registrar
        {
            Registrar()
            {
                regEri4<0, 0>();
                regEri4<1, 0>();
                regEri4<1, 1>();
                regEri4<2, 0>();
                regEri4<2, 1>();
                regEri4<2, 2>();
                regEri4<3, 0>();
                regEri4<3, 1>();
                regEri4<3, 2>();
                regEri4<3, 3>();
                regEri4<4, 0>();
                regEri4<4, 1>();
                regEri4<4, 2>();
                regEri4<4, 3>();
                regEri4<4, 4>();
                regEri3<0>();
                regEri3<1>();
                regEri3<2>();
                regEri3<3>();
                regEri3<4>();
                regEri3<5>();
                regEri2<0>();
                regEri2<1>();
                regEri2<2>();
                regEri2<3>();
                regEri2<4>();
                regEri2<5>();
                if constexpr (!kF32Unit && !kGUnit)
                    registerWave<PA, PB, PA, PB, MODE_DIAG, 1>();
            }
        } registrar;
    }
}
