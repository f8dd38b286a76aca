// What the kernels see of a shell-pair class.
#pragma once

#include <hip/hip_runtime.h>

namespace lbx
{
    // Device view of one pair class, passed by value to kernels.
    struct DPairs
    {
        const int *ao_a, *ao_b;     // AO offsets of the two shells, per pair
        const int *sh_a, *sh_b;     // shell indices, per pair (a == b detects diagonal pairs)
        const int *poff, *pcnt;     // first primitive pair and count, per pair
        const double4 *pp;          // per primitive pair: (p, Px, Py, Pz)
        const double *eb;           // E^T [ppair][tuv][mu nu]           (bra use)
        const double *ek;           // (-1)^{t+u+v} E^T [ppair][tuv][mu nu] (ket use)
        const int *order;           // sorted position -> pair index
        const double *q;            // Schwarz factor per sorted position
        int n;
        const float *eb32, *ek32;   // eb, ek rounded to FP32 (mixed precision; may be null)
        // nuclear gradient (may be null until the first gradient call)
        const int *atom_a, *atom_b;   // atom of each shell, per pair
        const double *ra;             // a / (a + b) per primitive pair
        const double *e1b, *e1k;      // d eb / d(A - B)_x, d ek / d(A - B)_x: [ppair][x][tuv][mu nu]
        const int *mol;               // molecule of each pair (batched contexts; may be null)
        const float *e1b32, *e1k32;   // e1b, e1k rounded to FP32 (mixed-precision gradient)
    };
}
