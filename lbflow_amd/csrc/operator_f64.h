// operator_f64.h -- product of a dense 9x9 / 19x19 FP64 operator with one
// vector per lane, the sums in the reference's order (j ascending, no FMA).
//
// The operator is the same for every lane, so its coefficients come through
// scalar loads and enter the multiplications as SGPR operands.  Read from LDS
// as broadcasts they cost a CU more time than the arithmetic (8 cycles of LDS
// per 16-byte read, 360 reads a wave, against 5800 cycles of FP64 on each of
// four SIMDs), and read through vector loads each one is a round trip.
#pragma once
#include <hip/hip_runtime.h>

#include "lattice.h"

namespace lbf {

// Packed form: for each group of 4 result rows k, for each j (padded to a
// multiple of 4) the 4 coefficients of x[j]: [k / 4][j][k % 4].
constexpr int op_rows4(int Q) { return (Q + 3) / 4; }
constexpr int op_packed(int Q) { return op_rows4(Q) * op_rows4(Q) * 16; }

typedef const double __attribute__((address_space(4))) cdouble;

// f[k] += sum_j op[k][j] x[j] (SET: f[k] = the sum).  Four sums run side by
// side, so a sum's next addition follows the seven instructions of the other
// three, and the coefficients arrive 16 at a time (4 j of 4 rows), the next 16
// requested as soon as the first of this 16 has been used: scalar loads return
// in any order, so a wait for one block waits for every load in flight, and a
// request issued before that wait would be waited for at once.
// MINV: the operator is the inverse transform; terms whose entry of M is 0
// are left out, as the reference leaves them out.
template <int Q, bool SET, bool MINV, int B>
__device__ __forceinline__ void op_block(cdouble* p, const double* x, double* f, double (&c)[16], double (&next)[16],
                                         double (&s)[4])
{
#pragma clang fp contract(off)
    constexpr int R = op_rows4(Q), K0 = 4 * (B / R), J0 = 4 * (B % R);
    bool requested = B + 1 >= R * R;
    auto request = [&]() __attribute__((always_inline)) {
        requested = true;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) next[i] = p[(B + 1) * 16 + i];
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (J0 + jj >= Q || K0 + k >= Q) continue;
            if (MINV && Lattice<Q>::M[J0 + jj][K0 + k] == 0) continue;
            const double v = c[jj * 4 + k] * x[J0 + jj];
            if (!requested) request();
            s[k] = J0 + jj == 0 ? v : s[k] + v;   // every row of M^-1 starts with a non-zero entry
        }
    if (!requested) request();   // a block of left-out terms
    if constexpr (B % R == R - 1) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (K0 + k < Q) f[K0 + k] = SET ? s[k] : f[K0 + k] + s[k];
    }
    if constexpr (B + 1 < R * R) op_block<Q, SET, MINV, B + 1>(p, x, f, next, c, s);
}

template <int Q, bool SET = false, bool MINV = false>
__device__ __forceinline__ void add_operator(const double* packed, const double* x, double* f)
{
    cdouble* p = (cdouble*)packed;
    double c[16], next[16], s[4];
#pragma unroll
    for (int i = 0; i < 16; ++i) c[i] = p[i];
    op_block<Q, SET, MINV, 0>(p, x, f, c, next, s);
}

}  // namespace lbf
