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

namespace lbf {

// Packed form: for each group of 4 result rows k, for each j (padded to a
// multiple of 4) the 4 coefficients of x[j]: [k / 4][j][k % 4].
constexpr int op_rows4(int Q) { return (Q + 3) / 4; }
constexpr int op_packed(int Q) { return op_rows4(Q) * op_rows4(Q) * 16; }

typedef const double __attribute__((address_space(4))) cdouble;

// f[k] += sum_j op[k][j] x[j].  Four sums run side by side, so a sum's next
// addition follows the seven instructions of the other three, and the
// coefficients arrive 16 at a time (4 j of 4 rows), the next 16 requested as
// soon as the first of this 16 has been used: scalar loads return in any
// order, so a wait for one block waits for every load in flight, and a
// request issued before that wait would be waited for at once.
template <int Q>
__device__ __forceinline__ void add_operator(const double* packed, const double* x, double* f)
{
#pragma clang fp contract(off)
    constexpr int R = op_rows4(Q);
    cdouble* p = (cdouble*)packed;
    double c[2][16], s[4];
#pragma unroll
    for (int i = 0; i < 16; ++i) c[0][i] = p[i];
#pragma unroll
    for (int b = 0; b < R * R; ++b) {
        const int k0 = 4 * (b / R), j0 = 4 * (b % R);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (j0 + jj >= Q || k0 + k >= Q) continue;
                const double v = c[b & 1][jj * 4 + k] * x[j0 + jj];
                if (jj == 0 && k == 0 && b + 1 < R * R) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < 16; ++i) c[(b + 1) & 1][i] = p[(b + 1) * 16 + i];
                    __builtin_amdgcn_sched_barrier(0);
                }
                s[k] = j0 + jj == 0 ? v : s[k] + v;
            }
        if (b % R == R - 1)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (k0 + k < Q) f[k0 + k] += s[k];
    }
}

}  // namespace lbf
