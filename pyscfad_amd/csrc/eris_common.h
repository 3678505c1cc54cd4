// Launchers of eris_kernels.hip (MP2 pair energies, DF integral producer).
#pragma once
#include <hip/hip_runtime.h>

namespace pamd {

hipError_t launch_mp2_pairs(int o, int v, const double *mo, const double *ovov, double *t2,
                            double *e_pair, hipStream_t s);
hipError_t launch_pack_lvv(const double *Lpq, int o, int n, int naux, double *Lvv,
                           hipStream_t s);
hipError_t launch_unpack_lvv_bar(const double *Lvv_bar, int o, int n, int naux, double *Lpq_bar,
                                 hipStream_t s);
hipError_t launch_zero_occ_rows(int o, int n, int naux, double *Lpq_bar, hipStream_t s);
// out = B + B^T (n x n)
hipError_t launch_add_transpose(const double *B, int n, double *out, hipStream_t s);
// out[P ld + (x / div) n + x % div] += sum over S parts of part[s][P][x], P < M, x < N
hipError_t launch_add_parts(const double *part, int S, int M, int N, double *out, long long ld, int n, int div,
                            hipStream_t s);

}  // namespace pamd
