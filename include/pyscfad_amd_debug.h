/*
 * Inspection entry points of libpyscfad_amd_cc.so, with no counterpart in the
 * reference.  All but the two pamd_debug_one_triple_* run no GPU work: they let
 * tests check, on the CPU, every address the contraction engine will touch
 * before a kernel runs.
 */
#ifndef PYSCFAD_AMD_DEBUG_H
#define PYSCFAD_AMD_DEBUG_H

#include "pyscfad_amd_ccsdt.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Record (do not launch) the contraction descriptors of one occupied triple
 * i <= j <= k: the three W-build GEMMs, plus the adjoint GEMMs when with_vjp.
 * bases[10]: base addresses to put in the descriptors for
 *   Vp, T2m, OOt, W, t2, Vb, Vpb, T2mb, part_p, part_h.
 * out receives min(n, max_desc) descriptors of *desc_bytes bytes each. */
int pamd_debug_gemm_descriptors(int nocc, int nvir, int i, int j, int k, int with_vjp,
                                const unsigned long long *bases, void *out, int max_desc,
                                int *n_desc, int *desc_bytes);

/* Record the adjoint contractions of two consecutive triples (i, j, kp) and
 * (i, j, k), kp < k, as the two-stream adjoint walk pairs them in the split
 * forms: the first triple's launches without its ovvv and hole-term t2
 * adjoints into index i and j, then the second triple's, those adjoints as
 * four-segment launches that also take the first triple's terms.
 * bases[11]: those of pamd_debug_gemm_descriptors, then the second triple's
 * Wbar (the first triple's Wbar is at bases[3]). */
int pamd_debug_paired_adjoint_descriptors(int nocc, int nvir, int i, int j, int kp, int k,
                                          const unsigned long long *bases, void *out,
                                          int max_desc, int *n_desc, int *desc_bytes);

/* Record the adjoint contractions of the triple (i, j, k), in any order of the
 * occupied indices (the projected walk takes (l, j, k) with j <= k and any l),
 * as the split-BF16x3 walks launch them: descriptors with the same launch[]
 * number run concurrently, in one launch.  bases[10]: those of
 * pamd_debug_gemm_descriptors; out and launch receive min(n, max_desc) entries. */
int pamd_debug_adjoint_launches(int nocc, int nvir, int i, int j, int k, const unsigned long long *bases,
                                void *out, int *launch, int max_desc, int *n_desc, int *desc_bytes);

/* 1 when a recorded descriptor (one of pamd_debug_gemm_descriptors' outputs)
 * runs on the FP64 engine's direct-to-LDS path (16-byte element pairs: fast
 * strides 1, other strides and index divisors even, 16-byte aligned bases),
 * 0 when it runs on the register-staged path. */
int pamd_debug_gemm_direct_ok(const void *desc);

/* 1 when a recorded descriptor, moved onto planar split-BF16x3 operands (each
 * FP64 element address 8 e becomes the bf16 address 2 e, bases being multiples
 * of 64 bytes, with plane stride plane_stride), runs on the split-BF16x3
 * engine's direct-to-LDS path (16-byte runs of 8 bf16: fast strides 1, other
 * strides, divisors, segment lengths or row counts multiples of 8), 0 when it
 * runs on the register-staged path. */
int pamd_debug_gemm_b3p_ok(const void *desc, long long plane_stride);

/* Split-K factors the adjoint uses for (particle, hole) partial buffers. */
int pamd_debug_split_factors(int nocc, int nvir, int *S_p, int *S_h);

/* The same for a given precision (PAMD_PREC_*): the split-BF16x3 engine sizes
 * its split-K for its own tile shapes and bounds the K range of one part. */
int pamd_debug_split_factors_prec(int nocc, int nvir, int precision, int *S_p, int *S_h);

/* Triples per batch that an FP64 call (nfrag = 0), or a projected one (nfrag > 0),
 * works on with a workspace of workspace_bytes; 0: one triple at a time. */
int pamd_debug_walk_batch(int nocc, int nvir, int nfrag, int with_vjp, size_t workspace_bytes, int *triples);
/* Bytes of that workspace which such a call uses (its batched walk; 0: none). */
int pamd_debug_walk_bytes(int nocc, int nvir, int nfrag, int with_vjp, size_t workspace_bytes, size_t *bytes);

/* pamd_ccsdt_energy_vjp and pamd_ccsdt_projected_energy_vjp, one triple at a time
 * whatever the workspace holds: what an FP64 call does when it holds no batch, for
 * tests that compare the walks.  two_streams: with the epilogue on the library's
 * side stream (needs pamd_ccsdt_workspace_size bytes), or on the call's alone. */
int pamd_debug_one_triple_vjp(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                              const double *t2, const double *ovvv, const double *ovoo, const double *ovov,
                              const double *fvo, double et_bar, int two_streams, void *workspace,
                              size_t workspace_bytes, double *e_out, double *mo_energy_bar, double *t1_bar,
                              double *t2_bar, double *ovvv_bar, double *ovoo_bar, double *ovov_bar,
                              double *fvo_bar, void *stream);
int pamd_debug_one_triple_projected_vjp(const pamd_ccsdt_config *cfg, const double *mo_energy, const double *t1,
                                        const double *t2, const double *ovvv, const double *ovoo,
                                        const double *ovov, const double *fvo, const double *ulo, int nfrag,
                                        double et_bar, void *workspace, size_t workspace_bytes, double *e_out,
                                        double *mo_energy_bar, double *t1_bar, double *t2_bar, double *ovvv_bar,
                                        double *ovoo_bar, double *ovov_bar, double *fvo_bar, double *ulo_bar,
                                        void *stream);

#ifdef __cplusplus
}
#endif
#endif
