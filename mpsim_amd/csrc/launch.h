// Host-side launchers shared between the kernel files and the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mpsx.h"

// d: the table on the device, or null: h (at most MPSX_SITE_NOW) goes with the launch.
hipError_t launch_one_site(hipStream_t s, const mpsx_site_op *h, const mpsx_site_op *d, int count,
                           int64_t max_pairs, uint32_t dmask);
hipError_t launch_put(hipStream_t s, void *dst, const void *src, size_t bytes);
hipError_t launch_scale(hipStream_t s, const mpsx_scale_op *d, int count, int64_t max_n);
hipError_t launch_gemm(hipStream_t s, const mpsx_gemm_op *h, const mpsx_gemm_op *d, int count, int64_t max_m,
                       int64_t max_n);
// The tall-narrow variant: every op without conjugation, k <= 32, n <= 256.
bool gemm_rows_fit(const mpsx_gemm_op &o);
hipError_t launch_gemm_rows(hipStream_t s, const mpsx_gemm_op *h, const mpsx_gemm_op *d,
                            int count);

// max_n: rows up to which the Gram problems take the direct eigensolver
// (eig_direct; 0: none do). small: 1 when the one-workgroup kernel takes the
// problems small_route selects; the others of these launches pass them by.
// group: what ProblemCtl.group starts from (0, or EIG_GROUP_LOST).
hipError_t launch_init_rows(hipStream_t s, bool f32, const mpsx_two_site_op *d, int count, char *ws,
                            int64_t rows, int max_n, int small, int group);
hipError_t launch_theta(hipStream_t s, bool f32, int D, const mpsx_two_site_op *d, int count, char *ws,
                        int64_t tiles);
hipError_t launch_theta_gen(hipStream_t s, bool f32, const mpsx_two_site_op *d, int count, char *ws,
                            int64_t tiles);
hipError_t launch_rownorm(hipStream_t s, bool f32, const mpsx_two_site_op *d, int count, char *ws,
                          int64_t rows, int small);
hipError_t launch_fro(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws,
                      double null_rel, int small);
hipError_t launch_owner(hipStream_t s, const mpsx_two_site_op *d, int count, int *owner);
hipError_t launch_jacobi_round(hipStream_t s, bool f32, int b, const mpsx_two_site_op *d, const int *owner,
                               char *ws, int small, int64_t pairs, int round, double tol, double tol_inner,
                               int inner_sweeps);
hipError_t launch_sweep_end(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws,
                            int sweep, bool fp32_phase, int small);
// unconverged, late: mpsx_svd_opts.unconverged and mpsx_two_site_async's word.
hipError_t launch_sort(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws,
                       int *unconverged, int *late, int max_n, int small);
hipError_t launch_gather(hipStream_t s, bool f32, const mpsx_two_site_op *d, int count, char *ws,
                         int64_t outs, int small);
// The one-workgroup kernel (small.hip), from theta to the factors.
hipError_t launch_small(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, double tol, double null_rel,
                        int *unconverged, int *late);
hipError_t launch_hgram(hipStream_t s, const mpsx_two_site_op *d, const int *owner, char *ws,
                        int64_t pairs, int max_nb, int stage, int max_n);
hipError_t launch_hsolve(hipStream_t s, bool f32h, const mpsx_two_site_op *d, const int *owner, char *ws,
                         int max_n, int64_t pairs, int round, double tol, double tol_inner, int inner_sweeps,
                         double abs_rel);
hipError_t launch_hupdate(hipStream_t s, bool f32h, const mpsx_two_site_op *d, const int *owner, char *ws,
                          int max_n, int64_t pairs, int ytiles, int round, int part);
hipError_t launch_hround(hipStream_t s, bool f32h, const mpsx_two_site_op *d, const int *owner, char *ws,
                         int max_n, int64_t pairs, int ytiles, int round, double tol, double tol_inner,
                         int inner_sweeps, double abs_rel);
hipError_t launch_hxcopy(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int64_t rows,
                         int max_n);
hipError_t launch_hxgemm(hipStream_t s, const mpsx_two_site_op *d, const int *owner, char *ws,
                         int64_t pairs, int ctiles, int mode, int max_nb, int max_n);
// QR preconditioning (plan.method 3): column order, X0 save and permute,
// and step `panel` (-1 factors panel 0) over `strips` 16-column strips, for
// the problems of at most 512 rows (`small`) and those above (`large`).
hipError_t launch_qr_order(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_c,
                           int max_r, int max_n);
hipError_t launch_qr_permute(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws,
                             int64_t rows, int max_n);
hipError_t launch_qr_step(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int panel,
                          int strips, int max_c, bool small, bool large, int max_n);
// Direct eigensolver (eig.hip) of the problems eig_direct selects: the
// tridiagonal form (`map`: room for `slots` int2, the workgroups of all their
// groups; `grouped`: some group has more than one; `ticket`: the workgroups take their
// places in the order they start; `no_wait`: a group's waits end at their first look), the eigensystem of T, and Y. n: the largest C among them; `small`,
// `large`: some of at most 512 rows, some above.
hipError_t launch_eig_tridiag(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, void *map, int max_n,
                              int slots, bool grouped, bool ticket, bool no_wait);
// H = X X^H, and at the end X <- Y X (tiles: 32 x 32 ones of the largest X).
hipError_t launch_eig_gram(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n, int n);
hipError_t launch_eig_apply(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n,
                            int64_t tiles);
hipError_t launch_eig_conquer(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n, int n);
hipError_t launch_eig_back(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n, int n,
                           bool small, bool large);
