/* rbh_testing.h - entry points of librbh.so for tests only.
 *
 * No counterpart in the reference.  They run one internal stage of the step
 * on caller data, or one of its launch rules, so that a test can check its
 * edge cases directly (sizes the step rarely produces).  They allocate device memory per call and
 * are not meant for production paths.
 */
#ifndef RBH_TESTING_H
#define RBH_TESTING_H

#include "rbh.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The step's device-wide exclusive prefix sum, on a host array: out[i] =
 * in[0] + ... + in[i-1] for i = 0..n (out holds n + 1 ints) and *total =
 * out[n].  in holds n elements of elem_bytes = 1 (unsigned char) or 4 (int).
 * cap (n <= cap <= 2^28) is the capacity the launch is sized for, as in the
 * step: the grid covers cap, and the live length n is read on the device.
 * Below 32768 the scan is one workgroup; from there on it is the single-pass
 * look-back scan (a wait for a predecessor that times out returns RBH_E_HIP). */
int rbh_prefix_sum(rbh_ctx* ctx, const void* in, int elem_bytes, int n, int cap, int* out, int* total);

/* The ellipsoid projection of the contact sweeps (anisotropic friction) in
 * FP64, on n independent inputs: z (3n) projected onto the ellipsoid of axes
 * mu (3n) times xn (n), with rbh_params' ellipsoid_tolerance,
 * ellipsoid_expansion and ellipsoid_max_iterations; out (3n). */
int rbh_prox_ellipsoid(rbh_ctx* ctx, int n, const double* z, const double* mu, const double* xn, double tolerance,
                       double expansion, int max_iterations, double* out);

/* Whether rbh_sdf_build takes its pruned form for these arguments: 1 or 0 (no
 * device needed). */
int rbh_sdf_is_pruned(const double* V, int nv, const int* T, int nt, const double* min_coord, const double* max_coord,
                      int I, int J, int K);

/* Pinned host memory the context holds for its transfers. */
int rbh_transfer_buffer(rbh_ctx* ctx, unsigned long long* bytes);

/* Workgroups of a lone scene's solve (no device needed): `units` colouring
 * units in the last step seen (0: none), rbh_tuning's lanes_per_group, and the
 * most workgroups that are resident at once. */
int rbh_coop_grid(int units, int lanes_per_group, int most);

/* The same for a scene of `bodies` bodies; units is 0 for a last step without
 * contacts, negative if no step was seen. */
int rbh_lone_grid(int units, int bodies, int lanes_per_group, int most);

/* How the hinge solve of a batch would be launched (no device needed): n
 * hinged scenes of bodies[i] bodies in hinges[i] hinges on `cus` compute units.
 * *staged: 1 if their rows are staged in LDS; *lds: bytes of a workgroup;
 * rows_at (n): where a scene's staged rows start. */
int rbh_hinge_launch(int precision_bytes, int cus, int n, const int* bodies, const int* hinges, int* staged,
                     long long* lds, int* rows_at);
/* Workgroups (of one wavefront) of the hinge solve that share a compute unit
 * at `lds` bytes each. */
int rbh_hinge_occupancy(rbh_ctx* ctx, int staged, long long lds, int* groups_per_cu);

#ifdef __cplusplus
}
#endif
#endif
