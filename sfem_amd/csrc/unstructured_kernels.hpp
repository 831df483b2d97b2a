// Host-callable launchers of the tet4/hex8 kernels (unstructured_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace sfem_amd {
int tet4_laplacian_apply(ptrdiff_t E, const int32_t *idx, const float *fff, const double *x, double *y,
                         hipStream_t s);
int tet4_laplacian_diag(ptrdiff_t E, const int32_t *idx, const float *fff, double *d, hipStream_t s);
int hex8_laplacian_apply(ptrdiff_t E, const int32_t *idx, const float *fff, const float *coeff, const double *x,
                         double *y, hipStream_t s);
int hex8_laplacian_diag(ptrdiff_t E, const int32_t *idx, const float *fff, const float *coeff, double *d,
                        hipStream_t s);
// T = double with float32 geometry words G, or T = float with bf16 words (uint16_t); coeff (nullable)
// scales mu and lambda per element; block: the symmetric 3x3 block diagonal [node][6] instead of the
// diagonal
template <typename T, typename G>
int hex8_elasticity_apply(ptrdiff_t E, const int32_t *idx, const G *adj, const G *det, double mu, double lambda,
                          const float *coeff, const T *x, T *y, hipStream_t s);
// Element patches (ElementPatches): elements of a full patch, and the patch kernels'
// LDS (x and y of every patch node) limit
constexpr int kPatchElements = 512;
constexpr size_t kPatchLdsLimit = 64 * 1024;
inline size_t patch_lds_bytes(int maxloc, int vs, size_t value_bytes) {
    return (size_t)vs * maxloc * (value_bytes + sizeof(double));  // x in the value type, y accumulated in FP64
}
struct PatchView {
    ptrdiff_t npatch{0}, E{0};
    int maxloc{0};
    const int32_t *start{nullptr}, *node_off{nullptr}, *nodes{nullptr};
    const uint16_t *lconn{nullptr};
};
// The Laplacian over the patches (nv 4: tet4, 8: hex8; fffp [6][E], coeffp [E] or null in patch-slot
// order), as hex8_elasticity_apply_patches below.
int laplacian_apply_patches(int nv, const PatchView &pv, const float *fffp, const float *coeffp, const double *x,
                            double *y, hipStream_t s);
// y += A x over the patches.  adjp [9][E], detp and coeffp [E] in patch-slot order (patch_gather_rows).
template <typename T, typename G>
int hex8_elasticity_apply_patches(const PatchView &pv, const G *adjp, const G *detp, const float *coeffp, double mu,
                                  double lambda, const T *x, T *y, hipStream_t s);
// out[k][s] = in[k][perm[s]] for k < rows, s < E
template <typename G>
int patch_gather_rows(int rows, ptrdiff_t E, const int32_t *perm, const G *in, G *out, hipStream_t s);
// hex8 applies node by node (small meshes): y = A x over all N nodes, off/ent the corners by node
// (NodeElements); mask (nullable, bit per component of each node): y = x there instead
int hex8_laplacian_apply_nodes(ptrdiff_t N, ptrdiff_t E, const int32_t *off, const int32_t *ent, const int32_t *idx,
                               const float *fff, const float *coeff, const double *x, double *y, const uint8_t *mask,
                               hipStream_t s);
template <typename T, typename G>
int hex8_elasticity_apply_nodes(ptrdiff_t N, ptrdiff_t E, const int32_t *off, const int32_t *ent, const int32_t *idx,
                                const G *adj, const G *det, double mu, double lambda, const float *coeff, const T *x,
                                T *y, const uint8_t *mask, hipStream_t s);
template <typename T, typename G>
int hex8_elasticity_diag(ptrdiff_t E, const int32_t *idx, const G *adj, const G *det, double mu, double lambda,
                         const float *coeff, int block, T *d, hipStream_t s);
}  // namespace sfem_amd
