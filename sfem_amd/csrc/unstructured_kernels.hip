// gfx950 kernels for tet4 and hex8 meshes: one element per lane, or a patch of elements per workgroup.
//
// Device layout: idx int32 SoA [nv][E] and geometry SoA [k][E] (the layout of the
// reference's device path, operators/cuda/cu_laplacian.hpp fff_stride), so a wave
// reads 64 consecutive words of every row: fully coalesced.  Scatter with FP64
// atomics, as cu_tet4_laplacian_apply_kernel (operators/tet4/cuda/cu_tet4_laplacian.cu:11-44).
#include <type_traits>

#include "common.hpp"
#include "unstructured_kernels.hpp"

namespace sfem_amd {

// ------------------------------------------------------------------ tet4 Laplacian
// e = K u with K from FFF (operators/tet4/tet4_laplacian_inline_cpu.hpp:54-73):
// grad u = (u1-u0, u2-u0, u3-u0) on the reference tet, t = FFF grad u,
// e1..3 = t, e0 = -(t0+t1+t2).
__global__ void tet4_laplacian_apply_kernel(const ptrdiff_t E, const int32_t *__restrict__ idx,
                                            const float *__restrict__ fff, const double *__restrict__ x,
                                            double *__restrict__ y) {
    for (ptrdiff_t e = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; e < E;
         e += (ptrdiff_t)gridDim.x * blockDim.x) {
        int32_t v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = idx[k * E + e];
        double f[6];
#pragma unroll
        for (int k = 0; k < 6; k++) f[k] = (double)fff[k * E + e];
        const double u0 = x[v[0]];
        const double g0 = x[v[1]] - u0, g1 = x[v[2]] - u0, g2 = x[v[3]] - u0;
        const double t0 = f[0] * g0 + f[1] * g1 + f[2] * g2;
        const double t1 = f[1] * g0 + f[3] * g1 + f[4] * g2;
        const double t2 = f[2] * g0 + f[4] * g1 + f[5] * g2;
        atomicAdd(&y[v[0]], -(t0 + t1 + t2));
        atomicAdd(&y[v[1]], t0);
        atomicAdd(&y[v[2]], t1);
        atomicAdd(&y[v[3]], t2);
    }
}

__global__ void tet4_laplacian_diag_kernel(const ptrdiff_t E, const int32_t *__restrict__ idx,
                                           const float *__restrict__ fff, double *__restrict__ d) {
    for (ptrdiff_t e = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; e < E;
         e += (ptrdiff_t)gridDim.x * blockDim.x) {
        double f[6];
#pragma unroll
        for (int k = 0; k < 6; k++) f[k] = (double)fff[k * E + e];
        // tet4_laplacian_diag_fff (operators/tet4/tet4_laplacian_inline_cpu.hpp:32-41)
        atomicAdd(&d[idx[0 * E + e]], f[0] + 2 * f[1] + 2 * f[2] + f[3] + 2 * f[4] + f[5]);
        atomicAdd(&d[idx[1 * E + e]], f[0]);
        atomicAdd(&d[idx[2 * E + e]], f[3]);
        atomicAdd(&d[idx[3 * E + e]], f[5]);
    }
}

// ------------------------------------------------------------------ hex8 Laplacian
// Exact Q1 integral with constant FFF by 2-point Gauss (the integrand is at most
// quadratic per direction): y_i = sum_q w_q grad phi_i(q) . G grad u(q).
__device__ __forceinline__ void q1_ref_grad(int n, double qx, double qy, double qz, double *g) {
    const int bx = hex8_cx(n), by = hex8_cy(n), bz = hex8_cz(n);
    const double fx = bx ? qx : 1 - qx, fy = by ? qy : 1 - qy, fz = bz ? qz : 1 - qz;
    const double sx = bx ? 1 : -1, sy = by ? 1 : -1, sz = bz ? 1 : -1;
    g[0] = sx * fy * fz;
    g[1] = fx * sy * fz;
    g[2] = fx * fy * sz;
}

__global__ void hex8_laplacian_apply_kernel(const ptrdiff_t E, const int32_t *__restrict__ idx,
                                            const float *__restrict__ fff, const float *__restrict__ coeff,
                                            const double *__restrict__ x, double *__restrict__ y) {
    const double gp[2] = {0.5 - 0.28867513459481288225, 0.5 + 0.28867513459481288225};
    for (ptrdiff_t e = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; e < E;
         e += (ptrdiff_t)gridDim.x * blockDim.x) {
        int32_t v[8];
        double u[8], out[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            v[k] = idx[k * E + e];
            u[k] = x[v[k]];
            out[k] = 0;
        }
        const double c = (coeff ? (double)coeff[e] : 1.0) * 0.125;
        double f[6];
#pragma unroll
        for (int k = 0; k < 6; k++) f[k] = (double)fff[k * E + e] * c;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const double qx = gp[q & 1], qy = gp[(q >> 1) & 1], qz = gp[q >> 2];
            double gu[3] = {0, 0, 0};
#pragma unroll
            for (int n = 0; n < 8; n++) {
                double g[3];
                q1_ref_grad(n, qx, qy, qz, g);
                gu[0] += g[0] * u[n];
                gu[1] += g[1] * u[n];
                gu[2] += g[2] * u[n];
            }
            const double t0 = f[0] * gu[0] + f[1] * gu[1] + f[2] * gu[2];
            const double t1 = f[1] * gu[0] + f[3] * gu[1] + f[4] * gu[2];
            const double t2 = f[2] * gu[0] + f[4] * gu[1] + f[5] * gu[2];
#pragma unroll
            for (int n = 0; n < 8; n++) {
                double g[3];
                q1_ref_grad(n, qx, qy, qz, g);
                out[n] += g[0] * t0 + g[1] * t1 + g[2] * t2;
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++) atomicAdd(&y[v[k]], out[k]);
    }
}

__global__ void hex8_laplacian_diag_kernel(const ptrdiff_t E, const int32_t *__restrict__ idx,
                                           const float *__restrict__ fff, const float *__restrict__ coeff,
                                           double *__restrict__ d) {
    for (ptrdiff_t e = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; e < E;
         e += (ptrdiff_t)gridDim.x * blockDim.x) {
        const double c = coeff ? (double)coeff[e] : 1.0;
        double f[6];
#pragma unroll
        for (int k = 0; k < 6; k++) f[k] = (double)fff[k * E + e] * c;
#pragma unroll
        for (int k = 0; k < 8; k++) atomicAdd(&d[idx[k * E + e]], hex8_laplacian_entry(f, k, k));
    }
}

// ------------------------------------------------------------------ hex8 elasticity
// Affine Q1 elasticity from the centre adjugate and determinant
// (operators/hex8/hex8_linear_elasticity.cpp:625-760), 2x2x2 Gauss (exact for a constant Jacobian):
// grad u = (sum_n u_n ghat_n) P^T with P = J^-T = adj^T/det; sigma = lambda tr(eps) I + 2 mu eps;
// y_n += w det sigma P ghat_n.  x, y interleaved xyz.
//
// Sum-factorised, one element per lane.  With the corners as a 2x2x2 tensor u[iz][iy][ix] and the
// 1-D Gauss points g_0, g_1, the reference derivative along x at point (qz, qy, qx) is the bilinear
// interpolation in (z, y) of the four x-differences u[iz][iy][1] - u[iz][iy][0], the same for both
// qx: each of the 9 (component, direction) gradients has 4 distinct values over the 8 points
// (16 operations each instead of 64).  The transpose runs the same steps backwards: the point
// values of each (component, direction) are first summed over the direction's own index, then
// spread bilinearly and differenced onto the corners.  About 1,000 operations per element against
// 3,700 for the plain point loop; T is the value type (double, or float for the FP32 operator with
// bf16 geometry words G).
template <typename T>
__device__ __forceinline__ void sf_interp2(const T a00, const T a01, const T a10, const T a11, const T g0, const T g1,
                                           T out[2][2]) {
    // out[q1][q2] = sum_ij B[q1][i] B[q2][j] a_ij with B[q][0] = 1 - g_q, B[q][1] = g_q
    const T r00 = a00 + g0 * (a01 - a00), r01 = a00 + g1 * (a01 - a00);
    const T r10 = a10 + g0 * (a11 - a10), r11 = a10 + g1 * (a11 - a10);
    out[0][0] = r00 + g0 * (r10 - r00);
    out[1][0] = r00 + g1 * (r10 - r00);
    out[0][1] = r01 + g0 * (r11 - r01);
    out[1][1] = r01 + g1 * (r11 - r01);
}
template <typename T>
__device__ __forceinline__ void sf_interp2_t(const T r[2][2], const T g0, const T g1, T &a00, T &a01, T &a10,
                                             T &a11) {
    // transpose of sf_interp2: a_ij = sum_{q1 q2} B[q1][i] B[q2][j] r[q1][q2]; first over q2:
    // H[q1][1] = sum_q2 g_q2 r[q1][q2], H[q1][0] = sum_q2 r[q1][q2] - H[q1][1]
    const T h01 = g0 * r[0][0] + g1 * r[0][1], h00 = (r[0][0] + r[0][1]) - h01;
    const T h11 = g0 * r[1][0] + g1 * r[1][1], h10 = (r[1][0] + r[1][1]) - h11;
    // then over q1 the same way
    a10 = g0 * h00 + g1 * h10;
    a11 = g0 * h01 + g1 * h11;
    a00 = (h00 + h10) - a10;
    a01 = (h01 + h11) - a11;
}

// One element: corner values load(n, d) (hex8 corner n, component d) in, store(n, d, v) of the 24
// products out; a64/det: the element's adjugate and determinant, c its coefficient.
template <typename T, typename Load, typename Store>
__device__ __forceinline__ void hex8_elasticity_sf_element(const double a64[9], const double det, const double c,
                                                           const double mu0, const double lambda0, Load load,
                                                           Store store) {
    // hex8 corner n -> tensor position iz*4 + iy*2 + ix
    constexpr int kT[8] = {0, 1, 3, 2, 4, 5, 7, 6};
    const T g0 = (T)(0.5 - 0.28867513459481288225), g1 = (T)(0.5 + 0.28867513459481288225);
    // P[a][k] = adj[a][k] / det for the physical gradient; the weight det/8 and the 1/det of the way
    // back leave adj/8 on the stress side, folded into mu and lambda
    const double idet = 1.0 / det;
    T P[9], A[9];
#pragma unroll
    for (int k = 0; k < 9; k++) {
        P[k] = (T)(a64[k] * idet);
        A[k] = (T)a64[k];
    }
    const T mu = (T)(mu0 * c * 0.125), lambda = (T)(lambda0 * c * 0.125);
    // gx[c][qz][qy], gy[c][qz][qx], gz[c][qy][qx]
    T gx[3][2][2], gy[3][2][2], gz[3][2][2];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        T u[8];
#pragma unroll
        for (int n = 0; n < 8; n++) u[kT[n]] = load(n, d);
        // x-differences at (iz, iy), interpolated in (z, y)
        sf_interp2<T>(u[1] - u[0], u[3] - u[2], u[5] - u[4], u[7] - u[6], g0, g1, gx[d]);
        // y-differences at (iz, ix), interpolated in (z, x)
        sf_interp2<T>(u[2] - u[0], u[3] - u[1], u[6] - u[4], u[7] - u[5], g0, g1, gy[d]);
        // z-differences at (iy, ix), interpolated in (y, x)
        sf_interp2<T>(u[4] - u[0], u[5] - u[1], u[6] - u[2], u[7] - u[3], g0, g1, gz[d]);
    }
    // point values of R[d][a] = sum_k S[d][k] adj[a][k], summed over the direction's own index
    T rx[3][2][2], ry[3][2][2], rz[3][2][2];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) rx[d][i][j] = ry[d][i][j] = rz[d][i][j] = 0;
#pragma unroll
    for (int qz = 0; qz < 2; qz++)
#pragma unroll
        for (int qy = 0; qy < 2; qy++)
#pragma unroll
            for (int qx = 0; qx < 2; qx++) {
                T F[3][3];
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const T h0 = gx[d][qz][qy], h1 = gy[d][qz][qx], h2 = gz[d][qy][qx];
#pragma unroll
                    for (int k = 0; k < 3; k++) F[d][k] = h0 * P[0 * 3 + k] + h1 * P[1 * 3 + k] + h2 * P[2 * 3 + k];
                }
                const T ltr = lambda * (F[0][0] + F[1][1] + F[2][2]);
                T S[3][3];
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    S[d][d] = 2 * mu * F[d][d] + ltr;
#pragma unroll
                    for (int k = d + 1; k < 3; k++) S[d][k] = S[k][d] = mu * (F[d][k] + F[k][d]);
                }
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    rx[d][qz][qy] += S[d][0] * A[0] + S[d][1] * A[1] + S[d][2] * A[2];
                    ry[d][qz][qx] += S[d][0] * A[3] + S[d][1] * A[4] + S[d][2] * A[5];
                    rz[d][qy][qx] += S[d][0] * A[6] + S[d][1] * A[7] + S[d][2] * A[8];
                }
            }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        T o[8];
        T a00, a01, a10, a11;
        sf_interp2_t<T>(rx[d], g0, g1, a00, a01, a10, a11);  // at (iz, iy): +x corner gets +, -x gets -
        o[1] = a00, o[0] = -a00, o[3] = a01, o[2] = -a01, o[5] = a10, o[4] = -a10, o[7] = a11, o[6] = -a11;
        sf_interp2_t<T>(ry[d], g0, g1, a00, a01, a10, a11);  // at (iz, ix)
        o[2] += a00, o[0] -= a00, o[3] += a01, o[1] -= a01, o[6] += a10, o[4] -= a10, o[7] += a11, o[5] -= a11;
        sf_interp2_t<T>(rz[d], g0, g1, a00, a01, a10, a11);  // at (iy, ix)
        o[4] += a00, o[0] -= a00, o[5] += a01, o[1] -= a01, o[6] += a10, o[2] -= a10, o[7] += a11, o[3] -= a11;
#pragma unroll
        for (int n = 0; n < 8; n++) store(n, d, o[kT[n]]);
    }
}

// Element-wise: one element per lane, products added to y with atomics.
template <typename T, typename G>
__global__ void __launch_bounds__(256)
    hex8_elasticity_apply_sf_kernel(const ptrdiff_t E, const int32_t *__restrict__ idx, const G *__restrict__ adjg,
                                    const G *__restrict__ detg, const double mu0, const double lambda0,
                                    const float *__restrict__ coeff, const T *__restrict__ x, T *__restrict__ y) {
    for (ptrdiff_t e = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; e < E;
         e += (ptrdiff_t)gridDim.x * blockDim.x) {
        int32_t v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = idx[k * E + e];
        double a64[9];
#pragma unroll
        for (int k = 0; k < 9; k++) a64[k] = load_geom<G>(adjg, k * E + e);
        hex8_elasticity_sf_element<T>(
            a64, load_geom<G>(detg, e), coeff ? (double)coeff[e] : 1.0, mu0, lambda0,
            [&](int n, int d) { return x[(ptrdiff_t)v[n] * 3 + d]; },
            [&](int n, int d, T val) { atomicAdd(&y[(ptrdiff_t)v[n] * 3 + d], val); });
    }
}

// Patch-wise (ElementPatches): one workgroup per patch.  The patch's nodes
// are gathered into LDS once (x), the elements accumulate into LDS (y, LDS atomics), then every patch
// node is added to y with a global atomic, consecutive lanes on consecutive entries of y: nodes that
// several patches share need no further pass.  (Shared nodes written to partials instead, summed by a
// gather kernel, the others added without atomics, a pass with its zero fill on one mesh: 72 against 52 us at 1.93M
// hexahedra, Laplacian; 175 against 131 us at 2.10M, FP64 elasticity (FP32 101 against 87), where a lane per node with
// its three components apart takes 244 us.  Three meshes in turn, which leave nothing in the caches: 56 and 154 us.)  It also lets several streams apply one operator, or add into one y.  The
// geometry and coefficient words are stored in patch-slot order, so every read of them coalesces.
// The LDS accumulator is FP64 for both value types: ds_add_f64 keeps pace with the arithmetic, while
// ds_add_f32 measured 7x the LDS busy cycles and 100x the LDS wait of the whole FP64 kernel here.

// patch nodes per thread at a time: their ids, then their values, each batch issued together (an entry per
// thread as in patch_add_y: 155 us an elasticity apply)
constexpr int kPatchBatch = 4;
template <typename T, int VS>
__device__ __forceinline__ void patch_gather_x(const int nloc, const int32_t *__restrict__ nodes,
                                               const T *__restrict__ x, T *__restrict__ sx, double *__restrict__ sy) {
    for (int i0 = threadIdx.x; i0 < nloc; i0 += kPatchBatch * blockDim.x) {
        ptrdiff_t gg[kPatchBatch];
#pragma unroll
        for (int b = 0; b < kPatchBatch; b++) {
            const int i = i0 + b * blockDim.x;
            gg[b] = nodes[i < nloc ? i : 0];
        }
        T xv[kPatchBatch][VS];
#pragma unroll
        for (int b = 0; b < kPatchBatch; b++)
#pragma unroll
            for (int c = 0; c < VS; c++) xv[b][c] = x[gg[b] * VS + c];
#pragma unroll
        for (int b = 0; b < kPatchBatch; b++) {
            const int i = i0 + b * blockDim.x;
            if (i < nloc)
#pragma unroll
                for (int c = 0; c < VS; c++) {
                    sx[i * VS + c] = xv[b][c];
                    sy[i * VS + c] = 0;
                }
        }
    }
}
// entries (node, component) per thread at a time
template <typename T, int VS>
__device__ __forceinline__ void patch_add_y(const int nloc, const int32_t *__restrict__ nodes,
                                            const double *__restrict__ sy, T *__restrict__ y) {
    const int n = nloc * VS;
    for (int i0 = threadIdx.x; i0 < n; i0 += kPatchBatch * blockDim.x) {
        ptrdiff_t gg[kPatchBatch];
#pragma unroll
        for (int b = 0; b < kPatchBatch; b++) {
            const int i = i0 + b * blockDim.x < n ? i0 + b * blockDim.x : 0, node = i / VS;
            gg[b] = (ptrdiff_t)nodes[node] * VS + (i - node * VS);
        }
#pragma unroll
        for (int b = 0; b < kPatchBatch; b++) {
            const int i = i0 + b * blockDim.x;
            if (i < n) atomicAdd(&y[gg[b]], (T)sy[i]);
        }
    }
}
// the local nodes of a slot's NV corners, four 16-bit ids to a word pair
template <int NV>
__device__ __forceinline__ void patch_local_nodes(const uint16_t *__restrict__ lconn, ptrdiff_t E, ptrdiff_t slot,
                                                  int (&l)[NV]) {
#pragma unroll
    for (int q = 0; q < NV / 4; q++) {
        const ushort4 w = reinterpret_cast<const ushort4 *>(lconn)[q * E + slot];
        l[4 * q] = w.x, l[4 * q + 1] = w.y, l[4 * q + 2] = w.z, l[4 * q + 3] = w.w;
    }
}

template <typename T, typename G>
__global__ void __launch_bounds__(256)
    hex8_elasticity_patch_kernel(const PatchView pv, const G *__restrict__ adjp, const G *__restrict__ detp,
                                 const float *__restrict__ coeffp, const double mu0, const double lambda0,
                                 const T *__restrict__ x, T *__restrict__ y) {
    extern __shared__ __align__(16) unsigned char patch_lds[];
    const ptrdiff_t p = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int off = pv.node_off[p], nloc = pv.node_off[p + 1] - off;
    double *sy = reinterpret_cast<double *>(patch_lds);
    T *sx = reinterpret_cast<T *>(sy + 3 * nloc);
    patch_gather_x<T, 3>(nloc, pv.nodes + off, x, sx, sy);
    __syncthreads();
    const int first = pv.start[p], cnt = pv.start[p + 1] - first;
    for (int t = threadIdx.x; t < cnt; t += blockDim.x) {
        const ptrdiff_t slot = first + t;
        int l[8];
        patch_local_nodes<8>(pv.lconn, pv.E, slot, l);
        double a64[9];
#pragma unroll
        for (int k = 0; k < 9; k++) a64[k] = load_geom<G>(adjp, k * pv.E + slot);
        hex8_elasticity_sf_element<T>(
            a64, load_geom<G>(detp, slot), coeffp ? (double)coeffp[slot] : 1.0, mu0, lambda0,
            [&](int n, int d) { return sx[l[n] * 3 + d]; },
            [&](int n, int d, T val) { atomicAdd(&sy[l[n] * 3 + d], (double)val); });
    }
    __syncthreads();
    patch_add_y<T, 3>(nloc, pv.nodes + off, sy, y);
}

// hex8 Laplacian of one element, sum-factorised as the elasticity element above.  The x-derivative at
// point (qz, qy, qx) does not depend on qx, so the sums over a direction's own index that the
// transpose needs act on the derivatives directly: rx = sum_qx t_x = 2 f0 gx + f1 sum_qx gy + f2 sum_qx gz.
// About 150 operations per element against 600 for the point loop.  f: FFF times coefficient / 8.
template <typename Load, typename Store>
__device__ __forceinline__ void hex8_laplacian_sf_element(const double f[6], Load load, Store store) {
    constexpr int kT[8] = {0, 1, 3, 2, 4, 5, 7, 6};  // hex8 corner n -> iz*4 + iy*2 + ix
    const double g0 = 0.5 - 0.28867513459481288225, g1 = 0.5 + 0.28867513459481288225;
    double u[8];
#pragma unroll
    for (int n = 0; n < 8; n++) u[kT[n]] = load(n);
    double gx[2][2], gy[2][2], gz[2][2];  // [qz][qy], [qz][qx], [qy][qx]
    sf_interp2<double>(u[1] - u[0], u[3] - u[2], u[5] - u[4], u[7] - u[6], g0, g1, gx);
    sf_interp2<double>(u[2] - u[0], u[3] - u[1], u[6] - u[4], u[7] - u[5], g0, g1, gy);
    sf_interp2<double>(u[4] - u[0], u[5] - u[1], u[6] - u[2], u[7] - u[3], g0, g1, gz);
    double rx[2][2], ry[2][2], rz[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            // (i, j) = (qz, qy), (qz, qx), (qy, qx)
            rx[i][j] = 2 * f[0] * gx[i][j] + f[1] * (gy[i][0] + gy[i][1]) + f[2] * (gz[j][0] + gz[j][1]);
            ry[i][j] = 2 * f[3] * gy[i][j] + f[1] * (gx[i][0] + gx[i][1]) + f[4] * (gz[0][j] + gz[1][j]);
            rz[i][j] = 2 * f[5] * gz[i][j] + f[2] * (gx[0][i] + gx[1][i]) + f[4] * (gy[0][j] + gy[1][j]);
        }
    double o[8], a00, a01, a10, a11;
    sf_interp2_t<double>(rx, g0, g1, a00, a01, a10, a11);  // at (iz, iy): +x corner gets +, -x gets -
    o[1] = a00, o[0] = -a00, o[3] = a01, o[2] = -a01, o[5] = a10, o[4] = -a10, o[7] = a11, o[6] = -a11;
    sf_interp2_t<double>(ry, g0, g1, a00, a01, a10, a11);  // at (iz, ix)
    o[2] += a00, o[0] -= a00, o[3] += a01, o[1] -= a01, o[6] += a10, o[4] -= a10, o[7] += a11, o[5] -= a11;
    sf_interp2_t<double>(rz, g0, g1, a00, a01, a10, a11);  // at (iy, ix)
    o[4] += a00, o[0] -= a00, o[5] += a01, o[1] -= a01, o[6] += a10, o[2] -= a10, o[7] += a11, o[3] -= a11;
#pragma unroll
    for (int n = 0; n < 8; n++) store(n, o[kT[n]]);
}

// The Laplacian over patches.  The element-wise kernels are bound by their global FP64 atomics (4 or 8
// per element), scattered meshes also by the gathers of x; here both stay in LDS.  What bounds this one:
// latency (two dependent loads before the sweep, one after it) and the ds_add_f64 of the sweep.
// 1.93M hexahedra: 47 us (696 us element-wise); 2.41M shuffled tetrahedra: 41 us (417 us).
template <int NV>
__global__ void __launch_bounds__(256)
    laplacian_patch_kernel(const PatchView pv, const float *__restrict__ fffp, const float *__restrict__ coeffp,
                           const double *__restrict__ x, double *__restrict__ y) {
    extern __shared__ __align__(16) unsigned char patch_lds[];
    const ptrdiff_t p = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int off = pv.node_off[p], nloc = pv.node_off[p + 1] - off;
    const int first = pv.start[p], cnt = pv.start[p + 1] - first;
    double *sy = reinterpret_cast<double *>(patch_lds), *sx = sy + nloc;
    // a thread's elements two at a time, the first two loaded before the gather (absent ones re-read the
    // patch's first slot and are not added)
    constexpr int EB = 2;
    int l[EB][NV];
    float w[EB][6], c[EB];
    auto load = [&](int t0) {
#pragma unroll
        for (int b = 0; b < EB; b++) {
            const int t = t0 + b * 256 < cnt ? t0 + b * 256 : 0;
            const ptrdiff_t slot = first + t;
            patch_local_nodes<NV>(pv.lconn, pv.E, slot, l[b]);
#pragma unroll
            for (int k = 0; k < 6; k++) w[b][k] = fffp[k * pv.E + slot];
            c[b] = coeffp ? coeffp[slot] : 1.f;
        }
    };
    load(threadIdx.x);
    patch_gather_x<double, 1>(nloc, pv.nodes + off, x, sx, sy);
    __syncthreads();
    for (int t0 = threadIdx.x; t0 < cnt; t0 += EB * 256) {
        if (t0 != (int)threadIdx.x) load(t0);
#pragma unroll
        for (int b = 0; b < EB; b++) {
            if (t0 + b * 256 >= cnt) continue;
            double f[6];
            if constexpr (NV == 8) {
#pragma unroll
                for (int k = 0; k < 6; k++) f[k] = (double)w[b][k] * ((double)c[b] * 0.125);
                hex8_laplacian_sf_element(
                    f, [&](int n) { return sx[l[b][n]]; }, [&](int n, double v) { atomicAdd(&sy[l[b][n]], v); });
            } else {
#pragma unroll
                for (int k = 0; k < 6; k++) f[k] = (double)w[b][k];
                const double u0 = sx[l[b][0]];
                const double h0 = sx[l[b][1]] - u0, h1 = sx[l[b][2]] - u0, h2 = sx[l[b][3]] - u0;
                const double t1 = f[0] * h0 + f[1] * h1 + f[2] * h2;
                const double t2 = f[1] * h0 + f[3] * h1 + f[4] * h2;
                const double t3 = f[2] * h0 + f[4] * h1 + f[5] * h2;
                atomicAdd(&sy[l[b][0]], -(t1 + t2 + t3));
                atomicAdd(&sy[l[b][1]], t1);
                atomicAdd(&sy[l[b][2]], t2);
                atomicAdd(&sy[l[b][3]], t3);
            }
        }
    }
    __syncthreads();
    patch_add_y<double, 1>(nloc, pv.nodes + off, sy, y);
}

// Node by node, for the small hex8 meshes inside a multigrid hierarchy (below kPatchMinElements), whose
// applies are all latency: eight lanes per node, one per element around it (more in turn), each evaluates its
// element and keeps the row of its own corner; a butterfly adds the eight.  Every node is written once: one launch
// without atomics (the element-wise form needs a zero fill before and a copy of the constrained rows after it),
// and the results are bitwise reproducible.  An element is evaluated eight times over; what bounds it is four dependent loads (range, corner, ids, values).
// Overwriting and constrained: FP32 elasticity, 512 elements, 19.5 (12.6 + fill 2.8 + copy 4.1) -> 6.7 us; FP64
// Laplacian, 4,096 elements, 12.8 -> 4.5 us.  Not used from kPatchMinElements on, where arithmetic counts.
template <int BS, typename T, typename Element>
__device__ __forceinline__ void hex8_node_apply(const ptrdiff_t N, const int32_t *__restrict__ off,
                                                const int32_t *__restrict__ ent, const T *__restrict__ x,
                                                T *__restrict__ y,
                                                const uint8_t *__restrict__ mask, Element element) {
    // every lane of a group of eight takes part in the butterfly, also past the last node
    const int lane = threadIdx.x & 7;
    for (ptrdiff_t t = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; t - lane < N * 8;
         t += (ptrdiff_t)gridDim.x * blockDim.x) {
        const ptrdiff_t g = t >> 3;
        const bool valid = g < N;
        const int j0 = valid ? off[g] : 0, j1 = valid ? off[g + 1] : 0;
        T acc[BS];
#pragma unroll
        for (int c = 0; c < BS; c++) acc[c] = 0;
        for (int j = j0 + lane; j < j1; j += 8) {
            const int32_t q = ent[j];
            element((ptrdiff_t)(q >> 3), q & 7, acc);
        }
#pragma unroll
        for (int m = 1; m < 8; m <<= 1)
#pragma unroll
            for (int c = 0; c < BS; c++) acc[c] += __shfl_xor(acc[c], m, 8);
        if (valid && lane < BS) {
            T v = acc[0];
#pragma unroll
            for (int c = 1; c < BS; c++) v = lane == c ? acc[c] : v;
            const ptrdiff_t i = g * BS + lane;
            y[i] = mask && ((mask[g] >> lane) & 1) ? x[i] : v;
        }
    }
}
__global__ void __launch_bounds__(256)
    hex8_laplacian_node_kernel(const ptrdiff_t N, const ptrdiff_t E, const int32_t *__restrict__ off,
                               const int32_t *__restrict__ ent, const int32_t *__restrict__ idx,
                               const float *__restrict__ fff, const float *__restrict__ coeff,
                               const double *__restrict__ x, double *__restrict__ y,
                               const uint8_t *__restrict__ mask) {
    hex8_node_apply<1, double>(N, off, ent, x, y, mask, [&](ptrdiff_t e, int n, double(&acc)[1]) {
        double u[8], f[6];
#pragma unroll
        for (int k = 0; k < 8; k++) u[k] = x[idx[k * E + e]];
        const double c = (coeff ? (double)coeff[e] : 1.0) * 0.125;
#pragma unroll
        for (int k = 0; k < 6; k++) f[k] = (double)fff[k * E + e] * c;
        hex8_laplacian_sf_element(
            f, [&](int k) { return u[k]; }, [&](int k, double v) { acc[0] += k == n ? v : 0.0; });
    });
}
template <typename T, typename G>
__global__ void __launch_bounds__(256)
    hex8_elasticity_node_kernel(const ptrdiff_t N, const ptrdiff_t E, const int32_t *__restrict__ off,
                                const int32_t *__restrict__ ent, const int32_t *__restrict__ idx,
                                const G *__restrict__ adjg, const G *__restrict__ detg, const double mu,
                                const double lambda, const float *__restrict__ coeff, const T *__restrict__ x,
                                T *__restrict__ y, const uint8_t *__restrict__ mask) {
    hex8_node_apply<3, T>(N, off, ent, x, y, mask, [&](ptrdiff_t e, int n, T(&acc)[3]) {
        T u[8][3];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const ptrdiff_t g = idx[k * E + e];
#pragma unroll
            for (int d = 0; d < 3; d++) u[k][d] = x[g * 3 + d];
        }
        double a[9];
#pragma unroll
        for (int k = 0; k < 9; k++) a[k] = load_geom<G>(adjg, k * E + e);
        hex8_elasticity_sf_element<T>(
            a, load_geom<G>(detg, e), coeff ? (double)coeff[e] : 1.0, mu, lambda,
            [&](int k, int d) { return u[k][d]; }, [&](int k, int d, T v) { acc[d] += k == n ? v : T(0); });
    });
}

// out[k][s] = in[k][perm[s]]: per-element rows in patch-slot order
template <typename G>
__global__ void patch_gather_rows_kernel(const int rows, const ptrdiff_t E, const int32_t *__restrict__ perm,
                                         const G *__restrict__ in, G *__restrict__ out) {
    for (ptrdiff_t i = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; i < rows * E;
         i += (ptrdiff_t)gridDim.x * blockDim.x) {
        const ptrdiff_t k = i / E, s = i - k * E;
        out[i] = in[k * E + perm[s]];
    }
}

// The same operator with eight lanes per element, one per Gauss point (small meshes, e.g. the hex8
// levels of a multigrid hierarchy, where one lane per element leaves most of the GPU idle): each
// lane evaluates its point's contribution to all 24 element rows, a butterfly over the eight lanes
// sums them, and lane n adds the rows of corner n.
__global__ void __launch_bounds__(256)
    hex8_elasticity_apply_qp_kernel(const ptrdiff_t E, const int32_t *__restrict__ idx,
                                    const float *__restrict__ adjg, const float *__restrict__ detg,
                                    const double mu0, const double lambda0, const float *__restrict__ coeff,
                                    const double *__restrict__ x, double *__restrict__ y) {
    const double gp[2] = {0.5 - 0.28867513459481288225, 0.5 + 0.28867513459481288225};
    const int q = threadIdx.x & 7;
    // every lane of a group of eight takes part in the butterfly, also past the last element
    for (ptrdiff_t t = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; t - q < E * 8;
         t += (ptrdiff_t)gridDim.x * blockDim.x) {
        const ptrdiff_t e = t >> 3;
        const bool valid = e < E;
        const ptrdiff_t ee = valid ? e : 0;
        int32_t v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = idx[k * E + ee];
        double adj[9];
#pragma unroll
        for (int k = 0; k < 9; k++) adj[k] = (double)adjg[k * E + ee];
        const double det = (double)detg[ee];
        const double c = coeff ? (double)coeff[ee] : 1.0;
        const double mu = mu0 * c, lambda = lambda0 * c;
        const double idet = 1.0 / det;
        const double w = det * 0.125;
        const double qx = gp[q & 1], qy = gp[(q >> 1) & 1], qz = gp[q >> 2];
        double Gh[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
        for (int n = 0; n < 8; n++) {
            double g[3];
            q1_ref_grad(n, qx, qy, qz, g);
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double u = x[(ptrdiff_t)v[n] * 3 + d];
                Gh[d][0] += u * g[0];
                Gh[d][1] += u * g[1];
                Gh[d][2] += u * g[2];
            }
        }
        double F[3][3];
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int k = 0; k < 3; k++)
                F[d][k] = (Gh[d][0] * adj[0 * 3 + k] + Gh[d][1] * adj[1 * 3 + k] + Gh[d][2] * adj[2 * 3 + k]) * idet;
        const double tr = F[0][0] + F[1][1] + F[2][2];
        double Sg[3][3];
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int k = 0; k < 3; k++) Sg[d][k] = mu * (F[d][k] + F[k][d]) + (d == k ? lambda * tr : 0.0);
        double R[3][3];
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int a = 0; a < 3; a++)
                R[d][a] = w * idet * (Sg[d][0] * adj[a * 3 + 0] + Sg[d][1] * adj[a * 3 + 1] + Sg[d][2] * adj[a * 3 + 2]);
        double out[3][8];
#pragma unroll
        for (int n = 0; n < 8; n++) {
            double g[3];
            q1_ref_grad(n, qx, qy, qz, g);
#pragma unroll
            for (int d = 0; d < 3; d++) out[d][n] = R[d][0] * g[0] + R[d][1] * g[1] + R[d][2] * g[2];
        }
#pragma unroll
        for (int m = 1; m < 8; m <<= 1)
#pragma unroll
            for (int n = 0; n < 8; n++)
#pragma unroll
                for (int d = 0; d < 3; d++) out[d][n] += __shfl_xor(out[d][n], m, 8);
        if (valid) {
#pragma unroll
            for (int n = 0; n < 8; n++)
                if (n == q) {
#pragma unroll
                    for (int d = 0; d < 3; d++) atomicAdd(&y[(ptrdiff_t)v[n] * 3 + d], out[d][n]);
                }
        }
    }
}

template <typename T, typename G>
__global__ void hex8_elasticity_diag_kernel(const ptrdiff_t E, const int32_t *__restrict__ idx,
                                            const G *__restrict__ adjg, const G *__restrict__ detg,
                                            const double mu0, const double lambda0, const float *__restrict__ coeff,
                                            const int block, T *__restrict__ d) {
  for (ptrdiff_t t = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; t < E * 8;
       t += (ptrdiff_t)gridDim.x * blockDim.x) {
    const ptrdiff_t e = t / 8;
    const int n = (int)(t - e * 8);
    double adj[9];
    for (int k = 0; k < 9; k++) adj[k] = load_geom<G>(adjg, k * E + e);
    const double det = load_geom<G>(detg, e);
    const double c = coeff ? (double)coeff[e] : 1.0;
    const int ca[6] = {0, 0, 0, 1, 1, 2}, cb[6] = {0, 1, 2, 1, 2, 2};
    const ptrdiff_t g = idx[n * E + e];
    if (block) {
        for (int k = 0; k < 6; k++)
            atomicAdd(&d[g * 6 + k],
                      (T)hex8_elasticity_entry(adj, det, mu0 * c, lambda0 * c, ca[k] * 8 + n, cb[k] * 8 + n));
    } else {
        for (int k = 0; k < 3; k++)
            atomicAdd(&d[g * 3 + k], (T)hex8_elasticity_entry(adj, det, mu0 * c, lambda0 * c, k * 8 + n, k * 8 + n));
    }
  }
}

// ------------------------------------------------------------------ launchers
int tet4_laplacian_apply(ptrdiff_t E, const int32_t *idx, const float *fff, const double *x, double *y,
                         hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    tet4_laplacian_apply_kernel<<<grid_for(E), kBlock, 0, s>>>(E, idx, fff, x, y);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
int tet4_laplacian_diag(ptrdiff_t E, const int32_t *idx, const float *fff, double *d, hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    tet4_laplacian_diag_kernel<<<grid_for(E), kBlock, 0, s>>>(E, idx, fff, d);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
int hex8_laplacian_apply(ptrdiff_t E, const int32_t *idx, const float *fff, const float *coeff, const double *x,
                         double *y, hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    hex8_laplacian_apply_kernel<<<grid_for(E), kBlock, 0, s>>>(E, idx, fff, coeff, x, y);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
int hex8_laplacian_diag(ptrdiff_t E, const int32_t *idx, const float *fff, const float *coeff, double *d,
                        hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    hex8_laplacian_diag_kernel<<<grid_for(E), kBlock, 0, s>>>(E, idx, fff, coeff, d);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
int hex8_laplacian_apply_nodes(ptrdiff_t N, ptrdiff_t E, const int32_t *off, const int32_t *ent, const int32_t *idx,
                               const float *fff, const float *coeff, const double *x, double *y, const uint8_t *mask,
                               hipStream_t s) {
    if (N == 0) return SFEM_SUCCESS;
    hex8_laplacian_node_kernel<<<grid_for(N * 8), kBlock, 0, s>>>(N, E, off, ent, idx, fff, coeff, x, y, mask);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template <typename T, typename G>
int hex8_elasticity_apply_nodes(ptrdiff_t N, ptrdiff_t E, const int32_t *off, const int32_t *ent, const int32_t *idx,
                                const G *adj, const G *det, double mu, double lambda, const float *coeff, const T *x,
                                T *y, const uint8_t *mask, hipStream_t s) {
    if (N == 0) return SFEM_SUCCESS;
    hex8_elasticity_node_kernel<T, G><<<grid_for(N * 8), kBlock, 0, s>>>(N, E, off, ent, idx, adj, det, mu, lambda, coeff, x,
                                                                         y, mask);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template int hex8_elasticity_apply_nodes<double, float>(ptrdiff_t, ptrdiff_t, const int32_t *, const int32_t *,
                                                        const int32_t *, const float *, const float *, double, double,
                                                        const float *, const double *, double *, const uint8_t *,
                                                        hipStream_t);
template int hex8_elasticity_apply_nodes<float, uint16_t>(ptrdiff_t, ptrdiff_t, const int32_t *, const int32_t *,
                                                          const int32_t *, const uint16_t *, const uint16_t *, double,
                                                          double, const float *, const float *, float *,
                                                          const uint8_t *, hipStream_t);
template <typename T, typename G>
int hex8_elasticity_apply(ptrdiff_t E, const int32_t *idx, const G *adj, const G *det, double mu, double lambda,
                          const float *coeff, const T *x, T *y, hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    // one lane per element fills the GPU only from ~2^18 elements on; below, the FP64 operator runs
    // a lane per Gauss point
    if constexpr (std::is_same<T, double>::value && std::is_same<G, float>::value) {
        if (E < (ptrdiff_t)1 << 18) {
            hex8_elasticity_apply_qp_kernel<<<grid_for(E * 8), kBlock, 0, s>>>(E, idx, adj, det, mu, lambda, coeff, x,
                                                                               y);
            SFEM_AMD_HIP_CHECK(hipGetLastError());
            return SFEM_SUCCESS;
        }
    }
    hex8_elasticity_apply_sf_kernel<T, G><<<grid_for(E), kBlock, 0, s>>>(E, idx, adj, det, mu, lambda, coeff, x, y);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template <typename T, typename G>
int hex8_elasticity_diag(ptrdiff_t E, const int32_t *idx, const G *adj, const G *det, double mu, double lambda,
                         const float *coeff, int block, T *d, hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    hex8_elasticity_diag_kernel<T, G>
        <<<grid_for(E * 8), kBlock, 0, s>>>(E, idx, adj, det, mu, lambda, coeff, block, d);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template <typename T, typename G>
int hex8_elasticity_apply_patches(const PatchView &pv, const G *adjp, const G *detp, const float *coeffp, double mu,
                                  double lambda, const T *x, T *y, hipStream_t s) {
    if (pv.npatch == 0) return SFEM_SUCCESS;
    const size_t lds = patch_lds_bytes(pv.maxloc, 3, sizeof(T));
    if (lds > kPatchLdsLimit) {
        set_last_error("hex8 elasticity patches: patch node count exceeds the LDS budget");
        return SFEM_FAILURE;
    }
    hex8_elasticity_patch_kernel<T, G><<<(unsigned)pv.npatch, 256, lds, s>>>(pv, adjp, detp, coeffp, mu, lambda, x, y);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
int laplacian_apply_patches(int nv, const PatchView &pv, const float *fffp, const float *coeffp, const double *x,
                            double *y, hipStream_t s) {
    if (pv.npatch == 0) return SFEM_SUCCESS;
    const size_t lds = patch_lds_bytes(pv.maxloc, 1, sizeof(double));
    if (lds > kPatchLdsLimit || (nv != 4 && nv != 8)) {
        set_last_error("Laplacian patches: tet4 or hex8, patch nodes within the LDS budget");
        return SFEM_FAILURE;
    }
    if (nv == 8)
        laplacian_patch_kernel<8><<<(unsigned)pv.npatch, 256, lds, s>>>(pv, fffp, coeffp, x, y);
    else
        laplacian_patch_kernel<4><<<(unsigned)pv.npatch, 256, lds, s>>>(pv, fffp, coeffp, x, y);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template <typename G>
int patch_gather_rows(int rows, ptrdiff_t E, const int32_t *perm, const G *in, G *out, hipStream_t s) {
    if (rows * E == 0) return SFEM_SUCCESS;
    patch_gather_rows_kernel<G><<<grid_for(rows * E), kBlock, 0, s>>>(rows, E, perm, in, out);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template int hex8_elasticity_apply_patches<double, float>(const PatchView &, const float *, const float *,
                                                          const float *, double, double, const double *, double *,
                                                          hipStream_t);
template int hex8_elasticity_apply_patches<float, uint16_t>(const PatchView &, const uint16_t *, const uint16_t *,
                                                            const float *, double, double, const float *, float *,
                                                            hipStream_t);
template int patch_gather_rows<float>(int, ptrdiff_t, const int32_t *, const float *, float *, hipStream_t);
template int patch_gather_rows<uint16_t>(int, ptrdiff_t, const int32_t *, const uint16_t *, uint16_t *, hipStream_t);
// FP64 operator on float32 geometry words; FP32 operator on bf16 words
template int hex8_elasticity_apply<double, float>(ptrdiff_t, const int32_t *, const float *, const float *, double,
                                                  double, const float *, const double *, double *, hipStream_t);
template int hex8_elasticity_apply<float, uint16_t>(ptrdiff_t, const int32_t *, const uint16_t *, const uint16_t *,
                                                    double, double, const float *, const float *, float *,
                                                    hipStream_t);
template int hex8_elasticity_diag<double, float>(ptrdiff_t, const int32_t *, const float *, const float *, double,
                                                 double, const float *, int, double *, hipStream_t);
template int hex8_elasticity_diag<float, uint16_t>(ptrdiff_t, const int32_t *, const uint16_t *, const uint16_t *,
                                                   double, double, const float *, int, float *, hipStream_t);

}  // namespace sfem_amd
