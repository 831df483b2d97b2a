// Host-callable launchers of cnn_kernels.hip (learned smoother).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace sfem_amd {
// out [E][Cout][nxe] from in [E][Cin][nxe] (act = relu if relu_in); half > 0: E = 2 half and the input
// holds half elements, the second half of the batch being their negatives
int cnn_conv_forward(int L, ptrdiff_t E, ptrdiff_t half, int Cin, int Cout, const float *in, const float *W, int relu_in,
                     float *out, hipStream_t s);
int cnn_conv_backward_data(int L, ptrdiff_t E, int Cin, int Cout, const float *dout, const float *W, const float *act_in,
                           int relu_in, float *din, hipStream_t s);
// Weight gradients of one layer as cnn_weight_partials(E) partials, `stride` floats apart (half as above);
// cnn_sum_weight_partials adds them for all nw weights into grad, unless loss[1] (device, the target's
// norm) is not positive, and writes loss[0..1] and (with_grad) the gradients to pinned host memory.
int cnn_weight_partials(ptrdiff_t E);
int cnn_conv_backward_weights(int L, ptrdiff_t E, ptrdiff_t half, int Cin, int Cout, const float *dout, const float *in,
                              int relu_in, ptrdiff_t stride, float *partial, hipStream_t s);
int cnn_sum_weight_partials(int nb, int nw, const float *partial, const double *loss, float *grad, double *host,
                            int with_grad, hipStream_t s);
int cnn_sub_halves(ptrdiff_t n, const float *a, const float *b, float *out, hipStream_t s);
// For the output o = ga - gb: loss[0..1] (device) = sum (o - t)^2, sum t^2, and dpm = +-2 (o - t) / loss[1]
// (part: 512 doubles, diff: n floats of workspace)
int cnn_loss_and_gradient(ptrdiff_t n, const float *ga, const float *gb, const float *t, float *diff, double *part,
                          double *loss, float *dpm, hipStream_t s);
int cnn_adam(int n, const float *g, float *w, float *m, float *v, float lr, float b1, float b2, float eps, int step,
             hipStream_t s);
// Element values of component comp of a bs-interleaved vector: out [E][nxe], or with channels the
// channel comp of out [E][bs][nxe]
template <typename T>
int gather_elements(ptrdiff_t E, int nxe, const int32_t *idx, int bs, int comp, const T *vec, const T *scale,
                    float *out, hipStream_t s, bool channels = false);
// vec[node * bs + comp] += alpha * val / count[node] over the element values (layout as gather_elements)
template <typename T>
int scatter_elements(ptrdiff_t E, int nxe, const int32_t *idx, int bs, int comp, const uint16_t *count, float alpha,
                     const float *val, T *vec, hipStream_t s, bool channels = false);
// fused BF16 MFMA inference (hidden 16, 4 layers, L <= 8); W16: bf16 weights of the 4 layers in
// MFMA lane order (kCnnPackedWeights entries, see cnn_pack_weights)
constexpr int kCnnPackedWeights = 512 + 2 * 7680 + 1024;
void cnn_pack_weights(const float *W, uint16_t *packed);
int cnn_infer_mfma(int L, ptrdiff_t E, const uint16_t *W16, const float *z, float *out, hipStream_t s);
}  // namespace sfem_amd
