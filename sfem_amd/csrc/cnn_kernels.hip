// Learned sshex8 smoother: a per-macro-element 3x3x3 CNN on the (L+1)^3 micro-grid (zero
// padding outside the element).  Training kernels run in FP32 (direct convolution with the
// element's channels staged in LDS); inference runs the fused network on MFMA with BF16
// weights and activations and FP32 accumulation.
//
// Layouts: activations [E][C][nxe] float (node index = lidx), weights [Cout][Cin][27] with
// offset k = (dz+1)*9 + (dy+1)*3 + (dx+1).
#include <atomic>

#include "cnn_kernels.hpp"
#include "common.hpp"

namespace sfem_amd {

// ------------------------------------------------------------------ FP32 convolutions
// The element's channels sit in LDS with a zero halo that lines and planes share: line stride
// L + 2 (the cell after a line's last node is both its x = L + 1 and the next line's x = -1),
// plane stride (L + 2)^2 likewise, so all 27 neighbours of a node are plain reads at constant
// offsets from one address, without tests.  At L = 8 a channel takes 1,111 words against 1,331
// for a halo of its own per line, which lets two blocks with 16 channels share a CU.
//
// A block works on NB consecutive nodes of one element and stages the planes that those and their
// neighbours lie in: all of them (NB >= the element's nodes) when the batch fills the GPU with a block
// per element, the few around 64 nodes when it does not (a training batch of 32 elements is 64 of
// the odd network): more and smaller blocks, several to a CU, so that one block's loads overlap
// another's products.
template <int L, int NB>
struct ConvShape {
    static constexpr int N1 = L + 1, NXE = N1 * N1 * N1, PLANE = N1 * N1;
    static constexpr bool FULL = NB >= NXE;
    static constexpr int LS = L + 2, PS = LS * LS, OFF = PS + LS + 1;
    // planes the block's nodes can touch, and the most nodes staged (a plane more on each side)
    static constexpr int PL = FULL || (NB - 1) / PLANE + 2 > N1 ? N1 : (NB - 1) / PLANE + 2;
    static constexpr int STAGED = (PL + 2 < N1 ? PL + 2 : N1) * PLANE;
    static constexpr int NPAD = PL * PS + (L + 1) * LS + L + 1 + OFF + 1;
    // channel strides (words) by the access of the matrix operand: 16 (mod 32) where a half-wave
    // reads 16 consecutive nodes of two channels, 2 (mod 32) where it reads two nodes of 16 channels:
    // either way its 32 words lie in different banks
    static constexpr int CSN = NPAD + ((16 - NPAD % 32) + 32) % 32;
    static constexpr int CSC = NPAD + ((2 - NPAD % 32) + 32) % 32;
    static constexpr int ROWS = FULL ? NXE : NB;  // nodes of the unpadded rows, read as CSC
    static constexpr int RSC = ROWS + ((2 - ROWS % 32) + 32) % 32;
};
// LDS cell of node v when the staged planes start at zlo - 1
template <int L>
__device__ __forceinline__ int conv_pad(int v, int zlo) {
    using S = ConvShape<L, 1 << 20>;
    const int x = v % S::N1, y = (v / S::N1) % S::N1, z = v / (S::N1 * S::N1);
    return (z - zlo) * S::PS + y * S::LS + x + S::OFF;
}
template <int L>
__host__ __device__ constexpr int conv_shift(int k) {
    using S = ConvShape<L, 1 << 20>;
    return (k / 9 - 1) * S::PS + ((k / 3) % 3 - 1) * S::LS + (k % 3 - 1);
}

// The planes around nodes [n0, n1) of C channels of one element: load() issues every load of a thread
// (CH >= C channels of its nodes, absent channels re-reading channel 0), store() puts them into the
// halo layout, after relu if asked, times sg; the halo and the absent channels are zero.
template <int L, int NB, int CS, int CH, int BLOCK>
struct ConvStage {
    using S = ConvShape<L, NB>;
    static constexpr int NV = (S::STAGED + BLOCK - 1) / BLOCK;
    float r[CH][NV];
    int v0, v1, zlo;
    __device__ __forceinline__ void load(const float *__restrict__ in, int C, int n0, int n1) {
        zlo = n0 / S::PLANE;
        const int zhi = (n1 - 1) / S::PLANE;
        v0 = (zlo > 0 ? zlo - 1 : 0) * S::PLANE;
        v1 = (zhi < L ? zhi + 2 : L + 1) * S::PLANE;
#pragma unroll
        for (int c = 0; c < CH; c++)
#pragma unroll
            for (int b = 0; b < NV; b++) {
                const int v = v0 + threadIdx.x + b * BLOCK;
                r[c][b] = in[(size_t)(c < C ? c : 0) * S::NXE + (v < v1 ? v : v0)];
            }
    }
    static __device__ __forceinline__ void clear(float *__restrict__ lds) {
        for (int i = threadIdx.x; i < CH * CS / 2; i += BLOCK) ((float2 *)lds)[i] = float2{0.f, 0.f};
    }
    // after clear() and a barrier
    __device__ __forceinline__ void store(float *__restrict__ lds, int C, bool relu, float sg) const {
#pragma unroll
        for (int b = 0; b < NV; b++) {
            const int v = v0 + threadIdx.x + b * BLOCK;
            if (v >= v1) continue;
            float *q = lds + conv_pad<L>(v, zlo);
#pragma unroll
            for (int c = 0; c < CH; c++)
                if (c < C) q[c * CS] = sg * (relu ? fmaxf(r[c][b], 0.f) : r[c][b]);
        }
    }
};
// element e of a batch whose second half is the negated first one (half > 0), see conv_mfma_kernel
__device__ __forceinline__ const float *conv_source(const float *in, ptrdiff_t e, ptrdiff_t half, size_t per, float &sg) {
    const bool neg = half > 0 && e >= half;
    sg = neg ? -1.f : 1.f;
    return in + (size_t)(neg ? e - half : e) * per;
}

typedef float cv_f4 __attribute__((ext_vector_type(4)));

// out[e][m][v] = sum_c sum_k w(m, c, k) act(in[e][c][v + off_k]), M output and C input channels (<= 16):
//   forward: w = W[m][c][k], act = relu if relu_in;
//   backward (bwd): w = W[c][m][26 - k], the gradient w.r.t. a layer's input from the gradient of its
//   output, zero where mask[e][m][v] <= 0 (the layer's input before its relu; null: no mask).
// half > 0: elements half .. 2 half - 1 of the input are the first half negated (the odd network's
// second evaluation), read from there.
//
// On the matrix cores in FP32 (16x16x4: M = output channels, N = 16 consecutive nodes, K = four input
// channels at one offset; one input channel (Q == 0): K = four offsets).  What bounds it: 108
// products of 32 cycles per tile at 16 -> 16 channels; the operand reads (one LDS word per lane and
// product, at constant offsets) take a quarter of that.  The weights stay in registers (27 Q per lane).
// A block is four waves; with NB = 64 each has one tile.  64 elements, L = 8, 16 -> 16:
// 15 us, where a node per thread with scalar products over LDS took 100 us (4 us of products at 154
// TFLOP/s; the rest is launch, load latency and staging).
template <int L, int Q, int NB>
__global__ void __launch_bounds__(256, 2)
    conv_mfma_kernel(const ptrdiff_t half, const int C, const int M, const float *__restrict__ in,
                     const float *__restrict__ W, const int relu_in, const int bwd, const float *__restrict__ mask,
                     float *__restrict__ out) {
    using S = ConvShape<L, NB>;
    constexpr int CS = S::CSN, QC = Q ? Q : 1;
    extern __shared__ __align__(16) float conv_lds[];
    const ptrdiff_t e = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int n0 = S::FULL ? 0 : (int)blockIdx.y * NB;
    const int n1 = S::FULL || n0 + NB > S::NXE ? S::NXE : n0 + NB;
    float sg;
    const float *src = conv_source(in, e, half, (size_t)C * S::NXE, sg);
    ConvStage<L, NB, CS, Q ? 4 * Q : 1, 256> st;
    st.load(src, C, n0, n1);
    float a[QC * 27];
    if constexpr (Q > 0) {
        // the weights through LDS (one coalesced read per block), rows two words apart mod 32 so that
        // the 16 rows a half-wave reads lie in different banks
        constexpr int NW = (16 * 4 * Q * 27 + 255) / 256;
        const int rows = bwd ? C : M, len = (bwd ? M : C) * 27, rs = len + 2, nw = rows * len;
        const unsigned inv = 0xffffffffu / (unsigned)len + 1;  // i / len = umulhi(i, inv) for i < 2^16
        float wr[NW];
#pragma unroll
        for (int j = 0; j < NW; j++) {
            const int i = threadIdx.x + j * 256;
            wr[j] = W[i < nw ? i : 0];
        }
#pragma unroll
        for (int j = 0; j < NW; j++) {
            const int i = threadIdx.x + j * 256;
            if (i < nw) conv_lds[i + 2 * (int)__umulhi((unsigned)i, inv)] = wr[j];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int ch = 4 * q + g;
            const bool ok = c < M && ch < C;
            const float *w = conv_lds + (ok ? (bwd ? ch * rs + c * 27 + 26 : c * rs + ch * 27) : 26);
#pragma unroll
            for (int k = 0; k < 27; k++) {
                const float v = w[bwd ? -k : k];
                a[q * 27 + k] = ok ? v : 0.f;
            }
        }
        __syncthreads();
    } else {
#pragma unroll
        for (int j = 0; j < 7; j++) {
            const int k = 4 * j + g;
            const bool ok = c < M && k < 27;
            const float v = W[ok ? c * 27 + (bwd ? 26 - k : k) : 0];
            a[j] = ok ? v : 0.f;
        }
    }
    st.clear(conv_lds);
    __syncthreads();
    st.store(conv_lds, C, relu_in != 0, sg);
    __syncthreads();
    int sh[7];
    if constexpr (Q == 0) {
#pragma unroll
        for (int j = 0; j < 7; j++) {
            const int k = 4 * j + g < 27 ? 4 * j + g : 13;
            sh[j] = (k / 9 - 1) * S::PS + ((k / 3) % 3 - 1) * S::LS + (k % 3 - 1);
        }
    }
    for (int t0 = n0 + 16 * wave; t0 < n1; t0 += 64) {
        const int n = t0 + c;
        const bool real = n < n1;
        const int base = conv_pad<L>(real ? n : n0, st.zlo);
        cv_f4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};  // two chains of products
        if constexpr (Q > 0) {
            const float *b = conv_lds + g * CS + base;
#pragma unroll
            for (int k = 0; k < 27; k++)
#pragma unroll
                for (int q = 0; q < Q; q++)
                    acc[(k * Q + q) & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        a[q * 27 + k], b[4 * q * CS + conv_shift<L>(k)], acc[(k * Q + q) & 1], 0, 0, 0);
        } else {
#pragma unroll
            for (int j = 0; j < 7; j++)
                acc[j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], conv_lds[base + sh[j]], acc[j & 1], 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = 4 * g + r;
            if (!real || m >= M) continue;
            const size_t o = ((size_t)e * M + m) * S::NXE + n;
            float v = acc[0][r] + acc[1][r];
            if (mask && mask[o] <= 0.f) v = 0.f;
            out[o] = v;
        }
    }
}

// The same convolution for at most three output channels (the network's last layer), where 13 to 15 of
// the matrix tile's 16 rows would be padding: 64 nodes at a time, each of the four waves taking every
// fourth input channel (weights uniform: scalar loads), summed over the waves in LDS in wave order.
// Bound by the LDS reads (27 C words per node).
template <int L, int M, int NB>
__global__ void __launch_bounds__(256)
    conv_narrow_kernel(const ptrdiff_t half, const int C, const float *__restrict__ in, const float *__restrict__ W,
                       const int relu_in, const int bwd, const float *__restrict__ mask, float *__restrict__ out) {
    using S = ConvShape<L, NB>;
    constexpr int CS = S::CSN;
    extern __shared__ __align__(16) float conv_lds[];
    __shared__ float red[4][M][64];
    const ptrdiff_t e = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = S::FULL ? 0 : (int)blockIdx.y * NB;
    const int n1 = S::FULL || n0 + NB > S::NXE ? S::NXE : n0 + NB;
    float sg;
    const float *src = conv_source(in, e, half, (size_t)C * S::NXE, sg);
    ConvStage<L, NB, CS, 16, 256> st;
    st.load(src, C, n0, n1);
    st.clear(conv_lds);
    __syncthreads();
    st.store(conv_lds, C, relu_in != 0, sg);
    __syncthreads();
    for (int t0 = n0; t0 < n1; t0 += 64) {
        const int v = t0 + lane;
        const float *b = conv_lds + conv_pad<L>(v < n1 ? v : n0, st.zlo);
        float acc[M];
#pragma unroll
        for (int m = 0; m < M; m++) acc[m] = 0.f;
        for (int ch = wave; ch < C; ch += 4) {
#pragma unroll
            for (int k = 0; k < 27; k++) {
                const float x = b[ch * CS + conv_shift<L>(k)];
#pragma unroll
                for (int m = 0; m < M; m++) acc[m] += W[bwd ? (ch * M + m) * 27 + 26 - k : (m * C + ch) * 27 + k] * x;
            }
        }
#pragma unroll
        for (int m = 0; m < M; m++) red[wave][m][lane] = acc[m];
        __syncthreads();
        for (int m = wave; m < M; m += 4)
            if (v < n1) {
                const size_t o = ((size_t)e * M + m) * S::NXE + v;
                const float s = (red[0][m][lane] + red[1][m][lane]) + (red[2][m][lane] + red[3][m][lane]);
                out[o] = mask && mask[o] <= 0.f ? 0.f : s;
            }
        __syncthreads();
    }
}

// Weight gradients, partial[block][co][ci][k] = sum over the block's elements and nodes of
// dout[co][v] act(in[ci][v + off_k]), on the matrix cores in FP32 with K = four nodes.
//
// Wide layers (more than three channels on both sides): M = co, N = ci, one 16x16 accumulator per
// offset; the eight waves of a block take seven offsets and every second step of four nodes each, and
// the two halves are added in LDS.  What bounds it: 27 products per four nodes (32 cycles each), the LDS
// reads take a third of that; the next step's operands are read before the current products.
// blockIdx.y takes a quarter of an element's nodes when the batch holds few elements (NB).  64
// elements, L = 8, 16 -> 16: 19 us, where one weight per thread with a scalar loop over the nodes took
// 143 us.
// C channels of nodes [n0, n1) as unpadded rows of stride RS (channels C .. 15 zero)
template <int NXE, int RS, int BLOCK>
__device__ __forceinline__ void conv_stage_rows(float *__restrict__ lds, const float *__restrict__ src, int C,
                                                bool relu, int n0, int n1) {
    for (int v = n0 + threadIdx.x; v < n1; v += BLOCK) {
        float r[16];
#pragma unroll
        for (int c = 0; c < 16; c++) r[c] = src[(size_t)(c < C ? c : 0) * NXE + v];
#pragma unroll
        for (int c = 0; c < 16; c++) lds[c * RS + v - n0] = c < C ? (relu ? fmaxf(r[c], 0.f) : r[c]) : 0.f;
    }
}
template <int L, int NB>
__global__ void __launch_bounds__(512)
    conv_weight_kernel(const ptrdiff_t E, const int Cin, const int Cout, const float *__restrict__ dout,
                       const float *__restrict__ in, const int relu_in, const ptrdiff_t stride,
                       float *__restrict__ partial) {
    using S = ConvShape<L, NB>;
    constexpr int KW = 7;
    extern __shared__ __align__(16) float conv_lds[];
    float *sin = conv_lds, *sd = conv_lds + 16 * S::CSC;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int kw = wave & 3, par = wave >> 2;
    const int n0 = S::FULL ? 0 : (int)blockIdx.y * NB;
    const int n1 = S::FULL || n0 + NB > S::NXE ? S::NXE : n0 + NB;
    int sh[KW];
    cv_f4 acc[KW];
#pragma unroll
    for (int j = 0; j < KW; j++) {
        const int k = kw * KW + j < 27 ? kw * KW + j : 13;
        sh[j] = c * S::CSC + (k / 9 - 1) * S::PS + ((k / 3) % 3 - 1) * S::LS + (k % 3 - 1);
        acc[j] = cv_f4{0.f, 0.f, 0.f, 0.f};
    }
    for (ptrdiff_t e = blockIdx.x; e < E; e += gridDim.x) {
        __syncthreads();
        ConvStage<L, NB, S::CSC, 16, 512> st;
        st.load(in + (size_t)e * Cin * S::NXE, Cin, n0, n1);
        st.clear(sin);
        conv_stage_rows<S::NXE, S::RSC, 512>(sd, dout + (size_t)e * Cout * S::NXE, Cout, false, n0, n1);
        __syncthreads();
        st.store(sin, Cin, relu_in != 0, 1.f);
        __syncthreads();
        float a, b[KW];
        auto operands = [&](int v0) {
            const int v = v0 + g;
            const bool ok = v < n1;
            const float x = sd[c * S::RSC + (ok ? v - n0 : 0)];
            a = ok ? x : 0.f;
            const float *q = sin + conv_pad<L>(ok ? v : n0, st.zlo);
#pragma unroll
            for (int j = 0; j < KW; j++) b[j] = q[sh[j]];
        };
        operands(n0 + 4 * par);
        for (int v0 = n0 + 4 * par; v0 < n1; v0 += 8) {
            const float ac = a;
            float bc[KW];
#pragma unroll
            for (int j = 0; j < KW; j++) bc[j] = b[j];
            operands(v0 + 8);  // past the end: a = 0 and node n0's values, not used
#pragma unroll
            for (int j = 0; j < KW; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ac, bc[j], acc[j], 0, 0, 0);
        }
    }
    // the second half's accumulators through LDS (28 KB: the staging space is at least as large)
    __syncthreads();
    cv_f4 *red = (cv_f4 *)conv_lds;
    if (par)
#pragma unroll
        for (int j = 0; j < KW; j++) red[(kw * KW + j) * 64 + lane] = acc[j];
    __syncthreads();
    cv_f4 other[KW];
    if (!par)
#pragma unroll
        for (int j = 0; j < KW; j++) other[j] = red[(kw * KW + j) * 64 + lane];
    __syncthreads();
    // into [co][ci][k] order in LDS, so that the partial is written in whole lines
    if (!par)
#pragma unroll
        for (int j = 0; j < KW; j++) {
            const int k = kw * KW + j;
            if (k >= 27 || c >= Cin) continue;
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (4 * g + r < Cout) conv_lds[((4 * g + r) * Cin + c) * 27 + k] = acc[j][r] + other[j][r];
        }
    __syncthreads();
    float *p = partial + (size_t)(blockIdx.y * gridDim.x + blockIdx.x) * stride;
    for (int i = threadIdx.x; i < Cout * Cin * 27; i += 512) p[i] = conv_lds[i];
}

// Narrow layers (at most three channels on one side, C there, R rows on the other): M = the rows, N =
// the 27 C (channel, offset) pairs in tiles of 16 columns, each lane with its column's address:
//   rows = dout, columns = act(in) at v + off_k   (cols_are_dout 0: the first layer)
//   rows = act(in), columns = dout at v - off_k   (cols_are_dout 1: the last layer)
// half: as in conv_mfma_kernel, for the first layer's input.
template <int L, int C, int NB>
__global__ void __launch_bounds__(256, 2)
    conv_weight_narrow_kernel(const ptrdiff_t E, const ptrdiff_t half, const int R, const int cols_are_dout,
                              const float *__restrict__ rows, const float *__restrict__ cols, const int relu_in,
                              const ptrdiff_t stride, float *__restrict__ partial) {
    using S = ConvShape<L, NB>;
    constexpr int NT = (27 * C + 15) / 16;
    extern __shared__ __align__(16) float conv_lds[];
    float *sc = conv_lds, *sr = conv_lds + C * S::CSN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int n0 = S::FULL ? 0 : (int)blockIdx.y * NB;
    const int n1 = S::FULL || n0 + NB > S::NXE ? S::NXE : n0 + NB;
    int col[NT];
    cv_f4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int j = 16 * t + c, ch = j < 27 * C ? j / 27 : 0, k = j < 27 * C ? j % 27 : 13;
        const int sft = (k / 9 - 1) * S::PS + ((k / 3) % 3 - 1) * S::LS + (k % 3 - 1);
        col[t] = ch * S::CSN + (cols_are_dout ? -sft : sft);
        acc[t] = cv_f4{0.f, 0.f, 0.f, 0.f};
    }
    for (ptrdiff_t e = blockIdx.x; e < E; e += gridDim.x) {
        __syncthreads();
        float sg;
        const float *src = conv_source(cols, e, half, (size_t)C * S::NXE, sg);
        ConvStage<L, NB, S::CSN, C, 256> st;
        st.load(src, C, n0, n1);
        st.clear(sc);
        conv_stage_rows<S::NXE, S::RSC, 256>(sr, rows + (size_t)e * R * S::NXE, R, cols_are_dout && relu_in, n0, n1);
        __syncthreads();
        st.store(sc, C, !cols_are_dout && relu_in, sg);
        __syncthreads();
        // the waves take every fourth step of four nodes; summed over the waves below
        for (int v0 = n0 + 4 * wave; v0 < n1; v0 += 16) {
            const int v = v0 + g;
            const bool ok = v < n1;
            const float x = sr[c * S::RSC + (ok ? v : n0) - n0];
            const float a = ok ? x : 0.f;
            const float *b = sc + conv_pad<L>(ok ? v : n0, st.zlo);
#pragma unroll
            for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[col[t]], acc[t], 0, 0, 0);
        }
    }
    // the four waves' accumulators, added in wave order (their LDS lies in the staging space)
    __syncthreads();
    cv_f4 *red = (cv_f4 *)conv_lds;
#pragma unroll
    for (int t = 0; t < NT; t++) red[(wave * NT + t) * 64 + lane] = acc[t];
    __syncthreads();
    float *p = partial + (size_t)(blockIdx.y * gridDim.x + blockIdx.x) * stride;
    for (int t = wave; t < NT; t += 4) {
        cv_f4 s = red[t * 64 + lane];
#pragma unroll
        for (int w = 1; w < 4; w++) s += red[(w * NT + t) * 64 + lane];
        const int j = 16 * t + c;
        if (j >= 27 * C) continue;
        const int ch = j / 27, k = j % 27;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = 4 * g + r;
            if (m < R) p[(cols_are_dout ? ch * R + m : m * C + ch) * 27 + k] = s[r];
        }
    }
}

// grad[t] = sum over the nb partials, 16 threads per weight (each every 16th partial), in a fixed order;
// nothing is written unless the target's norm (loss[1]) is positive.  The last block also copies the
// loss sums, and each block its gradients, into pinned host memory (host: 2 doubles, then the
// gradients as floats when with_grad).
__global__ void __launch_bounds__(1024)
    sum_weight_partials_kernel(const int nb, const int nw, const float *__restrict__ partial,
                               const double *__restrict__ loss, float *__restrict__ grad, double *__restrict__ host,
                               const int with_grad) {
    __shared__ float s[16][65];
    const int o = threadIdx.x & 63, j = threadIdx.x >> 6, t = blockIdx.x * 64 + o;
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x < 2) host[threadIdx.x] = loss[threadIdx.x];
    if (!(loss[1] > 0)) return;  // uniform
    float v = 0.f;
    if (t < nw) {
#pragma unroll 8
        for (int b = j; b < nb; b += 16) v += partial[(size_t)b * nw + t];
    }
    s[j][o] = v;
    __syncthreads();
    if (j == 0 && t < nw) {
#pragma unroll
        for (int i = 1; i < 16; i++) v += s[i][o];
        grad[t] = v;
        if (with_grad) ((float *)(host + 2))[t] = v;
    }
}

// out = a - b (the odd symmetrisation g(z) - g(-z))
__global__ void sub_halves_kernel(const ptrdiff_t n, const float *__restrict__ a, const float *__restrict__ b,
                                  float *__restrict__ out) {
    for (ptrdiff_t i = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (ptrdiff_t)gridDim.x * blockDim.x)
        out[i] = a[i] - b[i];
}

// o = a - b (the odd symmetrisation) against the target: part[b] = (sum (o - t)^2, sum t^2) over a
// fixed grid, o kept as the difference d = o - t
constexpr int kErrBlocks = 256;
__global__ void __launch_bounds__(256) sq_err_partial_kernel(const ptrdiff_t n, const float *__restrict__ ga,
                                                             const float *__restrict__ gb, const float *__restrict__ t,
                                                             float *__restrict__ diff, double *__restrict__ part) {
    __shared__ double s1[256], s2[256];
    double a = 0, b = 0;
    for (ptrdiff_t i = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (ptrdiff_t)gridDim.x * blockDim.x) {
        const float o = ga[i] - gb[i], ti = t[i];
        const double d = (double)o - (double)ti;
        diff[i] = o - ti;
        a += d * d;
        b += (double)ti * (double)ti;
    }
    s1[threadIdx.x] = a;
    s2[threadIdx.x] = b;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st) {
            s1[threadIdx.x] += s1[threadIdx.x + st];
            s2[threadIdx.x] += s2[threadIdx.x + st];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = s1[0];
        part[2 * blockIdx.x + 1] = s2[0];
    }
}

// The sums of the partials (every block sums all of them in the same order: no host round trip between
// the loss and the backward pass), then dpm = [2 d / norm; -2 d / norm]; block 0 keeps the sums.
__global__ void __launch_bounds__(256) dloss_kernel(const ptrdiff_t n, const float *__restrict__ diff,
                                                    const double *__restrict__ part, double *__restrict__ loss,
                                                    float *__restrict__ dpm) {
    __shared__ double s1[kErrBlocks], s2[kErrBlocks];
    s1[threadIdx.x] = part[2 * threadIdx.x];
    s2[threadIdx.x] = part[2 * threadIdx.x + 1];
    __syncthreads();
    for (int st = kErrBlocks / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) {
            s1[threadIdx.x] += s1[threadIdx.x + st];
            s2[threadIdx.x] += s2[threadIdx.x + st];
        }
        __syncthreads();
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        loss[0] = s1[0];
        loss[1] = s2[0];
    }
    const float inv_norm = (float)(1.0 / s2[0]);
    for (ptrdiff_t i = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (ptrdiff_t)gridDim.x * blockDim.x) {
        const float d = 2.f * diff[i] * inv_norm;
        dpm[i] = d;
        dpm[n + i] = -d;
    }
}
static_assert(kErrBlocks == 256, "dloss_kernel loads one partial per thread");

__global__ void adam_kernel(const int n, const float *__restrict__ g, float *__restrict__ w, float *__restrict__ m,
                            float *__restrict__ v, const float lr, const float b1, const float b2, const float eps,
                            const float c1, const float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// out[e * ld + off + v] = vec[idx[e][v]*bs + comp] * (scale ? scale[...] : 1)  (ld = nxe, off = 0: [E][nxe];
// ld = bs * nxe, off = comp * nxe: the channel comp of [E][bs][nxe])
template <typename T>
__global__ void gather_elements_kernel(const ptrdiff_t E, const int nxe, const int32_t *__restrict__ idx, const int bs,
                                       const int comp, const T *__restrict__ vec, const T *__restrict__ scale,
                                       const int ld, const int off, float *__restrict__ out) {
    const ptrdiff_t n = E * nxe;
    for (ptrdiff_t t = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (ptrdiff_t)gridDim.x * blockDim.x) {
        const ptrdiff_t d = (ptrdiff_t)idx[t] * bs + comp;
        const ptrdiff_t e = t / nxe;
        out[e * ld + off + (t - e * nxe)] = (float)(scale ? vec[d] * scale[d] : vec[d]);
    }
}

// vec[idx[e][v]*bs + comp] += alpha * val[e * ld + off + v] / count[idx]
template <typename T>
__global__ void scatter_elements_kernel(const ptrdiff_t E, const int nxe, const int32_t *__restrict__ idx, const int bs,
                                        const int comp, const uint16_t *__restrict__ count, const float alpha,
                                        const int ld, const int off, const float *__restrict__ val,
                                        T *__restrict__ vec) {
    const ptrdiff_t n = E * nxe;
    for (ptrdiff_t t = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (ptrdiff_t)gridDim.x * blockDim.x) {
        const int32_t g = idx[t];
        const ptrdiff_t e = t / nxe;
        atomicAdd(&vec[(ptrdiff_t)g * bs + comp], (T)(alpha * val[e * ld + off + (t - e * nxe)] / (float)count[g]));
    }
}

// ------------------------------------------------------------------ launchers
// Dynamic LDS above the default 64 KB needs the function attribute, once per function and device.
template <auto Fn>
static int raise_lds_limit(size_t bytes) {
    static std::atomic<uint64_t> done{0};
    if (bytes <= 64 * 1024) return SFEM_SUCCESS;
    int dev = 0;
    SFEM_AMD_HIP_CHECK(hipGetDevice(&dev));
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return SFEM_SUCCESS;
    SFEM_AMD_HIP_CHECK(
        hipFuncSetAttribute((const void *)Fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    done.fetch_or(bit, std::memory_order_acq_rel);
    return SFEM_SUCCESS;
}

// Blocks on whole elements once the batch alone fills the GPU (two blocks on each of 256 CUs); below,
// blocks on 64 nodes (convolutions) or a quarter of the nodes (weight gradients) of an element.
constexpr ptrdiff_t kConvFull = 512;
constexpr int kWhole = 1 << 20;
// whole steps of four nodes where that leaves the last of four blocks some
constexpr int conv_quarter(int nxe) { return 3 * ((nxe + 15) / 16 * 4) < nxe ? (nxe + 15) / 16 * 4 : (nxe + 3) / 4; }
template <int L>
constexpr int kQuarter = conv_quarter(nxe_of(L));
static_assert(3 * kQuarter<1> < nxe_of(1) && 4 * kQuarter<1> >= nxe_of(1) && 4 * kQuarter<8> >= nxe_of(8));

template <int L, int Q, int NB>
static int launch_conv_mfma(ptrdiff_t E, ptrdiff_t half, int C, int M, const float *in, const float *W, int relu_in,
                            int bwd, const float *mask, float *out, hipStream_t s) {
    using S = ConvShape<L, NB>;
    const size_t act = sizeof(float) * (size_t)(Q ? 4 * Q : 1) * S::CSN;
    const size_t w = Q ? sizeof(float) * (size_t)(bwd ? C : M) * ((bwd ? M : C) * 27 + 2) : 0;
    const size_t lds = act > w ? act : w;
    if (raise_lds_limit<conv_mfma_kernel<L, Q, NB>>(lds)) return SFEM_FAILURE;
    const dim3 grid((unsigned)E, S::FULL ? 1 : (S::NXE + NB - 1) / NB);
    conv_mfma_kernel<L, Q, NB><<<grid, 256, lds, s>>>(half, C, M, in, W, relu_in, bwd, mask, out);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template <int L, int M, int NB>
static int launch_conv_narrow(ptrdiff_t E, ptrdiff_t half, int C, const float *in, const float *W, int relu_in, int bwd,
                              const float *mask, float *out, hipStream_t s) {
    using S = ConvShape<L, NB>;
    const size_t lds = sizeof(float) * (size_t)16 * S::CSN;
    if (raise_lds_limit<conv_narrow_kernel<L, M, NB>>(lds)) return SFEM_FAILURE;
    const dim3 grid((unsigned)E, S::FULL ? 1 : (S::NXE + NB - 1) / NB);
    conv_narrow_kernel<L, M, NB><<<grid, 256, lds, s>>>(half, C, in, W, relu_in, bwd, mask, out);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template <int L, int NB>
static int launch_conv(ptrdiff_t E, ptrdiff_t half, int C, int M, const float *in, const float *W, int relu_in, int bwd,
                       const float *mask, float *out, hipStream_t s) {
    // one input channel: the matrix kernel's K runs over the offsets, whatever M; else at most three
    // output channels run without the matrix cores (conv_narrow_kernel)
    if (C > 1 && M == 1) return launch_conv_narrow<L, 1, NB>(E, half, C, in, W, relu_in, bwd, mask, out, s);
    if (C > 1 && M == 2) return launch_conv_narrow<L, 2, NB>(E, half, C, in, W, relu_in, bwd, mask, out, s);
    if (C > 1 && M == 3) return launch_conv_narrow<L, 3, NB>(E, half, C, in, W, relu_in, bwd, mask, out, s);
    switch (C == 1 ? 0 : (C + 3) / 4) {
        case 0: return launch_conv_mfma<L, 0, NB>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 1: return launch_conv_mfma<L, 1, NB>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 2: return launch_conv_mfma<L, 2, NB>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 3: return launch_conv_mfma<L, 3, NB>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 4: return launch_conv_mfma<L, 4, NB>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
    }
    set_last_error("cnn: at most 16 channels");
    return SFEM_FAILURE;
}
template <int L>
static int launch_conv_any(ptrdiff_t E, ptrdiff_t half, int C, int M, const float *in, const float *W, int relu_in,
                           int bwd, const float *mask, float *out, hipStream_t s) {
    if constexpr (nxe_of(L) > 64)
        if (E < kConvFull) return launch_conv<L, 64>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
    return launch_conv<L, kWhole>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
}
static int conv(int L, ptrdiff_t E, ptrdiff_t half, int C, int M, const float *in, const float *W, int relu_in, int bwd,
                const float *mask, float *out, hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    if (M > 16) {
        set_last_error("cnn: at most 16 channels");
        return SFEM_FAILURE;
    }
    switch (L) {
        case 1: return launch_conv_any<1>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 2: return launch_conv_any<2>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 3: return launch_conv_any<3>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 4: return launch_conv_any<4>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 5: return launch_conv_any<5>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 6: return launch_conv_any<6>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 7: return launch_conv_any<7>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
        case 8: return launch_conv_any<8>(E, half, C, M, in, W, relu_in, bwd, mask, out, s);
    }
    set_last_error("cnn: level must be 1..8");
    return SFEM_FAILURE;
}

int cnn_conv_forward(int L, ptrdiff_t E, ptrdiff_t half, int Cin, int Cout, const float *in, const float *W, int relu_in,
                     float *out, hipStream_t s) {
    return conv(L, E, half, Cin, Cout, in, W, relu_in, 0, nullptr, out, s);
}

int cnn_conv_backward_data(int L, ptrdiff_t E, int Cin, int Cout, const float *dout, const float *W, const float *act_in,
                           int relu_in, float *din, hipStream_t s) {
    return conv(L, E, 0, Cout, Cin, dout, W, 0, 1, relu_in ? act_in : nullptr, din, s);
}

// the weight-gradient kernels' grid: blocks on elements times blocks per element
static dim3 weight_grid(ptrdiff_t E) {
    return E < kConvFull / 4 ? dim3((unsigned)E, 4) : dim3((unsigned)(E < kConvFull ? E : kConvFull), 1);
}
int cnn_weight_partials(ptrdiff_t E) {
    const dim3 g = weight_grid(E);
    return (int)(g.x * g.y);
}
template <int L, int C, int NB>
static int launch_weight_narrow(ptrdiff_t E, ptrdiff_t half, int R, int cols_are_dout, const float *rows,
                                const float *cols, int relu_in, ptrdiff_t stride, float *partial, hipStream_t s) {
    using S = ConvShape<L, NB>;
    const size_t stage = sizeof(float) * ((size_t)C * S::CSN + 16 * (size_t)S::RSC);
    const size_t red = 16 * (size_t)64 * 4 * ((27 * C + 15) / 16);
    const size_t lds = stage > red ? stage : red;
    if (raise_lds_limit<conv_weight_narrow_kernel<L, C, NB>>(lds)) return SFEM_FAILURE;
    conv_weight_narrow_kernel<L, C, NB>
        <<<weight_grid(E), 256, lds, s>>>(E, half, R, cols_are_dout, rows, cols, relu_in, stride, partial);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template <int L, int NB>
static int launch_weight(ptrdiff_t E, ptrdiff_t half, int Cin, int Cout, const float *dout, const float *in, int relu_in,
                         ptrdiff_t stride, float *partial, hipStream_t s) {
    using S = ConvShape<L, NB>;
    if (Cin == 1) return launch_weight_narrow<L, 1, NB>(E, half, Cout, 0, dout, in, relu_in, stride, partial, s);
    if (Cin == 2) return launch_weight_narrow<L, 2, NB>(E, half, Cout, 0, dout, in, relu_in, stride, partial, s);
    if (Cin == 3) return launch_weight_narrow<L, 3, NB>(E, half, Cout, 0, dout, in, relu_in, stride, partial, s);
    if (Cout == 1) return launch_weight_narrow<L, 1, NB>(E, 0, Cin, 1, in, dout, relu_in, stride, partial, s);
    if (Cout == 2) return launch_weight_narrow<L, 2, NB>(E, 0, Cin, 1, in, dout, relu_in, stride, partial, s);
    if (Cout == 3) return launch_weight_narrow<L, 3, NB>(E, 0, Cin, 1, in, dout, relu_in, stride, partial, s);
    const size_t stage = sizeof(float) * 16 * (size_t)(S::CSC + S::RSC), red = 16 * (size_t)64 * 28;
    const size_t lds = stage > red ? stage : red;
    if (raise_lds_limit<conv_weight_kernel<L, NB>>(lds)) return SFEM_FAILURE;
    conv_weight_kernel<L, NB><<<weight_grid(E), 512, lds, s>>>(E, Cin, Cout, dout, in, relu_in, stride, partial);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}
template <int L>
static int launch_weight_any(ptrdiff_t E, ptrdiff_t half, int Cin, int Cout, const float *dout, const float *in,
                             int relu_in, ptrdiff_t stride, float *partial, hipStream_t s) {
    if (weight_grid(E).y > 1)
        return launch_weight<L, kQuarter<L>>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
    return launch_weight<L, kWhole>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
}
int cnn_conv_backward_weights(int L, ptrdiff_t E, ptrdiff_t half, int Cin, int Cout, const float *dout, const float *in,
                              int relu_in, ptrdiff_t stride, float *partial, hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    if (Cin > 16 || Cout > 16) {
        set_last_error("cnn: at most 16 channels");
        return SFEM_FAILURE;
    }
    switch (L) {
        case 1: return launch_weight_any<1>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
        case 2: return launch_weight_any<2>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
        case 3: return launch_weight_any<3>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
        case 4: return launch_weight_any<4>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
        case 5: return launch_weight_any<5>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
        case 6: return launch_weight_any<6>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
        case 7: return launch_weight_any<7>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
        case 8: return launch_weight_any<8>(E, half, Cin, Cout, dout, in, relu_in, stride, partial, s);
    }
    set_last_error("cnn: level must be 1..8");
    return SFEM_FAILURE;
}
int cnn_sum_weight_partials(int nb, int nw, const float *partial, const double *loss, float *grad, double *host,
                            int with_grad, hipStream_t s) {
    sum_weight_partials_kernel<<<(nw + 63) / 64, 1024, 0, s>>>(nb, nw, partial, loss, grad, host, with_grad);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}

int cnn_sub_halves(ptrdiff_t n, const float *a, const float *b, float *out, hipStream_t s) {
    sub_halves_kernel<<<grid_for(n), kBlock, 0, s>>>(n, a, b, out);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}

int cnn_loss_and_gradient(ptrdiff_t n, const float *ga, const float *gb, const float *t, float *diff, double *part,
                          double *loss, float *dpm, hipStream_t s) {
    sq_err_partial_kernel<<<kErrBlocks, 256, 0, s>>>(n, ga, gb, t, diff, part);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    dloss_kernel<<<grid_for(n), kBlock, 0, s>>>(n, diff, part, loss, dpm);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}

int cnn_adam(int n, const float *g, float *w, float *m, float *v, float lr, float b1, float b2, float eps, int step,
             hipStream_t s) {
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    adam_kernel<<<(n + 255) / 256, 256, 0, s>>>(n, g, w, m, v, lr, b1, b2, eps, c1, c2);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}

template <typename T>
int gather_elements(ptrdiff_t E, int nxe, const int32_t *idx, int bs, int comp, const T *vec, const T *scale,
                    float *out, hipStream_t s, bool channels) {
    if (E == 0) return SFEM_SUCCESS;
    gather_elements_kernel<T><<<grid_for(E * nxe), kBlock, 0, s>>>(E, nxe, idx, bs, comp, vec, scale,
                                                                   channels ? bs * nxe : nxe, channels ? comp * nxe : 0,
                                                                   out);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}

template <typename T>
int scatter_elements(ptrdiff_t E, int nxe, const int32_t *idx, int bs, int comp, const uint16_t *count, float alpha,
                     const float *val, T *vec, hipStream_t s, bool channels) {
    if (E == 0) return SFEM_SUCCESS;
    scatter_elements_kernel<T><<<grid_for(E * nxe), kBlock, 0, s>>>(E, nxe, idx, bs, comp, count, alpha,
                                                                    channels ? bs * nxe : nxe,
                                                                    channels ? comp * nxe : 0, val, vec);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}

template int gather_elements<double>(ptrdiff_t, int, const int32_t *, int, int, const double *, const double *, float *,
                                     hipStream_t, bool);
template int gather_elements<float>(ptrdiff_t, int, const int32_t *, int, int, const float *, const float *, float *,
                                    hipStream_t, bool);
template int scatter_elements<double>(ptrdiff_t, int, const int32_t *, int, int, const uint16_t *, float, const float *,
                                      double *, hipStream_t, bool);
template int scatter_elements<float>(ptrdiff_t, int, const int32_t *, int, int, const uint16_t *, float, const float *,
                                     float *, hipStream_t, bool);

// ------------------------------------------------------------------ fused BF16 MFMA inference
// One macro element per block (512 threads = 8 waves); the element's
// activations stay in LDS for all four layers and both signs of f(z) = g(z) - g(-z).  Nodes are
// processed in tiles of 16 (the MFMA N dimension); per tile and layer:
//   layer 1 (1 -> 16):  D[co][n]  = sum_{k<32} W1[co][k] z[n + off_k]         one 16x16x32 MFMA
//   layer 2,3 (16->16): D[co][n] += sum_{pairs p} W[co][ci,off] act[n + off]  14 16x16x32 MFMAs,
//                       K = 32 = two offsets x 16 input channels; each wave runs three tiles at
//                       once (three independent accumulation chains)
//   layer 4 (16 -> 1):  P[k][n]   = sum_ci W4[ci][k] act[ci][n] (16x16x16 MFMAs, 16 offsets k per
//                       pass, two passes), then out[n] = sum_k P[k][n + off_k] from LDS.
// Lane layouts (64 lanes, g = lane / 16, c = lane % 16):
//   16x16x32 A: row c, k = 8g + j (j < 8);  B: column c, k = 8g + j;  D: column c, rows 4g + r
//   16x16x16 A: row c, k = 4g + j (j < 4);  B: column c, k = 4g + j;  D: as above
// The input and the activations of layers 1-3 live on the element's grid with a one-point zero
// halo ((L+3)^3 points), so neighbour reads need no validity tests: one address per tile and a
// per-pair offset.  Activations are stored post-ReLU in BF16 as two channel planes
// [half][point][8 channels] (16-byte B reads).  Layer 4's stencil sum reads the unpadded P, with
// the padding node NXE (P == 0) standing in for missing neighbours.
typedef short mf_s4 __attribute__((ext_vector_type(4)));
typedef __bf16 mf_b8 __attribute__((ext_vector_type(8)));
typedef float mf_f4 __attribute__((ext_vector_type(4)));
typedef unsigned int mf_u4 __attribute__((ext_vector_type(4)));
typedef unsigned int mf_u2 __attribute__((ext_vector_type(2)));

typedef __bf16 mf_b2 __attribute__((ext_vector_type(2)));
typedef float mf_f2 __attribute__((ext_vector_type(2)));

// float -> bf16, round to nearest even: the conversions lower to gfx950's v_cvt_pk_bf16_f32
// (bf_pack converts two values with one instruction)
__device__ __forceinline__ __bf16 f2bf(float f) { return (__bf16)f; }
__device__ __forceinline__ unsigned bf_pack(float lo, float hi) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(mf_f2{lo, hi}, mf_b2));
}

template <int L>
struct CnnShape {
    static constexpr int N1 = L + 1;
    static constexpr int NXE = N1 * N1 * N1;
    // node tiles of 16 with at least one padding node (node NXE: P[k][NXE] == 0 stands in for the
    // missing neighbours of the layer-4 stencil sum)
    static constexpr int T = NXE / 16 + 1;
    static constexpr int NP = T * 16;
    // layers 1-3 hold the element on grids with a zero halo, so every node's 27 neighbours are in
    // range and read without tests: the input on the (L+3)^3 grid, the activations on a grid with
    // line stride SY and plane stride SZ chosen so that consecutive nodes, also across line and
    // plane ends, sit one 16-byte row apart mod 8 (eight lanes read all 32 LDS banks)
    static constexpr int P1 = L + 3;
    static constexpr int NH = P1 * P1 * P1;
    static constexpr int SY = L + 9;  // >= L + 3, = L + 1 (mod 8)
    static constexpr int SZ = P1 * SY + ((((L * SY + L + 1) - P1 * SY) % 8) + 8) % 8;  // = L SY + L + 1 (mod 8)
    static constexpr int NA = P1 * SZ;
    static constexpr int THREADS = 512;
    static constexpr int TPG = 3;  // tiles per wave iteration in the hidden layers
    // zs [NH] float | actX [2][NA][8] bf16 | actY [2][NA][8] bf16, aliased by P [16][NP] float
    // (actY is cleared again at the start of each sign)
    static constexpr size_t ZS = (sizeof(float) * NH + 15) / 16 * 16;
    static constexpr size_t ACT = 32 * (size_t)NA;
    static constexpr size_t LDS = ZS + ACT + (ACT > 64 * (size_t)NP ? ACT : 64 * (size_t)NP);
};

// Neighbour validity as bit tests.  cnn_avail: the directions in which node (x, y, z) has a
// neighbour (bits x-, x+, y-, y+, z-, z+) and bit 6 for a real node (in); cnn_need(o): the bits offset
// o requires (bit 7, never available, for the padding offsets o >= 27).  Offset o of the node exists
// iff (cnn_need(o) & ~cnn_avail) == 0.
template <int L>
__device__ __forceinline__ unsigned cnn_avail(int x, int y, int z, bool in) {
    return (unsigned)(x > 0) | (unsigned)(x < L) << 1 | (unsigned)(y > 0) << 2 | (unsigned)(y < L) << 3 |
           (unsigned)(z > 0) << 4 | (unsigned)(z < L) << 5 | (unsigned)in << 6;
}
__host__ __device__ constexpr unsigned cnn_need(int o) {
    return o >= 27 ? 128u
                   : 64u | (o % 3 == 0 ? 1u : 0u) | (o % 3 == 2 ? 2u : 0u) | ((o / 3) % 3 == 0 ? 4u : 0u) |
                         ((o / 3) % 3 == 2 ? 8u : 0u) | (o / 9 == 0 ? 16u : 0u) | (o / 9 == 2 ? 32u : 0u);
}

template <int L>
__device__ __forceinline__ int cnn_shift(int o) {
    constexpr int N1 = L + 1;
    return (o / 9 - 1) * N1 * N1 + ((o / 3) % 3 - 1) * N1 + (o % 3 - 1);
}

// node n = lidx(x, y, z) on a haloed grid with line stride SY and plane stride SZ;
// cnn_pshift(o): offset o there (0 for the zero-weight padding offsets o >= 27, which then read
// the node itself)
template <int L, int SY, int SZ>
__device__ __forceinline__ int cnn_pad(int n) {
    constexpr int N1 = L + 1;
    const int x = n % N1, y = (n / N1) % N1, z = n / (N1 * N1);
    return (x + 1) + (y + 1) * SY + (z + 1) * SZ;
}
template <int SY, int SZ>
__device__ __forceinline__ int cnn_pshift(int o) {
    return o >= 27 ? 0 : (o / 9 - 1) * SZ + ((o / 3) % 3 - 1) * SY + (o % 3 - 1);
}

// 4 channels (4g .. 4g+3) of grid point q, as stored from an MFMA D fragment
__device__ __forceinline__ unsigned short *act_quad(unsigned short *a, int NA, int q, int g) {
    return a + (g >> 1) * NA * 8 + q * 8 + 4 * (g & 1);
}

__device__ __forceinline__ mf_u2 relu_pack(const mf_f4 &acc, float sg) {
    mf_u2 o2;
    o2[0] = bf_pack(fmaxf(sg * acc[0], 0.f), fmaxf(sg * acc[1], 0.f));
    o2[1] = bf_pack(fmaxf(sg * acc[2], 0.f), fmaxf(sg * acc[3], 0.f));
    return o2;
}

template <int L>
__global__ void __launch_bounds__(512, 2) cnn_infer_kernel(const ptrdiff_t E, const unsigned short *__restrict__ W16,
                                                           const float *__restrict__ zin, float *__restrict__ out) {
    using S = CnnShape<L>;
    constexpr int NP = S::NP, NH = S::NH, NA = S::NA, P1 = S::P1, SY = S::SY, SZ = S::SZ, TPG = S::TPG,
                  NB = (S::NXE + S::THREADS - 1) / S::THREADS;
    extern __shared__ __align__(16) unsigned char cnn_smem[];
    float *zs = (float *)cnn_smem;
    unsigned short *actX = (unsigned short *)(cnn_smem + S::ZS);
    unsigned short *actY = actX + 16 * NA;
    float *P = (float *)actY;
    const ptrdiff_t e = blockIdx.x;
    if (e >= E) return;  // uniform per block
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = S::THREADS / 64;
    const int g = lane >> 4, c = lane & 15;

    // the input on its haloed grid; actX zeroed (the layers write only the interior points, so its
    // halo stays zero for both signs)
    {
        // all of this thread's input loads at once (halo and tail points read the element's first
        // value, a valid address, and store zero)
        constexpr int NBI = (NH + S::THREADS - 1) / S::THREADS;
        float zv[NBI];
#pragma unroll
        for (int b = 0; b < NBI; b++) {
            const int q = tid + b * S::THREADS;
            const int px = q % P1 - 1, py = (q / P1) % P1 - 1, pz = q / (P1 * P1) - 1;
            const bool in = q < NH && (unsigned)px <= (unsigned)L && (unsigned)py <= (unsigned)L &&
                            (unsigned)pz <= (unsigned)L;
            const float v = zin[(size_t)e * S::NXE + (in ? (pz * S::N1 + py) * S::N1 + px : 0)];
            zv[b] = in ? v : 0.f;
        }
#pragma unroll
        for (int b = 0; b < NBI; b++) {
            const int q = tid + b * S::THREADS;
            if (q < NH) zs[q] = zv[b];
        }
    }
    for (int i = tid; i < 2 * NA; i += S::THREADS) ((mf_u4 *)actX)[i] = mf_u4{0u, 0u, 0u, 0u};
    // weights in lane order: layer 1 [64][8], layers 2-3 [14][64][8], layer 4 [2][64][4]
    const mf_u4 w1 = *(const mf_u4 *)(W16 + lane * 8);
    int sh1[8];  // layer 1: lane group g gathers offsets 8g .. 8g+7
#pragma unroll
    for (int j = 0; j < 8; j++) sh1[j] = cnn_pshift<P1, P1 * P1>(8 * g + j);
    const bool hi = (g >> 1) != 0;  // hidden layers: lane groups 2, 3 take the pair's second offset
    float gplus[NB];
    __syncthreads();

    for (int sign = 0; sign < 2; sign++) {
        const float sg = sign ? -1.f : 1.f;
        // ---- layer 1: zs -> actX; actY (P of the previous sign) cleared for layer 2
        for (int i = tid; i < 2 * NA; i += S::THREADS) ((mf_u4 *)actY)[i] = mf_u4{0u, 0u, 0u, 0u};
        for (int t = wave; t < S::T; t += nw) {
            const int n = t * 16 + c;
            const bool real = n < S::NXE;
            const int qz = cnn_pad<L, P1, P1 * P1>(real ? n : 0);
            mf_b8 b;
#pragma unroll
            for (int j = 0; j < 8; j++) b[j] = f2bf(zs[qz + sh1[j]]);
            mf_f4 acc = {0.f, 0.f, 0.f, 0.f};
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mf_b8, w1), b, acc, 0, 0, 0);
            if (real) *(mf_u2 *)act_quad(actX, NA, cnn_pad<L, SY, SZ>(n), g) = relu_pack(acc, sg);
        }
        __syncthreads();
        // ---- layers 2 and 3: actX -> actY -> actX
#pragma unroll 1
        for (int layer = 0; layer < 2; layer++) {
            const unsigned short *ain = layer ? actY : actX;
            unsigned short *aout = layer ? actX : actY;
            const unsigned short *wl = W16 + 512 + layer * 7168;
            mf_u4 w[14];
#pragma unroll
            for (int p = 0; p < 14; p++) w[p] = *(const mf_u4 *)(wl + (p * 64 + lane) * 8);
            // byte addresses: the lane's channel plane plus 16 bytes per grid point
            const unsigned char *plane = (const unsigned char *)(ain + (g & 1) * NA * 8);
            for (int t = TPG * wave; t < S::T; t += TPG * nw) {
                int q[TPG], qb[TPG];
                bool real[TPG];
                mf_f4 acc[TPG];
#pragma unroll
                for (int h = 0; h < TPG; h++) {
                    const int n = (t + h) * 16 + c;
                    real[h] = n < S::NXE;
                    q[h] = cnn_pad<L, SY, SZ>(real[h] ? n : 0);
                    qb[h] = q[h] * 16;
                    acc[h] = mf_f4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int p = 0; p < 14; p++) {
                    const int shb = 16 * (hi ? cnn_pshift<SY, SZ>(2 * p + 1) : cnn_pshift<SY, SZ>(2 * p));
                    mf_u4 bv[TPG];
#pragma unroll
                    for (int h = 0; h < TPG; h++) bv[h] = *(const mf_u4 *)(plane + qb[h] + shb);
#pragma unroll
                    for (int h = 0; h < TPG; h++)
                        acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mf_b8, w[p]),
                                                                          __builtin_bit_cast(mf_b8, bv[h]), acc[h], 0,
                                                                          0, 0);
                }
#pragma unroll
                for (int h = 0; h < TPG; h++)
                    if (real[h]) *(mf_u2 *)act_quad(aout, NA, q[h], g) = relu_pack(acc[h], 1.f);
            }
            __syncthreads();
        }
        // ---- layer 4 in two passes of 16 offsets: P[r][n] = sum_ci W4[ci][16 pass + r] act[ci][n],
        // then v[n] += sum_r P[r][n + off_{16 pass + r}]
        float v[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) v[i] = 0.f;
#pragma unroll
        for (int pass = 0; pass < 2; pass++) {
            const mf_u2 w4 = *(const mf_u2 *)(W16 + 512 + 2 * 7168 + pass * 256 + lane * 4);
            for (int t = wave; t < S::T; t += nw) {
                const int n = t * 16 + c;
                const bool real = n < S::NXE;
                const mf_u2 ld = *(const mf_u2 *)act_quad(actX, NA, cnn_pad<L, SY, SZ>(real ? n : 0), g);
                const mf_u2 bv = real ? ld : mf_u2{0u, 0u};  // padding nodes: P[r][n] = 0
                mf_f4 a = {0.f, 0.f, 0.f, 0.f};
                a = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(mf_s4, w4), __builtin_bit_cast(mf_s4, bv),
                                                               a, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) P[(4 * g + r) * NP + n] = a[r];
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NB; i++) {
                const int n = tid + i * S::THREADS;
                if (n < S::NXE) {
                    const unsigned na = ~cnn_avail<L>(n % S::N1, (n / S::N1) % S::N1, n / (S::N1 * S::N1), true);
                    // missing neighbours add P[r][NXE] == 0 (the padding node's product)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int k = 16 * pass + r;
                        if (k < 27) v[i] += P[r * NP + ((cnn_need(k) & na) == 0 ? n + cnn_shift<L>(k) : S::NXE)];
                    }
                }
            }
            __syncthreads();  // P is rewritten by the next pass / sign
        }
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int n = tid + i * S::THREADS;
            if (n < S::NXE) {
                if (sign == 0)
                    gplus[i] = v[i];
                else
                    out[(size_t)e * S::NXE + n] = gplus[i] - v[i];
            }
        }
    }
}

template <int L>
static int launch_cnn_infer(ptrdiff_t E, const uint16_t *W16, const float *z, float *out, hipStream_t s) {
    using S = CnnShape<L>;
    static bool attr = false;
    if (!attr) {
        SFEM_AMD_HIP_CHECK(
            hipFuncSetAttribute((const void *)cnn_infer_kernel<L>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::LDS));
        attr = true;
    }
    cnn_infer_kernel<L><<<(unsigned)E, S::THREADS, S::LDS, s>>>(E, (const unsigned short *)W16, z, out);
    SFEM_AMD_HIP_CHECK(hipGetLastError());
    return SFEM_SUCCESS;
}

int cnn_infer_mfma(int L, ptrdiff_t E, const uint16_t *W16, const float *z, float *out, hipStream_t s) {
    if (E == 0) return SFEM_SUCCESS;
    switch (L) {
        case 1: return launch_cnn_infer<1>(E, W16, z, out, s);
        case 2: return launch_cnn_infer<2>(E, W16, z, out, s);
        case 3: return launch_cnn_infer<3>(E, W16, z, out, s);
        case 4: return launch_cnn_infer<4>(E, W16, z, out, s);
        case 5: return launch_cnn_infer<5>(E, W16, z, out, s);
        case 6: return launch_cnn_infer<6>(E, W16, z, out, s);
        case 7: return launch_cnn_infer<7>(E, W16, z, out, s);
        case 8: return launch_cnn_infer<8>(E, W16, z, out, s);
        default: set_last_error("cnn_infer_mfma: level must be 1..8"); return SFEM_FAILURE;
    }
}

}  // namespace sfem_amd
