// Learned sshex8 smoother: a per-macro-element 3x3x3 CNN on the (L+1)^3 micro-grid (zero
// padding outside the element).  Training kernels run in FP32 (direct convolution with the
// element's channels staged in LDS); inference runs the fused network on MFMA with BF16
// weights and activations and FP32 accumulation.
//
// Layouts: activations [E][C][nxe] float (node index = lidx), weights [Cout][Cin][27] with
// offset k = (dz+1)*9 + (dy+1)*3 + (dx+1).
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
// One macro element per block of eight waves (two elements for L <= 2), both signs of
// f(z) = g(z) - g(-z) side by side, the element swept plane by plane in z through all four layers: only
// a few planes of each layer live in LDS (65 KB at L = 8, two blocks per CU), and a hidden layer's
// products keep the three output planes that an input plane feeds in registers, so that one read of an
// operand serves three products.
//
// What bounds it: the hidden layers' products (15 per 16 cells, plane and sign at 16 cycles) and their operand
// reads (5 of 1 KB) take about the same time, 13,000 cycles per element at L = 8.  Whole-element layers (14
// products for 14 reads, 141 KB of LDS, one block per CU and nothing to overlap a layer's barriers) took
// 3.14 ms for 32,768 elements of L = 8; this form 1.56-1.64 ms (830-870 TFLOP/s; a large bf16 product
// reaches 1,190 on the same card), of which layers 1 and 4 take 0.2.
//
// A plane is its lines with one halo cell each, LS = L + 2 cells apart, so that the cell after a line's last
// node is a zero for both neighbours; columns of the matrix tiles are consecutive cells (the halo ones
// computed and not stored), so every address is a lane's base plus a constant.  Activations are
// BF16 after the relu, [sign][half of the channels][cell][8]: 16-byte operand reads.
//   layer 1 (1 -> 16):   D[co][n] = sum_{k < 32} W1[co][k] z[n + off_k]: one 16x16x32 product for both signs
//   layers 2, 3:         for each dz: D_dz[co][n] += sum W[co][ci, dz dy dx] act[n + dy dx], K = 32 = two of the
//                        nine (dy, dx) times 16 channels (the tenth is zero)
//   layer 4 (16 -> 1):   D[(dz, dy)][n] = sum W4[ci, dz dy dx] act[n + dx] for each sign, K = 32 = two dx times
//                        16 channels (the fourth dx is zero), rows the nine (dz, dy); the difference of the
//                        signs (formed alike, so f stays exactly odd) goes to a ring in LDS, and
//                        out = the sum of nine rows of three planes.
// Waves 0-3 run layers 1 and 2 and the output, waves 4-7 layers 3 and 4 (a hidden layer's weights stay in
// registers: 15 operands).  In step s: layer 1 plane s, layer 2 takes plane s - 1 and finishes s - 2, layer 3 takes s - 3 and
// finishes s - 4, layer 4 takes s - 5, and plane s - 7 goes out; every stage reads what the step before wrote:
// one barrier per step.
// Lane layouts (64 lanes, g = lane / 16, c = lane % 16), 16x16x32:
//   A: row c, k = 8g + j (j < 8);  B: column c, k = 8g + j;  D: column c, rows 4g + r
typedef __bf16 mf_b8 __attribute__((ext_vector_type(8)));
typedef float mf_f4 __attribute__((ext_vector_type(4)));
typedef unsigned int mf_u4 __attribute__((ext_vector_type(4)));
typedef unsigned int mf_u2 __attribute__((ext_vector_type(2)));
typedef __bf16 mf_b2 __attribute__((ext_vector_type(2)));
typedef float mf_f2 __attribute__((ext_vector_type(2)));

// two floats -> bf16, round to nearest even (gfx950's v_cvt_pk_bf16_f32)
__device__ __forceinline__ unsigned bf_pack(float lo, float hi) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(mf_f2{lo, hi}, mf_b2));
}
__device__ __forceinline__ mf_u2 relu_pack(const mf_f4 &acc, float sg) {
    mf_u2 o2;
    o2[0] = bf_pack(fmaxf(sg * acc[0], 0.f), fmaxf(sg * acc[1], 0.f));
    o2[1] = bf_pack(fmaxf(sg * acc[2], 0.f), fmaxf(sg * acc[3], 0.f));
    return o2;
}
__device__ __forceinline__ mf_f4 mf_mma(const mf_u4 &a, const mf_u4 &b, const mf_f4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mf_b8, a), __builtin_bit_cast(mf_b8, b), c, 0, 0,
                                                   0);
}

template <int L>
struct CnnShape {
    static constexpr int N1 = L + 1, NXE = N1 * N1 * N1, LS = L + 2, REAL = N1 * LS;
    static constexpr int TS = (REAL + 15) / 16;                  // tiles of a plane and sign
    static constexpr int WS = TS >= 2 ? 2 : 1, EPB = 2 / WS;     // waves per sign; elements per block
    static constexpr int TW = (TS + WS - 1) / WS;                // tiles per wave
    static constexpr int COLS = 16 * WS * TW;
    // cells of a plane with the halo around the columns' neighbourhoods; cell p is stored at p + LS + 1
    static constexpr int CELLS = (COLS + 2 * (LS + 1) + 7) / 8 * 8;
    static constexpr int HALF = CELLS * 16, SIGN = 2 * HALF, PLANE = 2 * SIGN, BUF = EPB * PLANE;  // bytes
    // the input: planes PS cells apart, sharing their halo lines
    static constexpr int PS = (L + 2) * LS, OFFZ = PS + LS + 1;
    static constexpr int ZN = (L * PS + COLS - 1 + 2 * OFFZ + 1 + 7) / 8 * 8;
    // layer 4's rows of a plane: a zero line on both sides; rows 4 (mod 8) words apart (bank spread of the
    // stores' row groups); a ring of four planes
    static constexpr int DROW = (REAL + 2 * LS + 7) / 8 * 8 + 4, DPLANE = 9 * DROW;
    static constexpr int STEPS = L + 8, THREADS = 512;
    static constexpr size_t LDS = (size_t)6 * BUF + sizeof(float) * 4 * EPB * DPLANE + 3 * 64 * 16 + 2 * (size_t)EPB * ZN;
};

// The nine (dy, dx) of a hidden layer as five pairs, (dy, -1) with (dy, 0), then (-1, 1) with (0, 1) and
// nothing with (1, 1): the second of a pair lies one cell, or one line, after the first, so a lane needs two
// addresses and constant offsets.
//
// One input plane through a hidden layer.  a, b: the lane's addresses for the first three and the last two
// pairs; o: its store address.  acc[d][h]: output plane zi - 1 + d of tile h.
template <int L>
__device__ __forceinline__ void cnn_hidden(const unsigned char *__restrict__ a, const unsigned char *__restrict__ b,
                                           unsigned char *__restrict__ o, const int zi, const mf_u4 (&w)[15],
                                           const bool (&real)[CnnShape<L>::TW], mf_f4 (&acc)[3][CnnShape<L>::TW]) {
    constexpr int TW = CnnShape<L>::TW, LS = CnnShape<L>::LS;
    if (zi <= L) {
#pragma unroll
        for (int p = 0; p < 5; p++) {
            const unsigned char *q = p < 3 ? a + 16 * ((p - 1) * LS - 1) : b + 16 * (p == 3 ? 1 - LS : 1);
            mf_u4 x[TW];
#pragma unroll
            for (int h = 0; h < TW; h++) x[h] = *(const mf_u4 *)(q + 256 * h);
#pragma unroll
            for (int d = 0; d < 3; d++)
#pragma unroll
                for (int h = 0; h < TW; h++) acc[d][h] = mf_mma(w[(2 - d) * 5 + p], x[h], acc[d][h]);
        }
    }
    if (zi >= 1)
#pragma unroll
        for (int h = 0; h < TW; h++)
            if (real[h]) *(mf_u2 *)(o + 256 * h) = relu_pack(acc[0][h], 1.f);
#pragma unroll
    for (int h = 0; h < TW; h++) {
        acc[0][h] = acc[1][h];
        acc[1][h] = acc[2][h];
        acc[2][h] = mf_f4{0.f, 0.f, 0.f, 0.f};
    }
}

template <int L>
__global__ void __launch_bounds__(512, 4) cnn_infer_kernel(const ptrdiff_t E, const unsigned short *__restrict__ W16,
                                                           const float *__restrict__ zin, float *__restrict__ out) {
    using S = CnnShape<L>;
    constexpr int N1 = S::N1, LS = S::LS, TW = S::TW, EPB = S::EPB;
    extern __shared__ __align__(16) unsigned char cnn_smem[];
    unsigned char *A1 = cnn_smem, *A2 = A1 + 2 * S::BUF, *A3 = A2 + 2 * S::BUF;
    float *D = (float *)(A3 + 2 * S::BUF);
    mf_u4 *WS14 = (mf_u4 *)(D + 4 * EPB * S::DPLANE);
    unsigned short *zs = (unsigned short *)(WS14 + 3 * 64);
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w4 = wave & 3;
    const ptrdiff_t e0 = (ptrdiff_t)blockIdx.x * EPB;

    // zero planes and rows (the stages write real nodes only), the input as bf16 in its halo layout
    for (int i = tid; i < (int)((6 * S::BUF + 16 * EPB * S::DPLANE) / 16); i += S::THREADS)
        ((mf_u4 *)cnn_smem)[i] = mf_u4{0u, 0u, 0u, 0u};
    for (int i = tid; i < EPB * S::ZN; i += S::THREADS) {
        const int el = i / S::ZN, q = i - el * S::ZN - (LS + 1);  // q = (z + 1) PS + y LS + x
        const int z = (q + S::PS) / S::PS - 2, r = (q + S::PS) % S::PS, y = r / LS, x = r % LS;
        const bool in = z >= 0 && z <= L && y <= L && x <= L && e0 + el < E;
        const float v = zin[(size_t)(in ? e0 + el : e0) * S::NXE + (in ? (z * N1 + y) * N1 + x : 0)];
        zs[i] = in ? (unsigned short)bf_pack(v, 0.f) : (unsigned short)0;
    }

    // the A operands of layers 1 and 4, read back where they are used
    for (int i = tid; i < 64 * 3; i += S::THREADS)
        WS14[i] = *(const mf_u4 *)(W16 + (i < 64 ? i * 8 : 512 + 2 * 7680 + (i - 64) * 8));

    // this wave's tiles in the hidden layers
    const int el = EPB == 1 ? 0 : w4 >> 1, sign = EPB == 1 ? w4 >> 1 : w4 & 1;
    const int p0 = (EPB == 1 ? (w4 & 1) * TW * 16 : 0) + c;
    const int base = el * S::PLANE + sign * S::SIGN + (p0 + LS + 1) * 16;
    const int ha = base + (g & 1) * S::HALF + (g >> 1) * 16, hb = base + (g & 1) * S::HALF + (g >> 1) * 16 * LS;
    const int store = base + (g >> 1) * S::HALF + 8 * (g & 1);
    bool real[TW];
#pragma unroll
    for (int h = 0; h < TW; h++) real[h] = p0 + 16 * h < S::REAL && (p0 + 16 * h) % LS <= L;
    mf_u4 w[15];
    const unsigned short *wl = W16 + 512 + (wave >> 2) * 7680;
#pragma unroll
    for (int i = 0; i < 15; i++) w[i] = *(const mf_u4 *)(wl + (i * 64 + lane) * 8);
    mf_f4 acc[3][TW];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int h = 0; h < TW; h++) acc[d][h] = mf_f4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();

    if (wave < 4) {
        // layer 1's gathers: lane groups 0-2 take plane dz = g - 1 without its last offset (dy, dx) = (1, 1),
        // group 3 the three last ones: one address and constant offsets, but for three slots
        const int zc = S::OFFZ + c, za = zc + (g < 3 ? g - 1 : 0) * S::PS;
        int zb[3];
#pragma unroll
        for (int j = 0; j < 3; j++) zb[j] = g < 3 ? za - LS + j - 1 : zc + (j - 1) * S::PS + LS + 1;
        for (int s = 0; s < S::STEPS; s++) {
            if (s <= L)
                for (int t = w4; t < EPB * S::TS; t += 4) {
                    const int le = EPB == 1 ? 0 : t / S::TS, p = (t - le * S::TS) * 16;
                    const unsigned short *q = zs + le * S::ZN + s * S::PS + p;
                    mf_u4 b;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int k0 = 2 * j, k1 = 2 * j + 1;
                        const unsigned lo = k0 < 3 ? q[zb[k0 < 3 ? k0 : 0]] : q[za + (k0 / 3 - 1) * LS + k0 % 3 - 1];
                        const unsigned hi = k1 < 3 ? q[zb[k1 < 3 ? k1 : 0]] : q[za + (k1 / 3 - 1) * LS + k1 % 3 - 1];
                        b[j] = lo | hi << 16;
                    }
                    const mf_f4 a = mf_mma(WS14[lane], b, mf_f4{0.f, 0.f, 0.f, 0.f});
                    unsigned char *o = A1 + (s & 1) * S::BUF + le * S::PLANE + (g >> 1) * S::HALF +
                                       (p + c + LS + 1) * 16 + 8 * (g & 1);
                    if (p + c < S::REAL && (p + c) % LS <= L) {
                        *(mf_u2 *)o = relu_pack(a, 1.f);
                        *(mf_u2 *)(o + S::SIGN) = relu_pack(a, -1.f);
                    }
                }
            if (s >= 1 && s <= L + 2) {
                const unsigned char *in = A1 + ((s - 1) & 1) * S::BUF;
                cnn_hidden<L>(in + ha, in + hb, A2 + (s & 1) * S::BUF + store, s - 1, w, real, acc);
            }
            if (s >= 7) {
                // plane s - 7 from the rows of planes s - 8, s - 7, s - 6
                const int z = s - 7;
                for (int i = tid; i < EPB * S::REAL; i += 256) {
                    const int le = EPB == 1 ? 0 : i / S::REAL, p = i - le * S::REAL, y = p / LS, x = p - y * LS;
                    if (x > L || e0 + le >= E) continue;
                    float v = 0.f;
#pragma unroll
                    for (int dz = -1; dz <= 1; dz++) {
                        if (z + dz < 0 || z + dz > L) continue;
                        const float *r = D + (((z + dz) & 3) * EPB + le) * S::DPLANE + LS + p + (dz + 1) * 3 * S::DROW;
#pragma unroll
                        for (int dy = -1; dy <= 1; dy++) v += r[(dy + 1) * S::DROW + dy * LS];
                    }
                    out[(size_t)(e0 + le) * S::NXE + (z * N1 + y) * N1 + x] = v;
                }
            }
            lds_barrier();
        }
    } else {
        for (int s = 0; s < S::STEPS; s++) {
            if (s >= 5 && s <= L + 5) {
                // plane s - 5 of layer 4's rows
                const mf_u4 wa = WS14[64 + lane], wb = WS14[128 + lane];
                for (int t = w4; t < EPB * S::TS; t += 4) {
                    const int le = EPB == 1 ? 0 : t / S::TS, p = (t - le * S::TS) * 16 + c;
                    // dx = -1 and 0, then 1 and none (the lanes g >= 2 read dx = 1 there too)
                    const unsigned char *q = A3 + ((s - 1) & 1) * S::BUF + le * S::PLANE + (g & 1) * S::HALF +
                                             (p + LS + (g >> 1)) * 16;
                    const unsigned char *q1 = q + (g < 2 ? 32 : 16);
                    mf_f4 d[2];
#pragma unroll
                    for (int sn = 0; sn < 2; sn++) {
                        d[sn] = mf_mma(wa, *(const mf_u4 *)(q + sn * S::SIGN), mf_f4{0.f, 0.f, 0.f, 0.f});
                        d[sn] = mf_mma(wb, *(const mf_u4 *)(q1 + sn * S::SIGN), d[sn]);
                    }
                    const mf_f4 a = d[0] - d[1];
                    float *o = D + (((s - 5) & 3) * EPB + le) * S::DPLANE + LS + p + 4 * g * S::DROW;
                    if (p < S::REAL) {
                        if (g < 3) o[0] = a[0];
                        if (g < 2) o[S::DROW] = a[1], o[2 * S::DROW] = a[2], o[3 * S::DROW] = a[3];
                    }
                }
            }
            if (s >= 3 && s <= L + 4) {
                const unsigned char *in = A2 + ((s - 1) & 1) * S::BUF;
                cnn_hidden<L>(in + ha, in + hb, A3 + (s & 1) * S::BUF + store, s - 3, w, real, acc);
            }
            lds_barrier();
        }
    }
}

template <int L>
static int launch_cnn_infer(ptrdiff_t E, const uint16_t *W16, const float *z, float *out, hipStream_t s) {
    using S = CnnShape<L>;
    if (raise_lds_limit<cnn_infer_kernel<L>>(S::LDS)) return SFEM_FAILURE;
    cnn_infer_kernel<L><<<(unsigned)((E + S::EPB - 1) / S::EPB), S::THREADS, S::LDS, s>>>(E, (const unsigned short *)W16, z,
                                                                                         out);
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
