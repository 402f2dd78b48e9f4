// mlp_kernels.hip -- the chemistry surrogate network on gfx950: FP32 training kernels and a
// BF16 MFMA inference kernel (no counterpart in the reference).
//
// Network: x[n_in] -> (W_l x + b_l, GELU) for the hidden layers of width H -> W_out h + b_out,
// with GELU in its tanh form (Hendrycks & Gimpel 2016):
//   GELU(z) = z/2 (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3))) = z / (1 + exp(-2 u)),
//   u = sqrt(2/pi) (z + 0.044715 z^3).
//
// Inference keeps a wave's 16 cells in registers through every layer.  Each layer is
// computed transposed, Y^T = W X^T, with v_mfma_f32_16x16x32_bf16:
//   A operand (16 x 32) = a 16-row block of W,  lane l holds A[l%16][slot (l/16, j)], j < 8
//   B operand (32 x 16) = 32 inputs x 16 cells,  lane l holds B[slot (l/16, j)][l%16]
//   D (16 x 16) = 16 outputs x 16 cells,          lane l holds D[4 (l/16) + i][l%16], i < 4
// The sum over K pairs slot (g, j) of A with slot (g, j) of B, so any assignment of input
// indices to slots works if A and B agree.  The B fragment of k-step s of the next layer is
// taken straight from this layer's D registers of row blocks 2s and 2s+1 (after bias, GELU
// and rounding to BF16): slot (g, j) holds input 32 s + 4 g + j for j < 4 and
// 32 s + 16 + 4 g + (j - 4) for j >= 4.  The packed weights of that layer use the same slot
// map, so activations never leave registers.  The first layer's slots are k = 8 g + j over
// the zero-padded inputs.  Packed fragments are 64 lanes x 8 BF16 = 1 KiB, one 16-byte load
// per lane.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "mlp_launch.hpp"

namespace gdtk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

constexpr float GELU_K = 0.7978845608028654f;   // sqrt(2/pi)
constexpr float GELU_C = 0.044715f;
// The same function for inference: z / (1 + 2^(z (A + B z^2))) with the hardware exp2 and
// reciprocal (A = -2 log2(e) sqrt(2/pi), B = 0.044715 A); the result is rounded to BF16.
__device__ __forceinline__ float gelu_fast(float z) {
    constexpr float A = -2.0f * 1.4426950408889634f * 0.7978845608028654f;
    constexpr float B = 0.044715f * A;
    const float w = z * fmaf(B, z * z, A);
    return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(w));
}

// FP32 -> BF16, round to nearest even (finite inputs).
__device__ __forceinline__ unsigned short f2bf(float f) {
    unsigned int u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

// Slot map of layer inputs: k-step s, lane group g, element j -> input index.
__device__ __host__ inline int slot_first(int s, int g, int j) { return 32 * s + 8 * g + j; }
__device__ __host__ inline int slot_chain(int s, int g, int j) { return 32 * s + (j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4)); }

//---------------------------------------------------------------------------------
// Lane-layout probe: D = A B for one 16x32 A and 32x16 B (row-major FP32 inputs, exact in
// BF16), through the MFMA instruction and the slot map above with slots k = 8 g + j.
__global__ void k_mfma_probe(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ D) {
    const int l = threadIdx.x;
    const int r = l & 15, g = l >> 4;
    u16x8 a, b;
    for (int j = 0; j < 8; ++j) {
        a[j] = f2bf(A[r * 32 + slot_first(0, g, j)]);
        b[j] = f2bf(B[slot_first(0, g, j) * 16 + r]);
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0,
                                                  0, 0);
    for (int i = 0; i < 4; ++i) D[(4 * g + i) * 16 + r] = acc[i];
}

hipError_t launch_mfma_probe(const float* A, const float* B, float* D, hipStream_t s) {
    hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, s, A, B, D);
    return hipGetLastError();
}

//---------------------------------------------------------------------------------
// Packing of FP32 weights W[out][in] (row-major) into BF16 fragments:
// frag[((rb * nks) + s) * 64 + lane][j] = W[16 rb + l%16][slot(s, l/16, j)], zero outside.
__global__ void k_mlp_pack(const float* __restrict__ W, int n_out, int n_in, int nrb, int nks, int chain,
                           unsigned short* __restrict__ frag) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int total = nrb * nks * 64 * 8;
    if (t >= total) return;
    const int j = t & 7, lane = (t >> 3) & 63, fs = t >> 9;
    const int s = fs % nks, rb = fs / nks;
    const int row = 16 * rb + (lane & 15), g = lane >> 4;
    const int k = chain ? slot_chain(s, g, j) : slot_first(s, g, j);
    const float v = (row < n_out && k < n_in) ? W[(size_t)row * n_in + k] : 0.0f;
    frag[t] = f2bf(v);
}

hipError_t launch_mlp_pack(const float* W, int n_out, int n_in, int chain, unsigned short* frag, hipStream_t s) {
    const int nrb = (n_out + 15) / 16, nks = (n_in + 31) / 32;
    const int total = nrb * nks * 64 * 8;
    hipLaunchKernelGGL(k_mlp_pack, dim3((total + 255) / 256), dim3(256), 0, s, W, n_out, n_in, nrb, nks, chain, frag);
    return hipGetLastError();
}

//---------------------------------------------------------------------------------
// Inference: x SoA [n_in][n] FP32 -> y SoA [n_out][n] FP32.  H hidden width (multiple of
// 32), NH hidden layers, n_in <= 32, n_out <= 16.  frag: packed layers in order; bias:
// FP32 biases in order.
//
// A workgroup of 8 waves (4 for H = 64) has 16 cells a wave.  The H x H layers stream their
// fragments through LDS two k-steps at a time (32 KiB for H = 256), loaded straight to LDS and
// double-buffered: one barrier a stage, the next stage's loads under this one's products.  The
// small first and last layers read their fragments from global memory (L2).  The sums start
// from the biases.
//
// GELU bounds it: per 16 x 16 block a third more vector cycles (two transcendental
// instructions a value) than the matrix cores need, and each of them waits for the other
// within a wave.  So the registers are held to 128 a wave (16 cells, not 32, and scalar
// addresses), for four waves a SIMD that fill each other's gaps: 2^19 cells through the
// 3 x 256 network in 239 us with the matrix cores busy for 60, against 432 us with one wave
// a SIMD of 32 cells each and 275 with two.
// count (may be null): the number of leading cells to evaluate, read from device memory (at
// most n, the arrays' stride); workgroups past it exit at once.
template <int H, int NH, int WAVES, int CB>
__global__ __launch_bounds__(64 * WAVES, 4) void k_mlp_infer(const float* __restrict__ x, int n_in, int n,
                                                      const unsigned* __restrict__ count,
                                                      const unsigned short* __restrict__ frag,
                                                      const float* __restrict__ bias, int n_out, float* __restrict__ y) {
    constexpr int CELLS = WAVES * CB * 16;
    const int stride = n;
    if (count) {
        const unsigned c = *count;
        n = (c < (unsigned)n) ? (int)c : n;
        if ((int64_t)blockIdx.x * CELLS >= n) return;
    }
    constexpr int NRB = H / 16, NKS = H / 32;
    constexpr int KS = 2;                                   // k-steps per stage
    constexpr int FRAG_PER_STEP = KS * NRB * 64;            // 16-byte fragments per stage
    constexpr int LOADS = FRAG_PER_STEP / (64 * WAVES);      // per thread
    static_assert(FRAG_PER_STEP % (64 * WAVES) == 0, "k-step fragments must split over the workgroup");
    __shared__ bf16x8 lds[2][FRAG_PER_STEP];
    __shared__ alignas(16) float bias_s[NH * H + 16];
    static_assert(__alignof__(bias_s) >= sizeof(f32x4), "read four biases at a time");
    for (int k = threadIdx.x; k < NH * H + n_out; k += 64 * WAVES) bias_s[k] = bias[k];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int cell0 = blockIdx.x * CELLS + wave * (CB * 16);
    const bf16x8* F = reinterpret_cast<const bf16x8*>(frag);
    const unsigned lane16 = 16 * lane;
    auto frag_at = [lane16](const bf16x8* f) {  // scalar base, 32-bit lane offset
        typedef const __attribute__((address_space(1))) char* gptr;
        return *(const __attribute__((address_space(1))) bf16x8*)((gptr)f + lane16);
    };

    bf16x8 act[CB][NKS];
    f32x4 acc[CB][NRB];
    // first layer: one k-step over the zero-padded inputs (slots k = 8 g + j)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        const int cell = cell0 + cb * 16 + r;
        u16x8 xb;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = 8 * g + j;
            xb[j] = (cell < n && k < n_in) ? f2bf(x[(size_t)k * stride + cell]) : (unsigned short)0;
        }
        act[cb][0] = __builtin_bit_cast(bf16x8, xb);
    }
    // the sums start from the biases: accumulator i of row block rb is row 16 rb + 4 g + i
    const float* bl = bias_s;
    auto start = [&] {
#pragma unroll
        for (int rb = 0; rb < NRB; ++rb) {
            const f32x4 b = *reinterpret_cast<const f32x4*>(bl + 16 * rb + 4 * g);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) acc[cb][rb] = b;
        }
        bl += H;
    };
    // k-step s of a layer: fragments Fl[(rb * NKS + s) * 64 + lane], rb < NRB, straight to LDS
    const bf16x8* Fl = F + NRB * 64;
    auto stage = [&](int s, int buf) {
#pragma unroll
        for (int q = 0; q < LOADS; ++q) {
            const int f = WAVES * q + wave, rb = f / KS, k = f % KS;
            const bf16x8* src = Fl + (rb * NKS + KS * s + k) * 64;
            asm("" : "+s"(src));  // stays a scalar base: lane addresses kept over the loop spill
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(
                    (const __attribute__((address_space(1))) char*)src + lane16),
                (__attribute__((address_space(3))) void*)(&lds[buf][f * 64]), 16, 0, 0);
        }
    };
    // this wave's loads have landed (s_waitcnt vmcnt(0)), then everybody's
    auto staged = [&] {
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
    };
    if (NH > 1) stage(0, 0);
    __syncthreads();  // biases in LDS
    start();
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb) {
        const bf16x8 a = frag_at(F + rb * 64);
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
            acc[cb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, act[cb][0], acc[cb][rb], 0, 0, 0);
        if (rb % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll 1
    for (int layer = 0; layer < NH; ++layer) {
        // GELU + BF16 -> B fragments of the next layer
#pragma unroll
        for (int s = 0; s < NKS; ++s)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                bf16x8 v;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = (__bf16)gelu_fast(acc[cb][2 * s][i]);
                    v[4 + i] = (__bf16)gelu_fast(acc[cb][2 * s + 1][i]);
                }
                act[cb][s] = v;
                __builtin_amdgcn_sched_barrier(0);
            }
        if (layer == NH - 1) break;
        start();
#pragma unroll
        for (int s = 0; s < NKS / KS; ++s) {
            const int buf = (NKS / KS == 1) ? layer & 1 : s & 1;
            staged();
            if (s + 1 < NKS / KS) {
                stage(s + 1, buf ^ 1);
            } else {
                Fl += NRB * NKS * 64;
                if (layer + 2 < NH) stage(0, buf ^ 1);
            }
#pragma unroll
            for (int rb = 0; rb < NRB; ++rb) {
#pragma unroll
                for (int k = 0; k < KS; ++k) {
                    const bf16x8 a = lds[buf][(rb * KS + k) * 64 + lane];
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb)
                        acc[cb][rb] =
                            __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, act[cb][KS * s + k], acc[cb][rb], 0, 0, 0);
                }
                if (rb % 2 == 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // output layer: one 16-row block, fragments from global
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NKS; ++s) o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag_at(Fl + s * 64), act[cb][s], o, 0, 0, 0);
        const int cell = cell0 + cb * 16 + r;
        if (cell < n) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 4 * g + i;
                if (row < n_out) y[(size_t)row * stride + cell] = o[i] + bl[row];
            }
        }
    }
}

hipError_t launch_mlp_infer(int H, int NH, const float* x, int n_in, int n, const unsigned short* frag,
                            const float* bias, int n_out, float* y, hipStream_t s, const unsigned* count) {
    if (n <= 0) return hipSuccess;
    auto grid = [n](int cells) { return dim3((unsigned)(((int64_t)n + cells - 1) / cells)); };
    if (H == 256 && NH == 3) {
        hipLaunchKernelGGL((k_mlp_infer<256, 3, 8, 1>), grid(128), dim3(512), 0, s, x, n_in, n, count, frag, bias,
                           n_out, y);
    } else if (H == 64 && NH == 2) {
        hipLaunchKernelGGL((k_mlp_infer<64, 2, 4, 1>), grid(64), dim3(256), 0, s, x, n_in, n, count, frag, bias,
                           n_out, y);
    } else {
        return hipErrorNotSupported;
    }
    return hipGetLastError();
}

//---------------------------------------------------------------------------------
// Training in FP32: three launches a batch.
//
// k_mlp_pass carries 16 cells through every layer and back: forward, squared error and its
// gradient, and the gradients dZ_l with respect to each layer's pre-activations.  Layers are
// computed transposed, Y^T = W X^T, on v_mfma_f32_16x16x4_f32 (FP32 operands, products and
// sums):
//   A operand (16 x 4): lane l holds A[l%16][slot l/16];  B operand (4 x 16): B[slot l/16][l%16];
//   D (16 x 16): lane l holds D[4 (l/16) + i][l%16], i < 4.
// With slot g of step (rb, i) standing for input 16 rb + 4 g + i, the four D registers of a
// row block are the B operands of the next layer's four steps over it, and the A operands of
// those steps are four consecutive weights of one row: one 16-byte load.  The waves share the
// output rows; what each of them has computed goes to the others through LDS in the register
// layout (16-byte reads and writes, no bank conflict).  The weights come from L2 a window of WN
// row blocks ahead of their use, across the products too, under the matrix instructions.  They
// are kept packed in operand order for both directions (k_mlp_update writes them with the
// parameters), 1 KiB without gaps a load: from the rows themselves, 16 of them 1 KiB apart, the
// same bytes arrived at a fifth of the rate.  The
// layers are passes of one loop: unrolled, the code ran through the instruction cache once,
// and waiting for its lines took longer than the work.  38 us for a batch of 4096, of which
// the matrix cores are busy 14; a whole training step 645 -> 75 us against one launch per
// product on the vector units and separate passes for bias, activation, sums and Adam.
//
// Activations and dZ are kept as [cell block][row][16 cells], which both this kernel's stores
// and k_mlp_weight_grad's 16-byte loads read and write without gaps.
constexpr int TC = 16;  // cells per block

// bias + GELU's value and derivative.  With s = 1 / (1 + exp(-2 u)) = (1 + tanh u) / 2:
// GELU(z) = z s and GELU'(z) = s + 2 z s (1 - s) u'(z), from one exponential.
__device__ __forceinline__ float gelu_pair(float z, float& grad) {
    const float z2 = z * z;
    const float u2 = 2.0f * GELU_K * (z + GELU_C * z2 * z);
    const float s = 1.0f / (1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * u2));
    grad = s + 2.0f * z * s * (1.0f - s) * (GELU_K * (1.0f + 3.0f * GELU_C * z2));
    return z * s;
}

__device__ __forceinline__ float round_bf16(float f) { return __uint_as_float((unsigned)f2bf(f) << 16); }

// Element i past a wave-uniform address, as T: scalar base, 32-bit lane offset.
template <class T>
__device__ __forceinline__ T ld_at(const float* base, unsigned i) {
    typedef __attribute__((address_space(1))) const char* gptr;
    typedef __attribute__((address_space(1))) const T* tptr;
    return *(tptr)((gptr)base + i * 4u);
}
__device__ __forceinline__ void st_at(float* base, unsigned i, float v) {
    typedef __attribute__((address_space(1))) char* gptr;
    typedef __attribute__((address_space(1))) float* tptr;
    *(tptr)((gptr)base + i * 4u) = v;
}

// WAVES waves share the H rows.  GRAD: 0 forward only (net.y_out), 1 with the backward pass.
template <int H, int NH, int WAVES, int GRAD>
__global__ __launch_bounds__(64 * WAVES, 2) void k_mlp_pass(MlpPass net) {
    constexpr int NRB = H / 16, OB = NRB / WAVES, WN = 4;
    static_assert(OB * WAVES == NRB, "row blocks must split over the waves");
    __shared__ f32x4 hs[2][NRB * 64];
    __shared__ f32x4 ys[WAVES * 64];
    __shared__ float xs[2 * 16 * TC];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int ob0 = wave * OB;  // this wave's first row block
    const unsigned rowoff = r * H + 4 * g, coloff = 4 * g * H + r, celloff = 4 * g * TC + r;
    const size_t blk = blockIdx.x;
    const size_t cell = blk * TC + r;
    const bool live = cell < (size_t)net.B;
    const int nrb0 = (net.n_in + 15) >> 4;  // 1 or 2

    // window q of the packed weights of a product (operand_at)
    f32x4 w[OB][WN];
    auto window = [&](const float* M, int q) {
#pragma unroll
        for (int ob = 0; ob < OB; ++ob)
#pragma unroll
            for (int j = 0; j < WN; ++j)
                w[ob][j] = ld_at<f32x4>(M + ((ob0 + ob) * NRB + q * WN + j) * 256, 4 * lane);
    };
    f32x4 acc[OB], h[OB], gp[NH][OB];
    // acc = M (the rows in hs[buf]); the first window of M is in w, and next's is afterwards
    auto product = [&](const float* M, const float* next, int buf) {
#pragma unroll
        for (int ob = 0; ob < OB; ++ob) acc[ob] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int q = 0; q < NRB / WN; ++q) {
            f32x4 cur[OB][WN], b[WN];
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                b[j] = hs[buf][(q * WN + j) * 64 + lane];
#pragma unroll
                for (int ob = 0; ob < OB; ++ob) cur[ob][j] = w[ob][j];
            }
            const bool last = q + 1 == NRB / WN;
            window(last ? next : M, last ? 0 : q + 1);
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int ob = 0; ob < OB; ++ob)
                        acc[ob] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur[ob][j][i], b[j][i], acc[ob], 0, 0, 0);
        }
    };
    window(net.Wf[1], 0);

    for (int e = threadIdx.x; e < 16 * TC * nrb0; e += 64 * WAVES) {
        const int k = e / TC;
        const size_t c = blk * TC + e % TC;
        float v = 0.0f;
        if (k < net.n_in && c < (size_t)net.B) {
            const size_t row = net.idx ? (size_t)net.idx[c] : c;
            v = net.x[(size_t)k * net.xk + row * net.xc];
            if (net.bf16) v = round_bf16(v);
        }
        xs[e] = v;
        if (GRAD) net.act[0][blk * (16 * TC * nrb0) + e] = v;
    }
    f32x4 yt = {0.f, 0.f, 0.f, 0.f};
    if (GRAD && live) {
        const size_t row = net.idx ? (size_t)net.idx[cell] : cell;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * g + i < net.n_out) yt[i] = net.y[(size_t)(4 * g + i) * net.yk + row * net.yc];
    }
    __syncthreads();

#pragma unroll
    for (int ob = 0; ob < OB; ++ob) acc[ob] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int rb = 0; rb < nrb0; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * rb + 4 * g + i;
            const float b = xs[k * TC + r];
#pragma unroll
            for (int ob = 0; ob < OB; ++ob) {
                const float a = (k < net.n_in) ? net.W[0][(16 * (ob0 + ob) + r) * net.n_in + k] : 0.0f;
                acc[ob] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc[ob], 0, 0, 0);
            }
        }
#pragma unroll 1
    for (int l = 0; l < NH; ++l) {
        // layer l: acc -> h, and on to the other waves
        f32x4 gl[OB];
#pragma unroll
        for (int ob = 0; ob < OB; ++ob) {
            const f32x4 bias = ld_at<f32x4>(net.b[l] + 16 * (ob0 + ob), 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float grad;
                float v = gelu_pair(acc[ob][i] + bias[i], grad);
                gl[ob][i] = grad;
                if (net.bf16) v = round_bf16(v);
                h[ob][i] = v;
                if (GRAD) st_at(net.act[l + 1] + (blk * H + 16 * (ob0 + ob) + i) * TC, celloff, v);
            }
            hs[l & 1][(ob0 + ob) * 64 + lane] = h[ob];
        }
        if (GRAD)
#pragma unroll
            for (int q = 0; q < NH; ++q)
                if (q == l)
#pragma unroll
                    for (int ob = 0; ob < OB; ++ob) gp[q][ob] = gl[ob];
        if (l + 1 == NH) break;
        __syncthreads();
        product(net.Wf[l + 1], (l + 2 < NH) ? net.Wf[l + 2] : GRAD ? net.Wb[NH - 1] : net.Wf[1], l & 1);
    }
    // Output layer: every wave's share of the sum over its own rows, added in the waves' order.
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ob = 0; ob < OB; ++ob) {
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
        if (r < net.n_out) a = ld_at<f32x4>(net.W[NH] + 16 * (ob0 + ob), rowoff);
#pragma unroll
        for (int i = 0; i < 4; ++i) o = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], h[ob][i], o, 0, 0, 0);
    }
    ys[wave * 64 + lane] = o;
    __syncthreads();
    o = ys[lane];
#pragma unroll
    for (int v = 1; v < WAVES; ++v) o += ys[v * 64 + lane];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (4 * g + i < net.n_out) o[i] += net.b[NH][4 * g + i];
    if (!GRAD) {
        if (wave == 0 && live)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * g + i < net.n_out) net.y_out[cell * net.n_out + 4 * g + i] = o[i];
        return;
    }
    // Mean-squared error and its gradient
    const float count = (float)((size_t)net.B * net.n_out);
    f32x4 dy = {0.f, 0.f, 0.f, 0.f};
    float e = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (live && 4 * g + i < net.n_out) {
            const float d = o[i] - yt[i];
            dy[i] = 2.0f * d / count;
            e += d * d;
        }
    if (wave == 0) {
#pragma unroll
        for (int q = 32; q > 0; q >>= 1) e += __shfl_xor(e, q);
        if (lane == 0) net.loss[blk] = e;
#pragma unroll
        for (int i = 0; i < 4; ++i) st_at(net.dz[NH] + (blk * 16 + i) * TC, celloff, dy[i]);
    }
#pragma unroll
    for (int ob = 0; ob < OB; ++ob) acc[ob] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int ob = 0; ob < OB; ++ob) {
            const float a = (4 * g + i < net.n_out) ? ld_at<float>(net.W[NH] + i * H + 16 * (ob0 + ob), coloff) : 0.0f;
            acc[ob] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, dy[i], acc[ob], 0, 0, 0);
        }
#pragma unroll 1
    for (int l = NH - 1; l >= 0; --l) {
        // dA_l in acc -> dZ_l
#pragma unroll
        for (int ob = 0; ob < OB; ++ob) {
            f32x4 gl = gp[0][ob];
#pragma unroll
            for (int q = 1; q < NH; ++q)
                if (q == l) gl = gp[q][ob];
            const f32x4 d = acc[ob] * gl;
#pragma unroll
            for (int i = 0; i < 4; ++i) st_at(net.dz[l] + (blk * H + 16 * (ob0 + ob) + i) * TC, celloff, d[i]);
            hs[l & 1][(ob0 + ob) * 64 + lane] = d;
        }
        if (l == 0) break;
        __syncthreads();
        product(net.Wb[l], net.Wb[l > 1 ? l - 1 : l], l & 1);
    }
}

int mlp_blocks(int B) { return (B + TC - 1) / TC; }

hipError_t launch_mlp_pass(int H, int NH, const MlpPass& net, int grad, hipStream_t s) {
    const dim3 grid((unsigned)mlp_blocks(net.B));
    if (H == 256 && NH == 3) {
        if (grad) hipLaunchKernelGGL((k_mlp_pass<256, 3, 8, 1>), grid, dim3(512), 0, s, net);
        else hipLaunchKernelGGL((k_mlp_pass<256, 3, 8, 0>), grid, dim3(512), 0, s, net);
    } else if (H == 64 && NH == 2) {
        if (grad) hipLaunchKernelGGL((k_mlp_pass<64, 2, 4, 1>), grid, dim3(256), 0, s, net);
        else hipLaunchKernelGGL((k_mlp_pass<64, 2, 4, 0>), grid, dim3(256), 0, s, net);
    } else {
        return hipErrorNotSupported;
    }
    return hipGetLastError();
}

// dW_l[o][k] = sum_b dZ_l[b][o] A_{l-1}[b][k] and db_l[o] = sum_b dZ_l[b][o], every layer in one
// launch.  A workgroup has one 64 x 64 tile of one layer over one share of the batch, each of
// its eight waves one half of the tile over a quarter of that share: 6 loads of 16 bytes feed
// 32 matrix instructions, and no LDS but to add the quarters in their order.  The
// shares' sums go to parts[share][parameter]; k_mlp_update adds them in order, so results do
// not depend on the scheduling.  The large tiles come first, one to a
// CU, the narrow first and last layers' behind them.  21 us for a batch of 4096 of the
// 3 x 256 network, 8 of them matrix instructions; more shares (8 to 16) or three cell blocks
// ahead took 21 to 30.
constexpr int WG_AHEAD = 2;  // cell blocks loaded ahead: the rows come from beyond L2, ~1 us
__global__ __launch_bounds__(512, 4) void k_mlp_weight_grad(MlpPass net, int nlayer, int nblk, int nsplit,
                                                            size_t nparam, float* __restrict__ parts) {
    __shared__ f32x4 red[4][16 * 64];
    __shared__ float redb[4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int quarter = wave >> 1, half = wave & 1;
    const int r = lane & 15, g = lane >> 4;
    const int split = blockIdx.x % nsplit;
    int job = blockIdx.x / nsplit, l = 0, ntk = 1;
    for (int q = 0; q < nlayer; ++q) {  // the grid has exactly the tiles of nlayer layers
        l = (q < nlayer - 2) ? q + 1 : (q == nlayer - 2) ? 0 : nlayer - 1;
        ntk = (net.in_w[l] + 63) >> 6;
        const int n = ((net.out_w[l] + 63) >> 6) * ntk;
        if (job < n) break;
        job -= n;
    }
    const int to = job / ntk, tk = job % ntk;
    const int no = net.out_w[l], ni = net.in_w[l];
    const int po = (no + 15) >> 4, pk = (ni + 15) >> 4;  // row blocks of dZ and of the input
    const int nob = po - 4 * to, nkb = pk - 4 * tk - 2 * half;  // of them in this wave's part
    const float* dz = net.dz[l] + 64 * to * TC;
    const float* in = net.act[l] + (64 * tk + 32 * half) * TC;
    const unsigned off = r * TC + 4 * g;
    const size_t so = (size_t)po * 16 * TC, sk = (size_t)pk * 16 * TC;
    f32x4 acc[4][2];
    float bsum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[p][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int64_t share = (int64_t)split * 4 + quarter, shares = (int64_t)nsplit * 4;
    const int c0 = (int)(share * nblk / shares), c1 = (int)((share + 1) * nblk / shares);
    f32x4 a[WG_AHEAD][4], b[WG_AHEAD][2];
    auto load = [&](int c, f32x4* pa, f32x4* pb) {
        c = (c < c1) ? c : c1 - 1;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            pa[p] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (p < nob) pa[p] = ld_at<f32x4>(dz + c * so + p * 16 * TC, off);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            pb[q] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (q < nkb) pb[q] = ld_at<f32x4>(in + c * sk + q * 16 * TC, off);
        }
    };
    if (c0 < c1)
#pragma unroll
        for (int z = 0; z < WG_AHEAD; ++z) load(c0 + z, a[z], b[z]);
#pragma unroll 1
    for (int c = c0; c < c1; ++c) {
        f32x4 ca[4], cb[2];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            ca[p] = a[0][p];
#pragma unroll
            for (int z = 1; z < WG_AHEAD; ++z) a[z - 1][p] = a[z][p];
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            cb[q] = b[0][q];
#pragma unroll
            for (int z = 1; z < WG_AHEAD; ++z) b[z - 1][q] = b[z][q];
        }
        load(c + WG_AHEAD, a[WG_AHEAD - 1], b[WG_AHEAD - 1]);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            if (p >= nob) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    acc[p][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(ca[p][i], cb[q][i], acc[p][q], 0, 0, 0);
            bsum[p] += (ca[p][0] + ca[p][1]) + (ca[p][2] + ca[p][3]);
        }
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
#pragma unroll
        for (int q = 0; q < 2; ++q) red[quarter][(4 * p + 2 * half + q) * 64 + lane] = acc[p][q];
        float t = bsum[p];
        t += __shfl_xor(t, 16);
        t += __shfl_xor(t, 32);
        if (g == 0 && half == 0) redb[quarter][16 * p + r] = t;
    }
    __syncthreads();
    float* out = parts + (size_t)split * nparam;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int tile = 2 * wave + q, p = tile >> 2, e = tile * 64 + lane;
        const f32x4 t = ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
        const int k = 64 * tk + 16 * (tile & 3) + r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 64 * to + 16 * p + 4 * g + i;
            if (row < no && k < ni) out[net.woff[l] + (size_t)row * ni + k] = t[i];
        }
    }
    if (tk == 0 && threadIdx.x < 64) {
        const int row = 64 * to + threadIdx.x;
        if (row < no)
            out[net.boff[l] + row] =
                ((redb[0][threadIdx.x] + redb[1][threadIdx.x]) + redb[2][threadIdx.x]) + redb[3][threadIdx.x];
    }
}

// Where element (row, k) of an H x H matrix lies in operand order: per row block and k block 64
// lanes with 4 consecutive k of one row each.
__device__ __forceinline__ unsigned operand_at(unsigned row, unsigned k, unsigned H) {
    return (((row / 16) * (H / 16) + k / 16) * 64 + (k % 16) / 4 * 16 + row % 16) * 4 + k % 4;
}
// Parameter i, if it is one of the sqn inner layers' H x H weights (one layer after another from
// parameter sq0 on, each with its H biases behind it), into the layer's operands of the forward
// product and, behind them, of the backward one.
__device__ __forceinline__ void pack_weight(size_t i, float v, int H, size_t sq0, size_t sqn,
                                            float* __restrict__ packed) {
    const unsigned sq = (unsigned)(H * H), per = sq + H;
    if (i < sq0 || i >= sq0 + sqn * per) return;
    const unsigned q = (unsigned)(i - sq0), l = q / per, e = q - l * per;
    if (e >= sq) return;
    float* dst = packed + (size_t)l * 2 * sq;
    dst[operand_at(e / H, e % H, H)] = v;
    dst[sq + operand_at(e % H, e / H, H)] = v;
}

__global__ void k_mlp_operands(size_t n, const float* __restrict__ w, float* __restrict__ packed, int H, size_t sq0,
                               size_t sqn) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) pack_weight(i, w[i], H, sq0, sqn, packed);
}

hipError_t launch_mlp_operands(size_t n, const float* w, float* packed, int H, size_t sq0, size_t sqn,
                               hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_operands, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, w, packed, H, sq0, sqn);
    return hipGetLastError();
}

static int grad_tiles(const MlpPass& net, int nlayer) {
    int n = 0;
    for (int l = 0; l < nlayer; ++l) n += ((net.out_w[l] + 63) / 64) * ((net.in_w[l] + 63) / 64);
    return n;
}

// Shares of the batch: at most one workgroup per CU (40 tiles of the 3 x 256 network by 6), and
// a cell block at least for every quarter.
int mlp_grad_splits(const MlpPass& net, int nlayer, int B) {
    const int tiles = grad_tiles(net, nlayer);
    int z = 240 / (tiles > 0 ? tiles : 1);
    const int most = mlp_blocks(B) / 4;
    z = z > 64 ? 64 : z;
    z = z > most ? most : z;
    return z < 1 ? 1 : z;
}

hipError_t launch_mlp_weight_grad(const MlpPass& net, int nlayer, int nsplit, size_t nparam, float* parts,
                                  hipStream_t s) {
    const dim3 grid((unsigned)(grad_tiles(net, nlayer) * nsplit));
    hipLaunchKernelGGL(k_mlp_weight_grad, grid, dim3(512), 0, s, net, nlayer, mlp_blocks(net.B), nsplit, nparam, parts);
    return hipGetLastError();
}

// g = the shares' sum, then g itself (grads != null) or one step of Adam (Kingma & Ba 2015)
// with bias correction; with wq the weights rounded to BF16 too, and the
// products' operands.
__global__ void k_mlp_update(size_t n, int nsplit, const float* __restrict__ parts, float* __restrict__ grads,
                             float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
                             float* __restrict__ wq, float* __restrict__ packed, int H, size_t sq0, size_t sqn, float lr,
                             float b1, float b2, float eps, float c1, float c2) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float gi = 0.0f;
#pragma unroll 8
    for (int z = 0; z < nsplit; ++z) gi += parts[z * n + i];
    if (grads) {
        grads[i] = gi;
        return;
    }
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    if (wq) {
        pi = round_bf16(pi);
        wq[i] = pi;
    }
    pack_weight(i, pi, H, sq0, sqn, packed);
}

hipError_t launch_mlp_sum_grads(size_t n, int nsplit, const float* parts, float* grads, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_update, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, nsplit, parts, grads,
                       nullptr, nullptr, nullptr, nullptr, nullptr, 0, (size_t)0, (size_t)0, 0.f, 0.f, 0.f, 0.f, 1.f,
                       1.f);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(size_t n, int nsplit, const float* parts, float* p, float* m, float* v, float* wq,
                           float* packed, int H, size_t sq0, size_t sqn, float lr, float b1, float b2, float eps, int t,
                           hipStream_t s) {
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    hipLaunchKernelGGL(k_mlp_update, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, nsplit, parts, nullptr, p,
                       m, v, wq, packed, H, sq0, sqn, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}

// out[i] = BF16(in[i]) (as FP32 values)
__global__ void k_round_bf16(size_t n, const float* __restrict__ in, float* __restrict__ out) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) out[t] = round_bf16(in[t]);
}

hipError_t launch_round_bf16(size_t n, const float* in, float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_round_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, in, out);
    return hipGetLastError();
}

}  // namespace gdtk
