// mlp_kernels.hip — BF16 MFMA kernels of the far-field surrogate network (gfx950): fused inference,
// and the training step's loss and gradient (three kernels), its Adam update and the packing of
// the weights into MFMA fragment order.
#include <hip/hip_runtime.h>

#include "mlp.hpp"

namespace sirius {

typedef float v16f __attribute__((ext_vector_type(16)));

// FP32 -> BF16, round to nearest even (NaN/Inf pass through)
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// GELU, tanh form: 0.5 z (1 + tanh(u)) = z / (1 + e^{-2u}), u = 0.7978845608 (z + 0.044715 z^3),
// with the hardware base-2 exponential and reciprocal (the same function in training and
// inference)
__device__ __forceinline__ float gelu_f(float z) {
    const float u2 = z * (2.3022081983f + 0.1029432617f * z * z);  // 2u log2(e)
    return z * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-u2));
}
__device__ __forceinline__ float gelu_df(float z) {
    float t = tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z));
    return 0.5f * (1.f + t) + 0.5f * z * (1.f - t * t) * 0.7978845608028654f * (1.f + 3.f * 0.044715f * z * z);
}

// ------------------------------------------------------------------------------------------
// Fused inference: the whole network for a tile of 128 rows in one kernel, with gfx950's
// v_mfma_f32_32x32x16_bf16 (A 32 x 16 and B 16 x 32 BF16 operands, 8 values per lane: lane
// l holds row / column l % 32 and k = 8 (l / 32) .. +7; C 32 x 32 FP32, 16 values per lane:
// column l % 32, rows 8 (r / 4) + 4 (l / 32) + r % 4).
//  - Each layer is computed transposed, H'^T = W H^T: the weights are the A operand (16 bytes per
//    lane, stored in fragment order so that a wave's load for one k-step is one contiguous
//    kilobyte, streamed from L2 MF_AHEAD k-steps ahead of the MFMAs) and the tile's
//    activations the B operand, read from LDS ([128][264] BF16, row = sample; rows padded by 8
//    values so that the 16-byte reads of eight consecutive lanes cover every bank once).
//  - A lane's accumulators then hold, for one sample, runs of four consecutive neurons: the bias
//    + GELU epilogue converts each run to BF16 with the hardware's paired conversion and writes
//    it back to the sample's LDS row with one 8-byte store, between two barriers.
//  - Wave w computes neurons 64 w .. 64 w + 63 for all 128 samples (2 x 4 tiles of 32 x 32, 128
//    accumulator registers).
//  - The output head (256 -> 6) keeps FP32 precision with three BF16 products: the last hidden
//    activation h = hi + lo and the head's weights W = W_hi + W_lo, each split into BF16 parts,
//    and y = W_hi hi + W_lo hi + W_hi lo (the W_lo lo term is below FP32's resolution of y). Each
//    wave multiplies its own 64 neurons straight from its accumulators; the four partial sums of a
//    sample meet in LDS.
// Bound by the vector unit (a GELU is five FP32 instructions at 1.8 ns per SIMD, an exponential and a
// reciprocal at 3.7; 512 per lane and tile with the rest are 10 us, 190 us for 600,001 rows) beside
// 121 us of MFMAs, which the two blocks of a CU overlap in part: 324 us for 600,001 rows (379 with the
// last layer's parts written to LDS and read back, high then low, by the head). Without the GELUs the
// kernel takes 285 us, without the head's former round trip 220. Tried: the two halves of a tile in
// alternate stages, GELU between the other half's MFMAs, with the weights read twice (352 us, 369 for
// this kernel on the same run); 512 threads of 32 neurons (514, 429 then); 256-row tiles (495, 435).
// ------------------------------------------------------------------------------------------
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));

constexpr int MF_ROWS = 128;
constexpr int MF_PITCH = 264;
constexpr int MF_AHEAD = 2;  // k-steps that the weights are fetched ahead (divides 16)

__device__ __forceinline__ v8bf ld8(const uint16_t* p) { return *(const v8bf*)p; }

__global__ __launch_bounds__(256, 2) void k_mlp_fused(MlpFusedArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t act[MF_ROWS * MF_PITCH];
    __shared__ __attribute__((aligned(16))) float bias_s[4 * MLP_H];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int li = lane & 31, lh = lane >> 5;
    for (int e = t; e < 4 * MLP_H; e += 256) bias_s[e] = a.b[e / MLP_H][e % MLP_H];
    const int64_t n = a.n_dev ? (int64_t)*a.n_dev : a.n;
    const int j0 = wave * 64;  // this wave's neurons
    // tiles of 128 rows, grid-stride (the row count may live on the device)
    for (int64_t row0 = (int64_t)blockIdx.x * MF_ROWS; row0 < n; row0 += (int64_t)gridDim.x * MF_ROWS) {
        __syncthreads();  // bias_s written; the previous tile's last reads of act are done
        // layer-0 input: x padded to 16 columns (row r of the tile is x[idx[r]] when gathered)
        for (int e = t; e < MF_ROWS * 16; e += 256) {
            const int r = e >> 4, k = e & 15;
            const int64_t gr = row0 + r;
            float v = 0.f;
            if (k < SIRIUS_MLP_IN && gr < n) v = a.x[(a.idx ? (int64_t)a.idx[gr] : gr) * a.x_stride + k];
            act[r * MF_PITCH + k] = f2bf(v);
        }
        __syncthreads();
        v16f acc[2][4];
        // the accumulators start at the layer's bias (row 8 q + 4 lh + e of tile mt is neuron
        // j0 + 32 mt + 8 q + 4 lh + e)
        auto init_bias = [&](int l) {
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 bb = *(const float4*)&bias_s[l * MLP_H + j0 + mt * 32 + 8 * q + 4 * lh];
#pragma unroll
                    for (int nt = 0; nt < 4; ++nt) {
                        acc[mt][nt][4 * q + 0] = bb.x;
                        acc[mt][nt][4 * q + 1] = bb.y;
                        acc[mt][nt][4 * q + 2] = bb.z;
                        acc[mt][nt][4 * q + 3] = bb.w;
                    }
                }
        };
        // ring of the weights' fragments, MF_AHEAD k-steps ahead of the MFMAs and on across layers (a
        // layer's first fragments are on their way during the previous layer's epilogue). This
        // lane's fragment of k-step ks, row tile mt of a layer: 1024 ks + 512 mt from its wf
        v8bf wq[MF_AHEAD][2];
        const uint32_t wf = 2 * (wave * 16384 + lane * 8);  // bytes
        auto rsrc = [&](int l) { return __builtin_amdgcn_make_buffer_rsrc((void*)a.w[l], 0, 2 * MLP_H * MLP_H, 0x00027000); };
        auto fragment = [&](__amdgpu_buffer_rsrc_t w, int ks, int mt) {
            typedef uint32_t v4u __attribute__((ext_vector_type(4)));
            const v4u u = __builtin_amdgcn_raw_buffer_load_b128(w, wf + 1024 * mt, 2048 * ks, 0);
            return __builtin_bit_cast(v8bf, u);
        };
#pragma unroll
        for (int ks = 0; ks < MF_AHEAD; ++ks)
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) wq[ks][mt] = fragment(rsrc(0), ks, mt);
        init_bias(0);
        {
            v8bf w[2];
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) w[mt] = ld8(a.w0 + (j0 + mt * 32 + li) * 16 + 8 * lh);
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const v8bf hv = ld8(&act[(nt * 32 + li) * MF_PITCH + 8 * lh]);
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[mt], hv, acc[mt][nt], 0, 0, 0);
            }
        }
        // one hidden layer's products: its weights from Wl, the next one's first from Wn
        auto products = [&](int l, __amdgpu_buffer_rsrc_t Wl, __amdgpu_buffer_rsrc_t Wn) {
            init_bias(l);
#pragma unroll
            for (int ks = 0; ks < MLP_H / 16; ++ks) {
                v8bf w[2];
#pragma unroll
                for (int mt = 0; mt < 2; ++mt) w[mt] = wq[ks % MF_AHEAD][mt];
                const int kn = ks + MF_AHEAD;
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
                    wq[ks % MF_AHEAD][mt] = kn < MLP_H / 16 ? fragment(Wl, kn, mt) : fragment(Wn, kn - MLP_H / 16, mt);
#pragma unroll
                for (int nt = 0; nt < 4; ++nt) {
                    const v8bf hv = ld8(&act[(nt * 32 + li) * MF_PITCH + ks * 16 + 8 * lh]);
#pragma unroll
                    for (int mt = 0; mt < 2; ++mt)
                        acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[mt], hv, acc[mt][nt], 0, 0, 0);
                }
            }
        };
        // GELU on runs of four neurons; BF16 back into the sample's LDS row
#pragma unroll 1
        for (int l = 0; l < 3; ++l) {
            if (l > 0) products(l, rsrc(l - 1), rsrc(l));
            __syncthreads();  // every wave has read this layer's input
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int nt = 0; nt < 4; ++nt) {
                        const v4bf hv = {(__bf16)gelu_f(acc[mt][nt][4 * q + 0]), (__bf16)gelu_f(acc[mt][nt][4 * q + 1]),
                                         (__bf16)gelu_f(acc[mt][nt][4 * q + 2]), (__bf16)gelu_f(acc[mt][nt][4 * q + 3])};
                        *(v4bf*)&act[(nt * 32 + li) * MF_PITCH + j0 + mt * 32 + 8 * q + 4 * lh] = hv;
                    }
            __syncthreads();
        }
        products(3, rsrc(2), rsrc(2));
        v8bf w4h[4], w4l[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            w4h[f] = ld8(a.w4h + ((wave * 4 + f) * 64 + lane) * 8);
            w4l[f] = ld8(a.w4l + ((wave * 4 + f) * 64 + lane) * 8);
        }
        __syncthreads();
        // The output head on this wave's 64 neurons, from the accumulators: a lane's runs q and q + 1 of a
        // row tile are 8 neurons of one sample, the B operand of one MFMA whose k order the packed head
        // weights share. y^T: rows 0..7 of the product, lane li's sample, outputs 4 lh + r.
        float* part = (float*)act;  // [wave][sample][6]: every wave has read this layer's input
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            v16f y;
#pragma unroll
            for (int r = 0; r < 16; ++r) y[r] = 0.f;
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                const int mt = f >> 1, q = 2 * (f & 1);
                v8bf hi, lo;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float h = gelu_f(acc[mt][nt][4 * q + e]);
                    hi[e] = (__bf16)h;
                    lo[e] = (__bf16)(h - (float)hi[e]);
                }
                y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w4h[f], hi, y, 0, 0, 0);
                y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w4l[f], hi, y, 0, 0, 0);
                y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w4h[f], lo, y, 0, 0, 0);
            }
            float* p = part + (wave * MF_ROWS + nt * 32 + li) * SIRIUS_MLP_OUT + 4 * lh;
            *(float2*)p = make_float2(y[0], y[1]);
            if (lh == 0) *(float2*)(p + 2) = make_float2(y[2], y[3]);
        }
        __syncthreads();
        const int64_t left = n - row0;
        const int rows = left < MF_ROWS ? (int)left : MF_ROWS;
        for (int e = t; e < rows * SIRIUS_MLP_OUT; e += 256) {
            float v = a.b4[e % SIRIUS_MLP_OUT];
#pragma unroll
            for (int w = 0; w < 4; ++w) v += part[w * MF_ROWS * SIRIUS_MLP_OUT + e];
            a.y[row0 * SIRIUS_MLP_OUT + e] = v;
        }
    }
}

// Grid: one block per tile up to `max_blocks` (two blocks fit a CU), each looping over tiles.
hipError_t launch_mlp_fused(const MlpFusedArgs& a, int64_t cap, int max_blocks, hipStream_t st) {
    if (cap <= 0) return hipSuccess;
    int64_t blocks = (cap + MF_ROWS - 1) / MF_ROWS;
    if (blocks > max_blocks) blocks = max_blocks;
    hipLaunchKernelGGL(k_mlp_fused, dim3((unsigned)blocks), dim3(256), 0, st, a);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Training: loss and gradient of a batch in three kernels.
//
// k_mlp_train runs the whole network forward and backward for 32 samples per block: 8 waves, wave w
// owning neurons 32 w .. 32 w + 31 of each layer. Samples are the rows of each product
// (v_mfma_f32_32x32x16_bf16, A the tile's activations from LDS, B the weights in fragment order),
// so a lane's accumulators hold one neuron j = 32 w + l % 32 for the 16 samples
// 8 q + 4 (l / 32) + e. Packed to BF16 these registers are an operand of the weight-gradient
// product as they stand (8 samples of one neuron): they go to memory as fragments, without a
// transpose. The layer's outputs also go back to LDS, row = sample, for the next layer, and the
// GELU derivatives stay in LDS, 16 per thread and layer, until the backward pass. Each product sums
// its k dimension in ascending order into one accumulator, as the hidden layers of the fused
// inference kernel do. The output head is FP32. The layers are loops and the derivatives' hyperbolic
// tangents are too: a block runs its code once, and unrolled (72 KB of instructions) the kernel
// spent its time fetching them: 61 us against 39 for 8192 rows (one block per CU; what is left is the
// chain of one block: the derivatives' tangents, the barriers and the weights' loads).
// Sums over samples whose result is small (every bias, the head's and the first layer's weights,
// the loss) leave one row of MLP_TILE_COLS partials per tile.
//
// k_mlp_wgrad forms dW_l = gz_l^T h_l of the three 256 x 256 layers from those fragments, split
// over the samples; k_mlp_grad_sum adds the splits and the tiles' rows in a fixed order.
//
// A batch of 8192 rows has 9.8 GFLOP of work and 1.9 MB of inputs and outputs (8 us at the rate of a
// large matrix product): launches, latency and the fragments' traffic bound it. 32 kernels with the
// activations and pre-activations in FP32 in memory took 490 us per call; these take 63 (39 + 10 + 6
// and the launches). 256 rows took 393 us and take 50, 65536 rows take 357.
// ------------------------------------------------------------------------------------------
constexpr int TR_ROWS = MLP_TRAIN_ROWS;
constexpr int TR_THREADS = 512;
constexpr int TR_PITCH = 264;     // BF16 values per LDS row: 16-byte reads of 8 lanes cover every bank once
constexpr int TR_H4_PITCH = 260;  // floats per LDS row of the last hidden activation
static_assert(TR_ROWS == 32 && MLP_H == 256, "one 32 x 32 product per wave and k step");
static_assert(TR_ROWS * TR_H4_PITCH * 4 <= 2 * TR_ROWS * TR_PITCH * 2, "the last activation fits the two tiles");

// The wave's 16 B fragments of a packed 256 x 256 matrix (k_pack_fused), one per k step: `stride`
// BF16 values apart, from this lane's offset on.
__device__ __forceinline__ void load_frags(v8bf wb[16], const uint16_t* p, int stride) {
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) wb[ks] = ld8(p + ks * stride);
}

// acc = A W^T for the tile in LDS and the wave's weight fragments
__device__ __forceinline__ v16f tile_product(const uint16_t* act, const v8bf wb[16], int li, int lh) {
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
        const v8bf a = ld8(act + li * TR_PITCH + 16 * ks + 8 * lh);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, wb[ks], acc, 0, 0, 0);
    }
    return acc;
}

// The wave's 16 values of its neuron column, rounded to BF16: into the LDS tile (row = sample) and
// to memory as the two operand fragments of the weight gradient.
__device__ __forceinline__ void put_tile(const float v[16], uint16_t* act, uint16_t* frag, int j, int lh) {
    __bf16 b[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        b[r] = (__bf16)v[r];
        __builtin_memcpy(act + (8 * (r >> 2) + 4 * lh + (r & 3)) * TR_PITCH + j, &b[r], 2);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        v8bf f;
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = b[8 * s + e];
        *(v8bf*)(frag + s * 64 * 8) = f;
    }
}

// z -> gelu'(z) in place for this thread's 16 values (one of a layer's rows of TR_THREADS values each)
__device__ __forceinline__ void derive(float* zs) {
#pragma unroll 1
    for (int r = 0; r < 16; r += 2) {
        const float z0 = zs[r * TR_THREADS], z1 = zs[(r + 1) * TR_THREADS];
        const float d0 = gelu_df(z0), d1 = gelu_df(z1);
        zs[r * TR_THREADS] = d0;
        zs[(r + 1) * TR_THREADS] = d1;
    }
}

__global__ __launch_bounds__(TR_THREADS) void k_mlp_train(MlpTrainArgs a) {
    // the activations' two tiles; between the forward and the backward pass the last hidden
    // activation in FP32
    __shared__ __attribute__((aligned(16))) uint16_t act[2][TR_ROWS * TR_PITCH];
    // pre-activations, then GELU derivatives of layers 0..2: [r][thread]. The last layer's pass through
    // the tiles' space and stay in registers.
    __shared__ float zs[3][16 * TR_THREADS];
    __shared__ float xs[TR_ROWS][8];          // the BF16 inputs, for the first layer's weight gradient
    __shared__ float ys[TR_ROWS][8];          // outputs
    __shared__ float gys[TR_ROWS][8];         // output gradients
    float* h4s = (float*)&act[0][0];
    static_assert(sizeof(act) >= 16 * TR_THREADS * sizeof(float), "room for the last layer's pre-activations");
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int li = lane & 31, lh = lane >> 5;
    const int j = 32 * w + li;  // this lane's neuron
    const int64_t T = blockIdx.x, row0 = T * TR_ROWS;
    // this lane's place in the packed weights (neuron block w, and column block w of a transpose) and
    // in a layer's fragments
    const int off_f = (w >> 1) * 16384 + (w & 1) * 512 + lane * 8, off_t = w * 8192 + lane * 8;
    const int64_t off_g = ((T * 8 + w) * 2 * 64 + lane) * 8;
    {
        const int r = t >> 4, k = t & 15;
        const int64_t i = row0 + r;
        const uint16_t v = (k < SIRIUS_MLP_IN && i < a.n) ? f2bf(a.x[i * SIRIUS_MLP_IN + k]) : (uint16_t)0;
        act[0][r * TR_PITCH + k] = v;
        if (k < 8) xs[r][k] = __uint_as_float((uint32_t)v << 16);
    }
    const v8bf w0 = ld8(a.w0 + j * 16 + 8 * lh);
    v8bf wb[16];
    load_frags(wb, a.wf + off_f, 1024);
    float h[16];
    __syncthreads();
    // ---- forward: hidden layers ----
    v16f acc;
    float d3[16];  // the last layer's GELU derivatives
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ld8(&act[0][li * TR_PITCH + 8 * lh]), w0, acc, 0, 0, 0);
#pragma unroll 1
    for (int l = 0;; ++l) {
        const float bias = a.b[l][j];
        float* z = (l < 3 ? zs[l] : h4s) + t;
        if (l == 3) __syncthreads();  // every wave has read the last layer's input
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float v = acc[r] + bias;
            z[r * TR_THREADS] = v;
            h[r] = gelu_f(v);
        }
        if (l < 3) put_tile(h, act[(l + 1) & 1], a.hf + l * a.frag + off_g, j, lh);
        derive(z);
        if (l == 3) break;
        __syncthreads();
        acc = tile_product(act[(l + 1) & 1], wb, li, lh);
        load_frags(wb, l < 2 ? a.wf + (l + 1) * MLP_H * MLP_H + off_f : a.wt + 2 * MLP_H * MLP_H + off_t,
                   l < 2 ? 1024 : 512);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) d3[r] = h4s[r * TR_THREADS + t];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) h4s[(8 * (r >> 2) + 4 * lh + (r & 3)) * TR_H4_PITCH + j] = h[r];
    __syncthreads();
    // ---- output head: wave w sums samples 4 w .. 4 w + 3, lane l neurons 4 l .. 4 l + 3 ----
    {
        float4 wv[SIRIUS_MLP_OUT];
#pragma unroll
        for (int o = 0; o < SIRIUS_MLP_OUT; ++o) wv[o] = *(const float4*)(a.W4 + o * MLP_H + 4 * lane);
        const float b4 = lane < SIRIUS_MLP_OUT ? a.b4[lane] : 0.f;
#pragma unroll 1
        for (int s = 4 * w; s < 4 * w + 4; ++s) {
            const float4 hv = *(const float4*)&h4s[s * TR_H4_PITCH + 4 * lane];
            float p[SIRIUS_MLP_OUT];
#pragma unroll
            for (int o = 0; o < SIRIUS_MLP_OUT; ++o)
                p[o] = fmaf(hv.w, wv[o].w, fmaf(hv.z, wv[o].z, fmaf(hv.y, wv[o].y, fmaf(hv.x, wv[o].x, 0.f))));
#pragma unroll
            for (int off = 32; off > 0; off >>= 1)
#pragma unroll
                for (int o = 0; o < SIRIUS_MLP_OUT; ++o) p[o] += __shfl_xor(p[o], off);
            float v = 0.f;
#pragma unroll
            for (int o = 0; o < SIRIUS_MLP_OUT; ++o) v = lane == o ? p[o] + b4 : v;
            if (lane < SIRIUS_MLP_OUT) ys[s][lane] = v;
        }
    }
    __syncthreads();
    // ---- loss and output gradient (1/n of the batch mean included); rows past n are zero ----
    float loss = 0.f;
    if (t < TR_ROWS) {
        const int64_t i = row0 + t;
        float g[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (i < a.n) {
            const float* y = ys[t];
            int c = a.cls[i];
            c = c < 0 ? 0 : (c > 2 ? 2 : c);
            float m = fmaxf(y[0], fmaxf(y[1], y[2]));
            float e0 = expf(y[0] - m), e1 = expf(y[1] - m), e2 = expf(y[2] - m);
            float s = e0 + e1 + e2;
            float yc = c == 0 ? y[0] : (c == 1 ? y[1] : y[2]);
            loss = -(yc - m - logf(s));
            const float inv_n = 1.f / (float)a.n;
            g[0] = (e0 / s - (c == 0)) * inv_n;
            g[1] = (e1 / s - (c == 1)) * inv_n;
            g[2] = (e2 / s - (c == 2)) * inv_n;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                float d = c == 0 ? y[3 + k] - a.dir[i * 3 + k] : 0.f;
                loss += (float)SIRIUS_MLP_DIR_WEIGHT * d * d;
                g[3 + k] = 2.f * (float)SIRIUS_MLP_DIR_WEIGHT * d * inv_n;
            }
        }
#pragma unroll
        for (int o = 0; o < 6; ++o) gys[t][o] = g[o];
    }
    __syncthreads();
    // the tile's row of partials; the two half-waves hold the same neurons for other samples
    float* row = a.part + T * MLP_TILE_COLS;
    auto put = [&](int col, float v) {
        v += __shfl_xor(v, 32);
        if (lh == 0) row[col + j] = v;
    };
    // ---- backward: head ----
    float g[16], db = 0.f;
    {
        float w4[SIRIUS_MLP_OUT], dw4[SIRIUS_MLP_OUT];
#pragma unroll
        for (int o = 0; o < SIRIUS_MLP_OUT; ++o) {
            w4[o] = a.W4[o * MLP_H + j];
            dw4[o] = 0.f;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float* gy = gys[8 * (r >> 2) + 4 * lh + (r & 3)];
            float dh = 0.f;
#pragma unroll
            for (int o = 0; o < SIRIUS_MLP_OUT; ++o) {
                dh = fmaf(gy[o], w4[o], dh);
                dw4[o] = fmaf(gy[o], h[r], dw4[o]);
            }
            g[r] = dh * d3[r];
            db += g[r];
        }
#pragma unroll
        for (int o = 0; o < SIRIUS_MLP_OUT; ++o) put(MLP_COL_DW4 + o * MLP_H, dw4[o]);
        put(MLP_COL_DB + 3 * MLP_H, db);
    }
    if (w == 0) {
        for (int off = 16; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
        if (lane == 0) row[MLP_COL_LOSS] = loss;
        if (lane < SIRIUS_MLP_OUT) {
            float db4 = 0.f;
            for (int i = 0; i < TR_ROWS; ++i) db4 += gys[i][lane];
            row[MLP_COL_DB4 + lane] = db4;
        }
    }
    // ---- backward: hidden layers ----
#pragma unroll 1
    for (int l = 3;; --l) {
        // gz_l is in g: the next product's A tile (h4s was read before the last barrier) and a
        // weight-gradient operand
        put_tile(g, act[l & 1], a.gf + (l - 1) * a.frag + off_g, j, lh);
        __syncthreads();
        acc = tile_product(act[l & 1], wb, li, lh);
        if (l > 1) load_frags(wb, a.wt + (l - 2) * MLP_H * MLP_H + off_t, 512);
        db = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            g[r] = acc[r] * zs[l - 1][r * TR_THREADS + t];
            db += g[r];
        }
        put(MLP_COL_DB + (l - 1) * MLP_H, db);
        if (l == 1) break;
    }
    // first layer's weights: the BF16 gradient times the BF16 inputs, summed in FP32
    float dw0[SIRIUS_MLP_IN] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float gb = (float)(__bf16)g[r];
        const float* x = xs[8 * (r >> 2) + 4 * lh + (r & 3)];
#pragma unroll
        for (int k = 0; k < SIRIUS_MLP_IN; ++k) dw0[k] = fmaf(gb, x[k], dw0[k]);
    }
#pragma unroll
    for (int k = 0; k < SIRIUS_MLP_IN; ++k) put(MLP_COL_DW0 + k * MLP_H, dw0[k]);
}

// dW_l = gz_l^T h_l for the hidden layers l = 1..3 (blockIdx.z = l - 1), 128 x 128 outputs per block
// (blockIdx.y), the 32-sample tiles of split blockIdx.x: four waves of 64 x 64. Both operands are
// read as the fragments k_mlp_train wrote, each a contiguous kilobyte per wave, two tiles ahead of
// the products.
__global__ __launch_bounds__(256) void k_mlp_wgrad(MlpWgradArgs a) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int l = blockIdx.z;
    const int jb = (blockIdx.y >> 1) * 4 + (w >> 1) * 2, kb = (blockIdx.y & 1) * 4 + (w & 1) * 2;
    const int64_t t0 = (int64_t)blockIdx.x * a.chunk, t1 = min(a.tiles, t0 + a.chunk);
    const uint16_t* A = a.gf + l * a.frag + (int64_t)jb * 2 * 512 + lane * 8;
    const uint16_t* B = a.hf + l * a.frag + (int64_t)kb * 2 * 512 + lane * 8;
    v16f acc[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
    constexpr int AHEAD = 2;
    v8bf fa[AHEAD][2][2], fb[AHEAD][2][2];  // [tile][block][half tile of 16 samples]
    auto load = [&](int64_t T, v8bf (&xa)[2][2], v8bf (&xb)[2][2]) {
        const int64_t at = T * (8 * 2 * 512);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                xa[m][s] = ld8(A + at + (m * 2 + s) * 512);
                xb[m][s] = ld8(B + at + (m * 2 + s) * 512);
            }
    };
#pragma unroll
    for (int q = 0; q < AHEAD; ++q)
        if (t0 + q < t1) load(t0 + q, fa[q], fb[q]);
    for (int64_t T = t0; T < t1; T += AHEAD) {
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
            if (T + q < t1) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int m = 0; m < 2; ++m)
#pragma unroll
                        for (int n = 0; n < 2; ++n)
                            acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[q][m][s], fb[q][n][s], acc[m][n], 0, 0, 0);
                if (T + q + AHEAD < t1) load(T + q + AHEAD, fa[q], fb[q]);
            }
        }
    }
    float* out = a.part + ((int64_t)blockIdx.x * 3 + l) * MLP_H * MLP_H;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = (jb + m) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                out[(int64_t)row * MLP_H + (kb + n) * 32 + (lane & 31)] = acc[m][n][r];
            }
}

// The gradient in the public layout: blocks 0 .. GS_W - 1 add the splits of the hidden layers'
// weights (four values per lane), the others the rows of per-tile partials (64 columns each, 16
// groups of rows, then the groups in order). The loss's column goes to *loss.
constexpr int GS_THREADS = 1024;
constexpr int GS_W = 3 * MLP_H * MLP_H / 4 / GS_THREADS;
static_assert(3 * MLP_H * MLP_H % (4 * GS_THREADS) == 0 && MLP_TILE_COLS % 64 == 0, "whole blocks");
__global__ __launch_bounds__(GS_THREADS) void k_mlp_grad_sum(MlpGradSumArgs a) {
    __shared__ float red[16][64];
    const int t = threadIdx.x;
    if (blockIdx.x < GS_W) {
        const int e = (blockIdx.x * GS_THREADS + t) * 4;
        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int q = 0; q < a.splits; ++q) {
            const float4 v = *(const float4*)(a.wpart + (int64_t)q * 3 * MLP_H * MLP_H + e);
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
        float* d = a.grad + a.off_w[1 + e / (MLP_H * MLP_H)] + e % (MLP_H * MLP_H);
        d[0] = s.x; d[1] = s.y; d[2] = s.z; d[3] = s.w;  // the caller's array may not be 16-byte aligned
        return;
    }
    const int c = (blockIdx.x - GS_W) * 64 + (t & 63), q = t >> 6;
    float s = 0.f;
    for (int r = q; r < a.rows; r += 16) s += a.part[(int64_t)r * MLP_TILE_COLS + c];
    red[q][t & 63] = s;
    __syncthreads();
    if (q) return;
    s = red[0][t];
#pragma unroll
    for (int k = 1; k < 16; ++k) s += red[k][t];
    if (c < MLP_COL_DW4) a.grad[a.off_b[c / MLP_H] + c % MLP_H] = s;
    else if (c < MLP_COL_DB4) a.grad[a.off_w[4] + c - MLP_COL_DW4] = s;
    else if (c < MLP_COL_LOSS) a.grad[a.off_b[4] + c - MLP_COL_DB4] = s;
    else if (c == MLP_COL_LOSS) *a.loss = s;
    else if (c >= MLP_COL_DW0 && c < MLP_COL_DW0 + SIRIUS_MLP_IN * MLP_H) {
        const int k = (c - MLP_COL_DW0) / MLP_H, o = (c - MLP_COL_DW0) % MLP_H;
        a.grad[a.off_w[0] + o * SIRIUS_MLP_IN + k] = s;
    }
}

hipError_t launch_mlp_train(const MlpTrainArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_train, dim3((unsigned)((a.n + TR_ROWS - 1) / TR_ROWS)), dim3(TR_THREADS), 0, st, a);
    return hipGetLastError();
}
hipError_t launch_mlp_wgrad(const MlpWgradArgs& a, int splits, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_wgrad, dim3((unsigned)splits, 4, 3), dim3(256), 0, st, a);
    return hipGetLastError();
}
hipError_t launch_mlp_grad_sum(const MlpGradSumArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_grad_sum, dim3(GS_W + MLP_TILE_COLS / 64), dim3(GS_THREADS), 0, st, a);
    return hipGetLastError();
}

// Operands of the inference and training kernels from the FP32 masters: W0 [256][16] (input columns padded), and the
// hidden layers' and the head's weights in MFMA fragment order: the 16-byte A operand of lane l
// for k-step ks, row tile mt of wave w sits at (((w 16 + ks) 2 + mt) 64 + l) 8 (hidden layer:
// row 64 w + 32 mt + l % 32, columns 16 ks + 8 (l / 32) .. +7), so each wave's weight load is one
// contiguous kilobyte; their transposes for the backward pass, the fragment of lane l for k-step ks,
// column block w at ((w 16 + ks) 64 + l) 8 (W[16 ks + 8 (l / 32) .. +7][32 w + l % 32]); the head's
// high and low BF16 parts (rows 6..31 zero) in the k order of the fused kernel's accumulators.
__global__ void k_pack_fused(const float* __restrict__ P, uint16_t* __restrict__ w0, uint16_t* __restrict__ wh,
                             uint16_t* __restrict__ wt, uint16_t* __restrict__ w4h, uint16_t* __restrict__ w4l, size_t off_w0, size_t off_w1,
                             size_t off_w2, size_t off_w3, size_t off_w4) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < MLP_H * 16) {
        const int j = e / 16, k = e % 16;
        w0[e] = k < SIRIUS_MLP_IN ? f2bf(P[off_w0 + (size_t)j * SIRIUS_MLP_IN + k]) : (uint16_t)0;
    }
    if (e < 3 * MLP_H * MLP_H) {
        const int l = e / (MLP_H * MLP_H), r = e % (MLP_H * MLP_H);
        const int i = r & 7, lane = (r >> 3) & 63, mt = (r >> 9) & 1, ks = (r >> 10) & 15, w = r >> 14;
        const int j = 64 * w + 32 * mt + (lane & 31), k = 16 * ks + 8 * (lane >> 5) + i;
        const size_t off = l == 0 ? off_w1 : (l == 1 ? off_w2 : off_w3);
        wh[e] = f2bf(P[off + (size_t)j * MLP_H + k]);
        const int tj = 16 * ((r >> 9) & 15) + 8 * (lane >> 5) + i, tk = 32 * (r >> 13) + (lane & 31);
        wt[e] = f2bf(P[off + (size_t)tj * MLP_H + tk]);
    }
    if (e < 32 * MLP_H) {
        // fragment (wave w, row tile mt, run pair): value i of lane l is W4[l % 32][64 w + 32 mt +
        // 16 pair + 8 (i / 4) + 4 (l / 32) + i % 4]
        const int i = e & 7, lane = (e >> 3) & 63, j = lane & 31;
        const int k = 16 * (e >> 9) + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        const float w = j < SIRIUS_MLP_OUT ? P[off_w4 + (size_t)j * MLP_H + k] : 0.f;
        const uint16_t hi = f2bf(w);
        w4h[e] = hi;
        w4l[e] = f2bf(w - __uint_as_float((uint32_t)hi << 16));
    }
}
hipError_t launch_pack_fused(const float* params, uint16_t* w0, uint16_t* wh, uint16_t* wt, uint16_t* w4h, uint16_t* w4l,
                             const size_t off_w[5], hipStream_t st) {
    hipLaunchKernelGGL(k_pack_fused, dim3((3 * MLP_H * MLP_H + 255) / 256), dim3(256), 0, st, params, w0, wh, wt, w4h, w4l,
                       off_w[0], off_w[1], off_w[2], off_w[3], off_w[4]);
    return hipGetLastError();
}

// Adam (beta1 0.9, beta2 0.999, eps 1e-8); c1 = 1 - beta1^t, c2 = 1 - beta2^t.
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int64_t P, float lr, float c1, float c2) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= P) return;
    float gi = g[e];
    float mi = 0.9f * m[e] + 0.1f * gi;
    float vi = 0.999f * v[e] + 0.001f * gi * gi;
    m[e] = mi;
    v[e] = vi;
    p[e] -= lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
}
hipError_t launch_adam(float* params, const float* grad, float* m, float* v, int64_t P, float lr, float c1, float c2,
                       hipStream_t st) {
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, st, params, grad, m, v, P, lr, c1, c2);
    return hipGetLastError();
}

}  // namespace sirius
