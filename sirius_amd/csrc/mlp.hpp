// mlp.hpp — the far-field surrogate network on the device: BF16 MFMA GEMMs with FP32
// accumulation and fused epilogues, the loss, Adam, and the surrogate's per-ray kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/sirius_hip.h"

namespace sirius {

constexpr int MLP_NL = 5;                      // weight layers
constexpr int MLP_H = SIRIUS_MLP_HIDDEN;       // 256

// Layer dims
constexpr int MLP_IN[MLP_NL] = {SIRIUS_MLP_IN, MLP_H, MLP_H, MLP_H, MLP_H};
constexpr int MLP_OUTD[MLP_NL] = {MLP_H, MLP_H, MLP_H, MLP_H, SIRIUS_MLP_OUT};

size_t mlp_param_count();
size_t mlp_param_offset_w(int l);  // offset of W_l in the public layout
size_t mlp_param_offset_b(int l);

// Training kernels (mlp_kernels.hip). k_mlp_train takes a tile of MLP_TRAIN_ROWS samples per block,
// which leaves one row of partial sums: columns MLP_COL_*.
constexpr int MLP_TRAIN_ROWS = 32;
constexpr int MLP_COL_DB = 0;                                          // db_0 .. db_3
constexpr int MLP_COL_DW4 = 4 * MLP_H;                                 // dW_4, row-major
constexpr int MLP_COL_DB4 = MLP_COL_DW4 + SIRIUS_MLP_OUT * MLP_H;      // db_4
constexpr int MLP_COL_LOSS = MLP_COL_DB4 + SIRIUS_MLP_OUT;
constexpr int MLP_COL_DW0 = MLP_COL_LOSS + 2;                          // dW_0, column-major
constexpr int MLP_TILE_COLS = (MLP_COL_DW0 + SIRIUS_MLP_IN * MLP_H + 63) / 64 * 64;
struct MlpTrainArgs {
    const float* x;        // n x 5
    const int32_t* cls;    // n
    const float* dir;      // n x 3
    int64_t n;
    const uint16_t* w0;    // packed operands (k_pack_fused): W_0, W_1..W_3 and their transposes
    const uint16_t* wf;
    const uint16_t* wt;
    const float* b[4];
    const float* W4;       // FP32 head
    const float* b4;
    uint16_t* hf;          // fragments of the inputs of layers 1..3, [3][tile][8][2][64][8] BF16, and
    uint16_t* gf;          // of the gradients with respect to their pre-activations
    int64_t frag;          // BF16 values of one layer's fragments
    float* part;           // [tiles][MLP_TILE_COLS]
};
struct MlpWgradArgs {
    const uint16_t* hf;    // as in MlpTrainArgs
    const uint16_t* gf;
    int64_t frag;
    int64_t tiles, chunk;  // 32-sample tiles, and how many each split takes
    float* part;           // [splits][3][256][256]
};
struct MlpGradSumArgs {
    const float* wpart;
    const float* part;
    int splits, rows;
    size_t off_w[MLP_NL], off_b[MLP_NL];
    float* grad;
    float* loss;           // sum of the batch's losses
};
hipError_t launch_mlp_train(const MlpTrainArgs& a, hipStream_t st);
hipError_t launch_mlp_wgrad(const MlpWgradArgs& a, int splits, hipStream_t st);
hipError_t launch_mlp_grad_sum(const MlpGradSumArgs& a, hipStream_t st);
hipError_t launch_adam(float* params, const float* grad, float* m, float* v, int64_t P, float lr, float c1, float c2,
                       hipStream_t st);

// Fused inference (k_mlp_fused): the whole network over rows of x in one kernel.
struct MlpFusedArgs {
    const float* x;        // inputs: row r at x[r * x_stride] (x[idx[r] * x_stride] when idx is set)
    int64_t n;             // rows (when n_dev is null)
    const uint32_t* n_dev; // rows, read on the device (null: n)
    const int32_t* idx;    // optional gather list
    int64_t x_stride;      // floats per input record (5 for packed inputs)
    const uint16_t* w0;    // [256][16] BF16, input columns padded to 16
    const uint16_t* w[3];  // layers 1..3, [256][256] BF16 in MFMA fragment order (k_pack_fused)
    const float* b[4];     // biases of layers 0..3, [256]
    const uint16_t* w4h;   // head weights, 32 rows (6..31 zero) x 256, BF16 high parts (k_pack_fused)
    const uint16_t* w4l;   // and low parts
    const float* b4;       // head bias [6]
    float* y;              // n x 6 outputs
};
hipError_t launch_mlp_fused(const MlpFusedArgs& a, int64_t cap, int max_blocks, hipStream_t st);

// Surrogate records (one per candidate ray, by ray id): network inputs (5), signed distance from
// the critical curve, the reference orbit's impact parameter, padding, the reference exit
// direction (3), padding. Calibration bins of the error gate, and the held-out rays a bin needs.
constexpr int SUR_REC = 12;
// The reference orbit of a ray starts at x0 + SUR_SPIN_SHIFT a e_phi (e_phi: the observer's
// azimuthal direction): the lens displaced as frame dragging displaces it to first order in a.
constexpr double SUR_SPIN_SHIFT = 1.1;
constexpr int SUR_BINS = 270;
constexpr uint32_t SUR_CAL_MIN = 20;
// off_w: parameter offsets of W_0 .. W_4 (mlp_param_offset_w)
hipError_t launch_pack_fused(const float* params, uint16_t* w0, uint16_t* wh, uint16_t* wt, uint16_t* w4h, uint16_t* w4l,
                             const size_t off_w[5], hipStream_t st);

// Device state of the network of one handle.
struct MlpState {
    float* params = nullptr;  // FP32 masters, public layout
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    float* grad = nullptr;
    int64_t step = 0;
    uint16_t* fw0 = nullptr;   // packed BF16 operands: W0 [256][16], hidden layers 1..3 (3 x 256 x 256,
    uint16_t* fwh = nullptr;   // fragment order), their transposes, head W_hi / W_lo, 32 x 256
    uint16_t* fwt = nullptr;
    uint16_t* fw4h = nullptr;
    uint16_t* fw4l = nullptr;
    float* loss_host = nullptr;  // pinned: the device writes each batch's loss sum here
    // calibration of the error gate (SUR_BINS each): held-out rays the network would answer,
    // misclassified ones, and the largest direction error (rad); all zero until calibrated, so
    // an uncalibrated network answers nothing
    float* cal_err = nullptr;
    uint32_t* cal_n = nullptr;
    uint32_t* cal_bad = nullptr;
    // the largest distance from the critical curve among a bin's held-out answers: the bin
    // answers no ray beyond it (the calibration holds no evidence there)
    float* cal_dmax = nullptr;
    // the training cameras' field of view: the largest |x| and |y| of a pixel centre's direction
    // on the image plane at unit distance. Rays outside this box lie outside the training set's
    // support in (alpha, beta) for their observer and are never answered.
    float sup_x = 0.f, sup_y = 0.f;
    bool ready = false;
};

}  // namespace sirius
