// gemm.h -- internal interface of the prefill GEMM kernels (gemm.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "formats.h"

// One group of a grouped GEMM (e.g. one expert): its weights and its tokens,
// octets [oct0, oct0 + n_oct) of the digit buffer.
struct GemmGroup {
    const uint8_t* W;
    int oct0, n_oct;
};

struct GemmArgs {
    const uint8_t* W;   // weights, Q4_K / Q6_K tile layout
    DracoLayout L;
    int n_in, T;
    // digitized activations (draco_gemm_digits_launch)
    const int8_t* xdig;
    const float* xsc;
    const float* xs32;
    const float* xs16;
    float* Y;           // Y[t * ldy + row]
    int ldy;
    // grouped launch (nullptr: one group = W, all tokens)
    const GemmGroup* groups;  // device array [n_groups]
    int n_groups;
    int max_oct;              // largest n_oct of any group
};

// device bytes of the digit buffer for T tokens of length n_in
size_t draco_gemm_digit_bytes(int T, int n_in);
// digitize X[T][n_in] (device) into buf; fills a.xdig/xsc/xs32/xs16, a.T, a.n_in
int draco_gemm_digits_launch(const float* X, int T, int n_in, uint8_t* buf, GemmArgs& a, hipStream_t st);
int draco_gemm_launch(GemmArgs& a, hipStream_t st);

// ---- f16-MFMA GEMM (gemmh.hip) ----
// One matrix of a launch: Y[t * ldy + row] = x_t . W[row].
struct GemmHSeg {
    const uint8_t* W;             // weights in their layout (draco_gemmh_serves)
    const uint8_t* const* bases;  // grouped launches: device table of each group's W
    DracoLayout L;
    float* Y;
    int ldy;
    int fm, rg0;                  // set by the launch
};
// Up to three matrices on the same activations in one launch (formats that
// draco_gemmh_mixes).  pair: seg[0] and seg[1] are a SwiGLU gate and up of one
// shape and format, and seg[0].Y receives silu(gate) * up.  groups: device
// array [max_tiles] with the group (expert) of every 32-token tile, or a
// negative number; the rows of a tile all belong to its group.
struct GemmHArgs {
    GemmHSeg seg[3];
    int nseg, pair;
    int n_in, T;
    const uint8_t* xh;            // activations from draco_gemmh_x_launch
    const int* groups;
    int max_tiles;
    int rpb, n_rg;                // set by the launch
};
bool draco_gemmh_serves(int code);  // Q4_K, Q5_K, Q6_K, Q8_0
bool draco_gemmh_mixes(int c0, int c1);
size_t draco_gemmh_x_bytes(int T, int n_in);
// rows (device, nullable): token t's values are row rows[t] of X, zeros where negative
int draco_gemmh_x_launch(const float* X, int T, int n_in, uint8_t* buf, hipStream_t st, const int* rows = nullptr);
int draco_gemmh_launch(GemmHArgs& a, hipStream_t st);

struct DracoMat;
// Y_i[t][row] = X[t] . W_i[row] for T token rows and n matrices on the same
// rows (X, Y device, token-major).  The block formats (draco_gemmh_serves): X's
// activation operands (f16 hi/lo) into `digits` (draco_gemm_digit_bytes(T,
// n_in) bytes), then f16-MFMA launches of up to three matrices each; F32 and
// F16: one GEMV per token.
struct GemmTo {
    const DracoMat* m;
    float* Y;
};
int draco_enqueue_gemms(const GemmTo* to, int n, const float* X, int T, uint8_t* digits, hipStream_t st);
// silu(gate . x) * (up . x) of T rows into G; U is scratch for formats whose pair is not one launch
int draco_enqueue_swiglu(const DracoMat& gate, const DracoMat& up, const float* X, int T, float* G, float* U,
                         uint8_t* digits, hipStream_t st);
// Y[t] for the tokens of every group against that group's W (same shape for all groups)
int draco_gemm_grouped_launch(GemmArgs& a, hipStream_t st);
