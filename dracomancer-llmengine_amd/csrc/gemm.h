// gemm.h -- internal interface of the prefill GEMM (gemmh.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "formats.h"

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
// activation operands (f16 hi/lo) into `digits` (draco_gemmh_x_bytes(T,
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
