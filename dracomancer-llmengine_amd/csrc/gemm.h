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
    float* part;                  // draco_gemmh_part_floats floats; null: rows are not split over blocks
    int rpb, n_rg, ksp, pps;      // set by the launch
};
// The blocks of a launch: the pairs (major, minor), major of M, minor of m.
// Blocks of one major share operands and lie on one XCD (block id mod 8)
// where that spreads evenly: the majors of whole eights go to an XCD each,
// the pairs of the other M % 8 majors in equal runs to all eight.
struct GemmHMap {
    int full, rem;  // blocks per XCD of the whole eights, of the rest
};
static inline __host__ __device__ GemmHMap gemmh_map(int M, int m) {
    return {(M >> 3) * m, ((M & 7) * m + 7) >> 3};
}
// block's pair (false: none)
static inline __host__ __device__ bool gemmh_place(int M, int m, int block, int& major, int& minor) {
    const GemmHMap g = gemmh_map(M, m);
    const int x = block & 7, loc = block >> 3;
    const bool whole = loc < g.full;
    const int i = whole ? loc : x * g.rem + loc - g.full, q = i / m;  // (one division)
    major = whole ? 8 * q + x : (M & ~7) + q;
    minor = i - q * m;
    return whole || (loc - g.full < g.rem && i < (M & 7) * m);
}
unsigned draco_gemmh_blocks(int M, int m);               // grid of the map above
int draco_gemmh_place(int M, int m, int block);          // major * m + minor or -1, for the map's test
void draco_gemmh_plan(int n_out, int n_in, int T, int* out);  // one matrix: slots, row tiles, row splits, passes a split
bool draco_gemmh_serves(int code);  // Q4_K, Q5_K, Q6_K, Q8_0
bool draco_gemmh_mixes(int c0, int c1);
size_t draco_gemmh_x_bytes(int T, int n_in);
// rows (device, nullable): token t's values are row rows[t] of X, zeros where negative
int draco_gemmh_x_launch(const float* X, int T, int n_in, uint8_t* buf, hipStream_t st, const int* rows = nullptr);
// floats of partial sums that the launch of these arguments would use (0: none)
size_t draco_gemmh_part_floats(const GemmHArgs& a);
int draco_gemmh_launch(GemmHArgs& a, hipStream_t st);

struct DracoMat;
// Y_i[t][row] = X[t] . W_i[row] for T token rows and n matrices on the same
// rows (X, Y device, token-major).  The block formats (draco_gemmh_serves): X's
// activation operands (f16 hi/lo) into `xh` (draco_gemmh_x_bytes(T,
// n_in) bytes), then f16-MFMA launches of up to three matrices each; F32 and
// F16, and Q8_0 / Q5_K of the shortest calls: one GEMV per token.
struct GemmTo {
    const DracoMat* m;
    float* Y;
};
int draco_enqueue_gemms(const GemmTo* to, int n, const float* X, int T, uint8_t* xh, hipStream_t st);
// silu(gate . x) * (up . x) of T rows into G; U is scratch for formats whose pair is not one launch
int draco_enqueue_swiglu(const DracoMat& gate, const DracoMat& up, const float* X, int T, float* G, float* U,
                         uint8_t* xh, hipStream_t st);
