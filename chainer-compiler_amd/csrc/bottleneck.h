// The tail of a bottleneck block (3x3 convolution, 1x1 expansion, residual sum) and the 1x1 reduction of the block behind it
// as one launch: what contract_api.hip hands to bottleneck.hip.
#pragma once

#include "conv_mfma.h"

namespace chx {

struct BottleneckArgs {
    const char* x;  // channels-last and dense: pixel m at x + m * x_px
    char *y, *z;    // the sum and the reduction's result (null: none), likewise
    int64_t x_px, y_px, z_px;
    const char *w1, *w2, *w3;  // fragments [32 channels out][K step of 32][lane][16]
    const int32_t* table;      // [mid + wide + next][4]: scale, bias, sum of the weights
    int32_t pixels, H, W;
    int32_t mid, wide, next;  // channels in front of, behind the expansion, and of the reduction's result (0: none)
    uint32_t x_flip, y_flip, z_flip;
    int32_t fill;                 // x's zero point in the signed range, four times
    int32_t corr1, corr2, corr3;  // what the zero points leave of the sums of the weights
    float s1, s2, s3;             // scale of each convolution's input
    QuantProduct q1, q2, q3;
    ResidualAdd res;
    // the launch (filled by plan_bottleneck)
    int32_t px_tiles, px_waves, groups, lds;  // tiles of 32 pixels of a work-group, wavefronts that share them, groups of wavefronts, bytes of LDS
    int32_t patch_rows, at_mid, at_wide, at_table, tiles, xcd_chunk, quads_log2;  // log2(wide / 256)
    uint32_t w_mul, w_shift, h_mul, h_shift;
};

// From the sizes above; EUNSUPPORTED where the block does not fit or single launches are faster.
int plan_bottleneck(BottleneckArgs* a);
int launch_bottleneck(const BottleneckArgs& a, hipStream_t s);
// Weights [rows, C, KH, KW] (int8, zero points 0) as fragments, K in the order (kh, kw, c), with their table.
int pack_bottleneck(const chx_hip_tensor& w, const chx_hip_tensor& scale, const chx_hip_tensor* bias, char* fragments, int32_t* table, hipStream_t s);
// More than four times as many channels behind the expansion as in front of it are faster as single launches (up to 2.0 times,
// of 400 drawn blocks).
constexpr bool bottleneck_takes_channels(int64_t mid, int64_t wide, int64_t next) {
    return (mid == 64 || mid == 128 || mid == 256) && wide >= 256 && wide <= 4 * mid && (wide & (wide - 1)) == 0 && next % 32 == 0 && next <= 1024;
}

}  // namespace chx
