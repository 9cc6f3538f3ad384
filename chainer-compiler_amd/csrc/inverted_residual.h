// An inverted residual block (1x1 expansion, depthwise 3x3, 1x1 projection, optionally the residual sum behind it) as one
// launch: what contract_api.hip hands to inverted_residual.hip.
#pragma once

#include "conv_mfma.h"

namespace chx {

struct InvertedResidualArgs {
    const char* x;  // channels-last, a pixel's channels in whole 16-byte chunks
    char* y;        // likewise
    int64_t x_n, x_px, y_n, y_px;  // bytes from one image, one pixel to the next
    const char* w1;        // fragments [hid tile][K step][lane][16]
    const char* w3;        // fragments [oc tile][hid tile][lane][16]
    const int32_t* t1;     // [hid][4]: scale, bias, sum of the weights
    const int32_t* t2;     // [hid][8]: the filter's rows as byte triples, scale, bias, sum
    const int32_t* t3;     // [oc][4]: as t1
    int32_t N, H, W, OH, OW, OC;
    int32_t hid_tiles, hid_tiles_padded;  // of 32 expanded channels; what w1, w3, t1 and t2 are laid out for (a multiple of 8, zeros at the end)
    int32_t x_chunks, KS;  // 16-byte chunks of a pixel, K steps of the expansion that w1 has: 1, 3 or 5
    uint32_t x_flip, y_flip;
    int32_t corr1, corr2, corr3;  // what the zero points leave of the sums of the weights
    float s1, s2, s3;             // scale of each convolution's input
    QuantProduct q1, q2, q3;
    int32_t fill;                 // the zero point of the expansion's result in the signed range, four times
    ResidualAdd res;              // res.r null: none
    // the launch (filled by plan_inverted_residual)
    int32_t G, lds;  // tiles of 32 expanded channels per interval; bytes of LDS
    int32_t buffers;  // of expanded and of convolved channels: 2, the three parts for three chunks at a time, or 1
    int32_t R, rows, pitch, pixels, px_bytes, pitch_o, items, tiles_px, tiles_oc, cs, cs2, intervals;
    int32_t at_mask, at_hid, at_dw, at_t3, blocks, strips, xcd_chunk;
    uint32_t strips_mul, strips_shift, pitch_mul, pitch_shift, pitch_o_mul, pitch_o_shift, row_mul, row_shift, chunks_mul, chunks_shift, oct_mul, oct_shift, blk_mul, blk_shift;
};

// From the sizes above; EUNSUPPORTED where the block does not fit (LDS, channels) or single launches are faster.
int plan_inverted_residual(InvertedResidualArgs* a, int stride);
int launch_inverted_residual(const InvertedResidualArgs& a, int stride, hipStream_t s);
// Weights of a 1x1 convolution [rows, K] (int8, zero points 0) as MFMA fragments, with their tables; `projection`: rows are
// output channels in the order that leaves a lane sixteen neighbouring ones.
int pack_inverted_point(const chx_hip_tensor& w, const chx_hip_tensor& scale, const chx_hip_tensor* bias, bool projection, int row_tiles, int k_tiles,
                        char* fragments, int32_t* table, hipStream_t s);
int pack_inverted_depthwise(const chx_hip_tensor& w, const chx_hip_tensor& scale, const chx_hip_tensor* bias, int tiles, int32_t* table, hipStream_t s);
constexpr int kInvertedMaxIn = 160;  // input channels
constexpr int kInvertedMaxOut = 320;

}  // namespace chx
