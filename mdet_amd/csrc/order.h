// Row order and projection of the exhaustive pair stage (tnf_order.hip), as
// the pair pipeline (tnf_pairs.hip) uses them.
#pragma once

#include "hip_common.h"

namespace mdet {

// A fixed number of leading directions of the TNF rows, found from the rows
// themselves: |P (a - b)| <= |a - b| for every pair of rows, so a pair whose
// projections are farther apart than a radius is farther apart than it.
constexpr int PROJ_D = 28;   // dimensions
constexpr int PROJ_KS = 2;   // MFMA k-steps: 28 dimensions and 4 threshold slots
constexpr int PROJ_W = 32;   // floats per projected row: the dimensions, then 4 words of k_project

struct ProjOrder {
    uint32_t* perm = nullptr;  // device: position -> row (context buffer)
    float* y = nullptr;        // device: projected rows, n x PROJ_W, by row (context buffer)
};

// Queues, without a host round trip: the directions, the projected rows, and
// the order of the rows by the nearest of a number of centres in them (rows of
// one population end up close together; rows holding a NaN or an infinity
// come last).
// fmt: the format the caller rounds the rows to afterwards; each row's margin
// in proj_frags then covers twice that rounding's error.
enum ProjFormat { PROJ_F32 = 0, PROJ_BF16 = 1, PROJ_F16 = 2 };
int proj_order(mdet_ctx* ctx, const float* tnf_dev, uint32_t n, ProjFormat fmt, ProjOrder* out);
// FP16 MFMA fragments of the projected rows in that order, n_pad rows (a
// multiple of 32; the ones past n never pass), with the threshold in the last
// slots: the product of a row-role and a column-role row is > 0 for every pair
// of rows at distance R (plus both rows' margins) or less.  frag: n_pad / 32 x PROJ_KS x 64 entries;
// frag_a: n_pad / 32 x 64 (the row-role form of the last k-step).
int proj_frags(mdet_ctx* ctx, const ProjOrder& o, uint32_t n, uint32_t n_pad, float R, uint4* frag, uint4* frag_a);
// Boxes of `tiles` 32-row tiles (those past n empty) in that order: box[d * T + t]
// (lowest, highest), margin[t].  Rows of two tiles within R of each other project
// to within R + both margins.
int proj_boxes(mdet_ctx* ctx, const ProjOrder& o, uint32_t n, uint32_t tiles, uint32_t T, float2* box, float* margin);
// The projected rows alone; proj_frags and proj_boxes then take any order of
// any of the rows (perm, with n its length).
int proj_rows(mdet_ctx* ctx, const float* tnf_dev, uint32_t n, ProjFormat fmt, float** y);

}  // namespace mdet
