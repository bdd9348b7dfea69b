// The many-row int8 GEMM (w8a16_rows.hip): more than one decode launch's rows at once.
#pragma once

#include "common.h"

namespace mx {
namespace w8a16 {

struct RowsPlan {
    int MT;   // 16-row tiles per workgroup; 0: the shape is not for this launch
    int NPW;  // n-tiles per wave (4 waves per workgroup)
    int KS;   // k ranges; more than one writes fp32 partials [KS][M][N]
};

// The plan of an M-row launch whose partials may take up to partial_bytes (0: no ranges).
RowsPlan plan_rows(int64_t M, int NT, int KT, size_t partial_bytes);

// Whether the launch's indices hold this shape.
bool rows_fit(int64_t M, int64_t xs, int NT);

// y = x W^T (+ bias), or its SwiGLU product for an interleaved gate||up weight where gu; with
// pl.KS > 1 the scaled partials instead of y.
void launch_rows(bool gu, const RowsPlan& pl, const uint16_t* x, int64_t xs, int M, const uint8_t* w,
                 const uint16_t* scale, const uint16_t* bias, uint16_t* y, int64_t ys, int NT, int KT, float* partial,
                 hipStream_t st);

}  // namespace w8a16
}  // namespace mx
