// qgemm.h -- the 32x32 form of the batched GEMM (qgemm_wide.hip) as its
// dispatcher (qgemm.hip) sees it.
#pragma once

#include "common.h"

namespace qraf_hip {
// sets the dynamic-LDS attribute of every form (qraf_hip_init)
int qgemm_wide_init();
// a form's tile (batch rows x weight rows) and K groups (pairs of blocks per iteration)
struct QwTile {
    int mt, nt, wk;
};
constexpr int QW_FORM_COUNT = 4;
QwTile qgemm_wide_tile(int form);
// Y (+ add), or with S > 1 S partial slices [S][M][N] of bps blocks (even) each,
// or with act_hi / act_lo (S 1) the SwiGLU planes of interleaved gate/up rows
int launch_qgemm_wide(int form, const void* Wt, uint32_t dtype, int N, int K, const uint16_t* xh, const uint16_t* xl,
                      int M, float* Y, const float* add, int S, int bps, uint16_t* act_hi, uint16_t* act_lo,
                      hipStream_t s);
}  // namespace qraf_hip
