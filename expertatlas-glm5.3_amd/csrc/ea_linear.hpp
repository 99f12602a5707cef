// What the EXL3 linear's two sources share: the input rotation launch, the launches for any number of rows up to 128,
// and the finish of a 128-column block.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ea_device.hpp"
#include "ea_exl3.h"

namespace ea {

// xh_j [m, kdim] of each job (ea_exl3_rot_in).
int launch_lin_rot_in(hipStream_t s, const void* x, int x_dtype, const ea_rot_jobs* jobs, uint32_t njobs, uint32_t m,
                      uint32_t kdim);

// One linear over the jobs for m rows (1 to 128), any split count: ea_linear_rows.hip. rot: the jobs' rotation when x is
// the unrotated input (kdim % 128 == 0).
int launch_linear_rows(hipStream_t s, const ea_jobs& jobs, const ea_rot_jobs* rot, int m, int kdim, uint32_t k2,
                       uint32_t cb, const void* x, int x_dtype);

// One row's 128 outputs of a column block from their fp32 sums (two a lane; svh and bias already loaded as two fp16 a
// word): FWHT, * HAD_SCALE * svh (+ bias), stored as y_dtype (exl3_linear.cu:69-81).
__device__ __forceinline__ void finish_store_pre(float v0, float v1, int lane, uint32_t sw, bool has_bias, uint32_t bw,
                                                 void* y, int y_dtype, size_t at) {
    fwht128_w64(v0, v1, lane);
    v0 = v0 * HAD_SCALE * h2f((uint16_t)(sw & 0xffffu));
    v1 = v1 * HAD_SCALE * h2f((uint16_t)(sw >> 16));
    if (has_bias) {
        v0 += h2f((uint16_t)(bw & 0xffffu));
        v1 += h2f((uint16_t)(bw >> 16));
    }
    store_act(y, y_dtype, at, v0);
    store_act(y, y_dtype, at + 1, v1);
}

}  // namespace ea
