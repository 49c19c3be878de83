// The vertical advection by two wavefronts per strip: the launches (nk of 33 to 144 levels, every field below 4 GiB, one
// layout for every field but wcon; the caller checks), one per form in vadv_duo_*.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace gt355 {
    int vadv_duo_f64(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,
        const gt355_field *ut, double dtr, int ni, int nj, int nk, hipStream_t stream);
    int vadv_duo_mixed(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,
        const gt355_field *ut, double dtr, int ni, int nj, int nk, hipStream_t stream);
    // dtr: a float's value
    int vadv_duo_f32(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,
        const gt355_field *ut, double dtr, int ni, int nj, int nk, hipStream_t stream);
} // namespace gt355
