// The kernel of vadv_duo.hpp and its launch for one storage and compute type.
#pragma once

#include <hip/hip_runtime.h>

#include "column_duo.hpp"
#include "common.hpp"
#include "vadv_duo.hpp"

namespace gt355 {
    namespace {
        // Two wavefronts per strip (column_duo.hpp), one strip per workgroup.
        template <class ST, class CT, int NBLK>
        __global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1, 1)))
        vadv_duo_kernel(ST *__restrict__ uts_f, const ST *__restrict__ us_f, const ST *__restrict__ wc_f,
            const ST *__restrict__ up_f, const ST *__restrict__ ut_f, CT dtr, int ni, int nk, int64_t sj, int64_t sk,
            int64_t wsj, int64_t wsk, int strips_i, int nxcd) {
            using duo = column_duo<ST, CT, NBLK>;
            __shared__ typename duo::shared sh;
            const int it = xcd_remap(blockIdx.x, gridDim.x, nxcd);
            const int lane = threadIdx.x & 63;
            // (wave-uniform: the two roles are branches, not masks)
            if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0) {
                const int si = it % strips_i, j = it / strips_i;
                // lanes past ni take column ni-1, computing and storing its bits again
                const int i = min(si * 64 + lane, ni - 1);
                const column_src f{make_rsrc(uts_f), make_rsrc(us_f), make_rsrc(wc_f), make_rsrc(up_f),
                    make_rsrc(ut_f), (uint32_t)(sk * (int64_t)sizeof(ST)), (uint32_t)(wsk * (int64_t)sizeof(ST)), nk};
                duo::coefficients(f, dtr, (uint32_t)(((int64_t)j * sj + i) * (int64_t)sizeof(ST)),
                    (uint32_t)(((int64_t)j * wsj + i) * (int64_t)sizeof(ST)), sh, lane);
            } else {
                duo::recurrence(nk, dtr, sh, lane);
            }
        }

        // One instantiation per number of 8-level blocks.
        template <class ST, class CT, int NBLK>
        int launch_duo_blocks(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,
            const gt355_field *ut, double dtr, int ni, int nj, int nk, hipStream_t stream) {
            const int strips_i = (ni + 63) / 64;
            vadv_duo_kernel<ST, CT, NBLK><<<strips_i * nj, 128, 0, stream>>>((ST *)uts->origin, (const ST *)us->origin,
                (const ST *)wc->origin, (const ST *)up->origin, (const ST *)ut->origin, CT(dtr), ni, nk, uts->stride[1],
                uts->stride[2], wc->stride[1], wc->stride[2], strips_i, xcd_count());
            return check_launch("gt355_vadv");
        }

        template <class ST, class CT>
        int launch_duo(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,
            const gt355_field *ut, double dtr, int ni, int nj, int nk, hipStream_t stream) {
            switch ((nk + 7) / 8) {
#define GT355_DUO(N)                                                                                            \
    case N:                                                                                                     \
        return launch_duo_blocks<ST, CT, N>(uts, us, wc, up, ut, dtr, ni, nj, nk, stream);
                GT355_DUO(5) GT355_DUO(6) GT355_DUO(7) GT355_DUO(8) GT355_DUO(9) GT355_DUO(10) GT355_DUO(11)
                GT355_DUO(12) GT355_DUO(13) GT355_DUO(14) GT355_DUO(15) GT355_DUO(16) GT355_DUO(17)
                GT355_DUO(18)
#undef GT355_DUO
            }
            set_error("gt355_vadv: nk %d has no two-wavefront kernel", nk);
            return GT355_EUNSUP;
        }
    } // namespace
} // namespace gt355
