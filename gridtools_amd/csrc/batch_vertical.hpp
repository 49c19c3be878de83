// The vertical phase of the two-phase batching form: the column sweep (column.hpp) over the strips of many domains of
// different depths in one persistent launch.  Instantiated by vadv_f64.hip, vadv_mixed.hip and vadv_f32.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "column.hpp"
#include "common.hpp"

namespace gt355 {

    // One domain of a batch.
    struct bdom {
        const void *in, *coeff, *wcon, *u_pos, *utens;
        void *lap, *u_stage, *utens_stage;
        int64_t sj, sk;   // shared layout of every field but wcon (origins at grid point (0,0,0))
        int64_t wsj, wsk; // wcon layout
        int32_t ni, nj, nk, tiles_i;
    };

    // Work item: 64 columns (from i0) of row j of one domain.
    struct sitem {
        int32_t dom, i0, j, pad;
    };

    // The items' depth classes, deepest first: class n takes depths above vertical_above(n) up to the class before it.
    constexpr int VCLASSES = 8;
    // Depths of at most VMAXK; the levels below the top block of 8 that a wavefront of the vertical phase keeps in its
    // scratch, past the 128 that the deepest split (FP64 arithmetic, from 81 or 113 levels) has in registers and LDS.
    constexpr int VMAXK = 144, VTAIL_ROWS = (VMAXK - 128 - 1) / 8 * 8;
    struct vertical_plan {
        int end[VCLASSES]; // items are sorted by class: those of class n end here
    };
    constexpr int vertical_above(int n) {
        constexpr int above[VCLASSES] = {112, 80, 72, 64, 56, 48, 40, 0};
        return above[n];
    }

    // Launches the vertical phase (grid wavefronts, each striding through the items) on `stream`.
    void batch_vertical_f64(const bdom *doms, const sitem *items, const vertical_plan &plan, int grid, double dtr,
        void *scratch, int nxcd, hipStream_t stream);
    void batch_vertical_mixed(const bdom *doms, const sitem *items, const vertical_plan &plan, int grid, double dtr,
        void *scratch, int nxcd, hipStream_t stream);
    void batch_vertical_f32(const bdom *doms, const sitem *items, const vertical_plan &plan, int grid, float dtr,
        void *scratch, int nxcd, hipStream_t stream);

    namespace {
        // A wavefront's items of one class, from `it` on; leaves the first item past the class in `it`.
        template <class ST, class CT, int R, int D, int TL, int NB, bool PARK, bool DEEP, int MINK = R + TL + 1>
        __device__ __forceinline__ void vertical_class(const bdom *__restrict__ doms, const sitem *__restrict__ items,
            int end, int &it, CT dtr, char *lds, rsrc_t sc) {
            if (it >= end)
                return;
            asm volatile("" ::: "memory"); // the classes share the LDS under different types
            ST(*s_up)[64] = (ST(*)[64])lds;
            CT *s_tail = (CT *)(lds + (PARK ? (R + TL) * 64 * sizeof(ST) : 0));
            auto take = [&](int n, column_src &f, uint32_t &cb, uint32_t &wb) {
                const sitem e = items[n];
                const bdom &m = doms[e.dom];
                f = column_src{make_rsrc(m.utens_stage), make_rsrc(m.u_stage), make_rsrc(m.wcon), make_rsrc(m.u_pos),
                    make_rsrc(m.utens), (uint32_t)(m.sk * (int64_t)sizeof(ST)),
                    (uint32_t)(m.wsk * (int64_t)sizeof(ST)), m.nk};
                // lanes past ni take column ni-1, computing and storing its bits again
                const int i = min(e.i0 + (int)threadIdx.x, m.ni - 1);
                cb = (uint32_t)((e.j * m.sj + i) * (int64_t)sizeof(ST));
                wb = (uint32_t)((e.j * m.wsj + i) * (int64_t)sizeof(ST));
            };
            column_sweep<ST, CT, R, D, TL, NB, PARK, DEEP, MINK> sw;
            column_src f;
            uint32_t cb, wb;
            take(it, f, cb, wb);
            sw.prologue(f, cb, wb);
            for (;;) {
                const int nx = it + (int)gridDim.x;
                column_src nf = f;
                uint32_t ncb = cb, nwb = wb;
                sw.sweep(f, dtr, cb, wb, s_up, s_tail, sc, [&]() {
                    if (nx < end) {
                        take(nx, nf, ncb, nwb);
                        sw.prologue(nf, ncb, nwb);
                    }
                });
                it = nx;
                if (nx >= end)
                    break;
                f = nf;
                cb = ncb;
                wb = nwb;
            }
        }

        // One wavefront per SIMD walks the items (deepest first) with a static stride, no counters; the classes follow each
        // other in the code, each a loop over its items with the loads of the next item started in the sweep before, so
        // a wavefront fills its pipeline once per class.  Measured against one sweep of 80 clamped steps with the levels past
        // them through scratch (16 domains of 48..384 x 48..384 x 40..137 points, 60 M in all): FP32 storage, FP64
        // compute 338 -> 282 us, 5.5 TB/s of the 1.56 GB it moves (a tenth more than the fields' bytes: partial strips
        // and the wcon line shared by neighbours).  Bound by the memory; a launch per round of strips was slower (6
        // domains 356 us against 343 for both phases), 4 levels of load-ahead about the same (533 against 529).
        template <class ST, class CT>
        __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1)))
        batch_vertical_kernel(const bdom *__restrict__ doms, const sitem *__restrict__ items, vertical_plan plan,
            CT dtr, CT *__restrict__ scratch, int nxcd) {
            constexpr bool F32 = sizeof(CT) == 4, S32 = sizeof(ST) == 4;
            // u_pos of R + TL levels and ccol/dcol of TL levels, at most a quarter of the CU's LDS
            __shared__ __attribute__((aligned(16))) char lds[40 << 10];
            const rsrc_t sc = make_rsrc(scratch + (int64_t)blockIdx.x * (VTAIL_ROWS * 128));
            int it = xcd_remap_groups(blockIdx.x, gridDim.x, nxcd, XCD_GROUP);
#define GT355_VCLASS(N, ...) vertical_class<ST, CT, __VA_ARGS__>(doms, items, plan.end[N], it, dtr, lds, sc)
            if constexpr (F32) {
                GT355_VCLASS(0, 136, 8, 0, 32, true, false, 113);
                GT355_VCLASS(1, 104, 8, 0, 32, true, false, 81);
            } else if constexpr (S32) {
                GT355_VCLASS(0, 88, 8, 40, 16, false, true, 113);
                GT355_VCLASS(1, 96, 8, 8, 32, true, false, 81);
            } else {
                GT355_VCLASS(1, 88, 4, 40, 16, false, true, 81); // with class 0
            }
            GT355_VCLASS(2, 72, 8, 0, 32, true, false);
            GT355_VCLASS(3, 64, 8, 0, 32, true, false);
            GT355_VCLASS(4, 56, 8, 0, 32, true, false);
            GT355_VCLASS(5, 48, 8, 0, 32, true, false);
            GT355_VCLASS(6, 40, 8, 0, 32, true, false);
            GT355_VCLASS(7, 32, 8, 0, 32, true, false, 2);
#undef GT355_VCLASS
        }

        template <class ST, class CT>
        void launch_batch_vertical(const bdom *doms, const sitem *items, const vertical_plan &plan, int grid, CT dtr,
            void *scratch, int nxcd, hipStream_t stream) {
            batch_vertical_kernel<ST, CT><<<grid, 64, 0, stream>>>(doms, items, plan, dtr, (CT *)scratch, nxcd);
        }
    } // namespace
} // namespace gt355
