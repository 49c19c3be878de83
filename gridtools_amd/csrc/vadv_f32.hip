// Vertical advection, FP32 storage and compute (vadv_launch.hpp), and the batching form's vertical phase (batch_vertical.hpp).
#include "batch_vertical.hpp"
#include "vadv_launch.hpp"

namespace gt355 {
    int vadv_f32(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,
        const gt355_field *ut, double dtr_stage, int ni, int nj, int nk, hipStream_t stream, void *ext_buf,
        size_t ext_bytes) {
        return launch_vadv<float, float>(uts, us, wc, up, ut, dtr_stage, ni, nj, nk, stream, ext_buf, ext_bytes);
    }
    void batch_vertical_f32(const bdom *doms, const sitem *items, const vertical_plan &plan, int grid, float dtr,
        void *scratch, int nxcd, hipStream_t stream) {
        launch_batch_vertical<float, float>(doms, items, plan, grid, dtr, scratch, nxcd, stream);
    }
} // namespace gt355
