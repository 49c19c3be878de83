// Vertical advection by two wavefronts per strip, FP64 (vadv_duo_launch.hpp).
#include "vadv_duo_launch.hpp"

namespace gt355 {
    int vadv_duo_f64(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,
        const gt355_field *ut, double dtr, int ni, int nj, int nk, hipStream_t stream) {
        return launch_duo<double, double>(uts, us, wc, up, ut, dtr, ni, nj, nk, stream);
    }
} // namespace gt355
