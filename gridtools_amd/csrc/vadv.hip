// Vertical advection entry points: argument checks, the no-allocation form's scratch, the dispatch by type to
// vadv_f64.hip, vadv_mixed.hip and vadv_f32.hip (kernels and launch: vadv_launch.hpp, column.hpp).
#include <hip/hip_runtime.h>

#include <mutex>

#include "common.hpp"

namespace gt355 {
    // ext_buf == nullptr: scratch from the stream's pool, else ext_bytes at ext_buf (vadv_launch.hpp: launch_vadv)
#define GT355_VADV_DECL(name)                                                                                    \
    int name(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,         \
        const gt355_field *ut, double dtr_stage, int ni, int nj, int nk, hipStream_t stream, void *ext_buf,       \
        size_t ext_bytes)
    GT355_VADV_DECL(vadv_f64);
    GT355_VADV_DECL(vadv_mixed);
    GT355_VADV_DECL(vadv_f32);
#undef GT355_VADV_DECL

    namespace {
        // The no-allocation entry point's ccol/dcol buffer: a file-scope device array, one copy per device for the
        // life of the process.  Host code never uses its name as an address (on the host it names a stand-in): the
        // device address comes from hipGetSymbolAddress, once per device, with that device current.
        constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(64) << 20;
        static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

        constexpr int NOALLOC_MAX_DEVICES = 64;
        std::mutex g_noalloc_mutex;
        void *g_noalloc_ptr[NOALLOC_MAX_DEVICES] = {};

        // The current device's address of `scratch`.
        int noalloc_scratch(void **out) {
            int dev = 0;
            GT355_HIP(hipGetDevice(&dev));
            GT355_CHECK(dev >= 0 && dev < NOALLOC_MAX_DEVICES, "gt355_vadv_noalloc: device %d", dev);
            std::lock_guard<std::mutex> lock(g_noalloc_mutex);
            if (!g_noalloc_ptr[dev]) {
                void *p = nullptr;
                hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
                if (e != hipSuccess)
                    return hip_fail(e, "gt355_vadv_noalloc: hipGetSymbolAddress(scratch)");
                GT355_CHECK(p != nullptr, "gt355_vadv_noalloc: no device address for the static scratch");
                g_noalloc_ptr[dev] = p;
            }
            *out = g_noalloc_ptr[dev];
            return GT355_OK;
        }
    } // namespace

    // Called by gt355_init with the selected device current: resolves the static scratch's address there.
    int noalloc_setup() {
        void *p = nullptr;
        return noalloc_scratch(&p);
    }
} // namespace gt355

using namespace gt355;

namespace {
    int vadv_entry(int precision, const gt355_field *utens_stage, const gt355_field *u_stage, const gt355_field *wcon,
        const gt355_field *u_pos, const gt355_field *utens, double dtr_stage, int ni, int nj, int nk, void *stream,
        bool noalloc) {
    GT355_CHECK(ni >= 0 && nj >= 0, "gt355_vadv: negative size");
    GT355_CHECK(nk >= 2, "gt355_vadv: nk = %d, the spec needs at least 2 levels (first and last level)", nk);
    GT355_CHECK(utens_stage && u_stage && wcon && u_pos && utens, "gt355_vadv: null field");
    if (ni == 0 || nj == 0)
        return GT355_OK;
    int dtype = utens_stage->dtype;
    GT355_CHECK(dtype == GT355_F64 || dtype == GT355_F32, "gt355_vadv: dtype %d", dtype);
    GT355_CHECK(precision == GT355_NATIVE || (precision == GT355_WIDEN && dtype == GT355_F32),
        "gt355_vadv: precision %d with dtype %d", precision, dtype);
    int rc;
    if ((rc = check_field(utens_stage, "utens_stage", dtype, 0, ni, 0, nj, 0, nk)))
        return rc;
    if ((rc = check_field(u_stage, "u_stage", dtype, 0, ni, 0, nj, 0, nk)))
        return rc;
    if ((rc = check_field(wcon, "wcon", dtype, 0, ni + 1, 0, nj, 0, nk)))
        return rc;
    if ((rc = check_field(u_pos, "u_pos", dtype, 0, ni, 0, nj, 0, nk)))
        return rc;
    if ((rc = check_field(utens, "utens", dtype, 0, ni, 0, nj, 0, nk)))
        return rc;
    // inside a deferred-run scope gt355_vadv is recorded and runs at the scope's flush; the no-allocation entry
    // point always runs at once (the flush may build a batch), after what the scope recorded before it
    if (!noalloc && defer_active(stream))
        return defer_vadv(precision, utens_stage, u_stage, wcon, u_pos, utens, dtr_stage, ni, nj, nk, stream);
    if (noalloc && (rc = defer_flush(stream)))
        return rc;
    hipStream_t s = (hipStream_t)stream;
    void *buf = nullptr;
    const size_t bytes = noalloc ? NOALLOC_SCRATCH_BYTES : 0;
    if (noalloc && (rc = noalloc_scratch(&buf)))
        return rc;
    if (dtype == GT355_F64)
        return vadv_f64(utens_stage, u_stage, wcon, u_pos, utens, dtr_stage, ni, nj, nk, s, buf, bytes);
    if (precision == GT355_WIDEN)
        return vadv_mixed(utens_stage, u_stage, wcon, u_pos, utens, dtr_stage, ni, nj, nk, s, buf, bytes);
    return vadv_f32(utens_stage, u_stage, wcon, u_pos, utens, dtr_stage, ni, nj, nk, s, buf, bytes);
    }
} // namespace

extern "C" int gt355_vadv(int precision, const gt355_field *utens_stage, const gt355_field *u_stage,
    const gt355_field *wcon, const gt355_field *u_pos, const gt355_field *utens, double dtr_stage, int ni, int nj,
    int nk, void *stream) {
    return vadv_entry(precision, utens_stage, u_stage, wcon, u_pos, utens, dtr_stage, ni, nj, nk, stream, false);
}

extern "C" int gt355_vadv_noalloc(int precision, const gt355_field *utens_stage, const gt355_field *u_stage,
    const gt355_field *wcon, const gt355_field *u_pos, const gt355_field *utens, double dtr_stage, int ni, int nj,
    int nk, void *stream) {
    return vadv_entry(precision, utens_stage, u_stage, wcon, u_pos, utens, dtr_stage, ni, nj, nk, stream, true);
}
