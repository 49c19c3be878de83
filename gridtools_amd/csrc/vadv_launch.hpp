// Vertical advection (implicit tridiagonal Thomas solve per column) for gfx950: the kernels and their launch for one
// storage and compute type, instantiated by vadv_f64.hip, vadv_mixed.hip and vadv_f32.hip.
//
// Reference: tests/regression/vertical_advection_dycore.cpp:32-150.  The spec is
//   multi_pass(execute_forward().k_cached(flush, ccol, dcol).k_cached(fill, u_stage).stage(u_forward...),
//              execute_backward().k_cached(data_col).stage(u_backward...))
// and the reference gpu backend fuses both multistages into one launch (stencil/gpu/entry_point.hpp:48-59,
// 107-124) with one thread per column, u_stage/data_col in register rings (gpu/k_cache.hpp:23-46) and
// ccol/dcol flushed to HBM temporaries that the backward sweep reads back (gpu/fill_flush.hpp:298-321).
//
// Here, too, one lane owns one column and both sweeps run in one launch (column.hpp), with the k-caches in VGPRs and
// ccol/dcol on chip as far as it holds them: registers, then LDS, then the wavefront's scratch.  Fields that span 4 GiB
// or more, past the 32-bit buffer offsets, take vadv_scratch_kernel: ccol/dcol in a per-launch scratch buffer in the
// k-major layout the lanes read coalesced.
// Results are the functors', operation by operation (built with -ffp-contract=off).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "column.hpp"
#include "common.hpp"
#include "functors.hpp"
#include "vadv_duo.hpp"

namespace gt355 {
    namespace {

        // One column per lane; ccol/dcol of levels 0..nk-2 go to scratch (k-major, column-minor).
        template <class ST, class CT>
        __global__ void __launch_bounds__(256) vadv_scratch_kernel(ST *__restrict__ uts_f,
            const ST *__restrict__ us_f, const ST *__restrict__ wc_f, const ST *__restrict__ up_f,
            const ST *__restrict__ ut_f, CT dtr, int ni, int nj, int nk, int64_t sj, int64_t sk, int64_t wsj,
            int64_t wsk, CT *__restrict__ cd_buf, int64_t plane) {
            const int i = blockIdx.x * 64 + (threadIdx.x & 63);
            const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
            if (i >= ni || j >= nj)
                return;
            const int64_t col = (int64_t)j * sj + i;
            const int64_t wcol = (int64_t)j * wsj + i;
            const int64_t scol = (int64_t)j * ni + i; // scratch column index, plane = ni*nj
            CT *__restrict__ sc = cd_buf + scol;
            CT *__restrict__ sd = cd_buf + (int64_t)(nk - 1) * plane + scol;

            // k = 0
            CT us_c = CT(us_f[col]);
            CT us_p = CT(us_f[col + sk]);
            CT w_p_i = CT(wc_f[wcol + wsk]);
            CT w_p_ip = CT(wc_f[wcol + wsk + 1]);
            CT up = CT(up_f[col]);
            fwd_out<CT> r = forward_first<CT>(dtr, w_p_i, w_p_ip, us_c, us_p, up, CT(ut_f[col]), CT(uts_f[col]));
            sc[0] = r.c;
            sd[0] = r.d;
            CT cc_m = r.c, dc_m = r.d;
#pragma unroll 4
            for (int k = 1; k < nk - 1; ++k) {
                const int64_t p = col + (int64_t)k * sk;
                CT us_m = us_c;
                us_c = us_p;
                us_p = CT(us_f[p + sk]);
                CT w_c_i = w_p_i, w_c_ip = w_p_ip;
                w_p_i = CT(wc_f[wcol + (int64_t)(k + 1) * wsk]);
                w_p_ip = CT(wc_f[wcol + (int64_t)(k + 1) * wsk + 1]);
                up = CT(up_f[p]);
                r = forward_body<CT>(dtr, w_c_i, w_c_ip, w_p_i, w_p_ip, us_m, us_c, us_p, up, CT(ut_f[p]),
                    CT(uts_f[p]), cc_m, dc_m, false);
                sc[(int64_t)k * plane] = r.c;
                sd[(int64_t)k * plane] = r.d;
                cc_m = r.c;
                dc_m = r.d;
            }
            // k = nk-1
            {
                const int64_t p = col + (int64_t)(nk - 1) * sk;
                CT us_m = us_c;
                us_c = us_p;
                up = CT(up_f[p]);
                CT dc = forward_last<CT>(
                    dtr, w_p_i, w_p_ip, us_m, us_c, up, CT(ut_f[p]), CT(uts_f[p]), cc_m, dc_m);
                // u_backward_function::apply(last_level) (vertical_advection_dycore.cpp:117-121)
                uts_f[p] = ST(dtr * (dc - up));
                CT data = dc;
                // u_backward_function::apply(modify<0,-1>) (vertical_advection_dycore.cpp:110-115)
#pragma unroll 4
                for (int k = nk - 2; k >= 0; --k) {
                    const int64_t q = col + (int64_t)k * sk;
                    CT cc = sc[(int64_t)k * plane];
                    CT dd = sd[(int64_t)k * plane];
                    CT dt = dd - cc * data;
                    uts_f[q] = ST(dtr * (dt - CT(up_f[q])));
                    data = dt;
                }
            }
        }

        // The persistent column sweep: WPE wavefronts per SIMD walk the strips (64 columns of one row; the strips of a row
        // consecutive) with a static stride, so that the wavefronts in flight stay on neighbouring strips.  Each starts
        // the next strip's first D levels of loads NB levels before the end of a strip's backward sweep, so the next
        // forward sweep needs no pipeline fill.  Measured against the former kernels (one level bucket per 16 levels,
        // selects at every level), us: 256x256x80 FP64 37.7 (39.7), mixed 20.4 (21.7); 300x300x40 FP64 28
        // (38), FP32 17 (22); 512x512x40 mixed 40.6 (54.2); 300x300x137 FP64 128 (209 through memory).
        template <class ST, class CT, int R, int D, int TL, int NB, bool PARK, bool DEEP, int MINK, int WPE, int CPOL_W>
        __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
        vadv_column_kernel(ST *__restrict__ uts_f, const ST *__restrict__ us_f, const ST *__restrict__ wc_f,
            const ST *__restrict__ up_f, const ST *__restrict__ ut_f, CT dtr, int ni, int nk, int64_t sj, int64_t sk,
            int64_t wsj, int64_t wsk, int strips_i, int first, int nitems, int nxcd,
            CT *scratch, int tail_rows) {
            __shared__ ST s_up[PARK ? R + TL : 1][64];
            __shared__ CT s_tail[TL > 0 ? TL * 128 : 1];
            column_src f{make_rsrc(uts_f), make_rsrc(us_f), make_rsrc(wc_f), make_rsrc(up_f), make_rsrc(ut_f),
                (uint32_t)(sk * (int64_t)sizeof(ST)), (uint32_t)(wsk * (int64_t)sizeof(ST)), nk};
            const rsrc_t sc = make_rsrc(scratch + (int64_t)blockIdx.x * tail_rows * 128);
            // the lane's byte offsets in strip `it` (lanes past ni take column ni-1, computing and storing its bits again)
            auto offsets = [&](int it, uint32_t &cb, uint32_t &wb) {
                const int si = it % strips_i, j = it / strips_i;
                const int i = min(si * 64 + (int)threadIdx.x, ni - 1);
                cb = (uint32_t)(((int64_t)j * sj + i) * (int64_t)sizeof(ST));
                wb = (uint32_t)(((int64_t)j * wsj + i) * (int64_t)sizeof(ST));
            };
            int it = first + xcd_remap(blockIdx.x, gridDim.x, nxcd);
            if (it >= nitems)
                return; // a whole wavefront leaves; there is no barrier in this kernel
            column_sweep<ST, CT, R, D, TL, NB, PARK, DEEP, MINK, CPOL_W> sw;
            uint32_t cb, wb;
            offsets(it, cb, wb);
            sw.prologue(f, cb, wb);
            for (; it < nitems; it += gridDim.x) {
                const int nx = it + (int)gridDim.x;
                uint32_t ncb = cb, nwb = wb;
                sw.sweep(f, dtr, cb, wb, s_up, s_tail, sc, [&]() {
                    if (nx < nitems) {
                        offsets(nx, ncb, nwb);
                        sw.prologue(f, ncb, nwb);
                    }
                });
                cb = ncb;
                wb = nwb;
            }
        }

        template <class ST, class CT>
        struct vadv_args {
            const gt355_field *uts, *us, *wc, *up, *ut;
            CT dtr;
            int ni, nj, nk;
            hipStream_t stream;
            // scratch: the caller's buffer of ext_bytes, or the stream's pool; shape: ccol/dcol of all columns (nk > 80)
            void *ext;
            size_t ext_bytes, shape;
        };

        // The pool's buffer for launches that use `bytes` of it.  Never less than 64 MiB or, if that is less, the shape's
        // ccol/dcol: the launches of any shape of no more ccol/dcol then fit a buffer that it finds while it is captured,
        // in fewer wavefronts or in chunks of rows.
        template <class ST, class CT>
        int pool_scratch(const vadv_args<ST, CT> &a, size_t bytes, void **buf, size_t *have) {
            return scratch_for(a.stream, std::max(bytes, std::min(a.shape, size_t(64) << 20)), a.shape, buf, have);
        }

        // Launches one instantiation: at most WPE wavefronts per SIMD, fewer if the scratch of the levels past R + TL
        // would exceed the caller's buffer or, of the pool, 256 MiB and the shape's ccol/dcol, and as many launches as keep
        // each at `rounds` strips per wavefront (0: one launch).  Returns false, launching nothing, if not even a quarter of
        // the wavefronts fit.  Where under half the lanes have a column the time is the rounds', not the memory's, and
        // vadv_scratch_kernel, which runs all strips at once, takes those that would need more rounds for lack of scratch (us,
        // wavefronts as the shape's ccol/dcol hold / all / vadv_scratch_kernel: FP64 3x4096x300 859 / 519 / 564, FP32
        // 2x4096x300 938 / 319 / 323) and, over several rounds, those with half as many levels again in scratch as on chip
        // (FP64 16x4096x300 542 against 526, 400 levels 788 and 707; FP32 320 and 319, 474 and 430).
        template <class ST, class CT, int R, int D, int TL, int NB, bool PARK, bool DEEP, int MINK, int WPE,
            int CPOL_W = 0>
        bool launch_column_as(const vadv_args<ST, CT> &a, int rounds, int *rc) {
            const int strips_i = (a.ni + 63) / 64;
            const int64_t items = (int64_t)strips_i * a.nj;
            if (items >= (int64_t(1) << 31) - (1 << 20))
                return false;
            const int tail_rows = DEEP && a.nk > R + TL + 8 ? (a.nk - R - TL - 1) / 8 * 8 : 0;
            const size_t wave_bytes = (size_t)tail_rows * 128 * sizeof(CT);
            const int64_t want = std::min<int64_t>(items, (int64_t)cu_count() * 4 * WPE);
            auto fit = [&](size_t bytes) -> int64_t {
                const int64_t n = wave_bytes ? std::min<int64_t>(want, (int64_t)(bytes / wave_bytes)) : want;
                const bool few_lanes = a.ni < strips_i * 32, deep = tail_rows * 2 >= (R + TL + 8) * 3;
                return n * 4 < want || (few_lanes && (n < want || (deep && want < items))) ? 0 : n;
            };
            void *buf = a.ext;
            int64_t waves = fit(a.ext ? a.ext_bytes : std::max(a.shape, size_t(256) << 20));
            *rc = GT355_OK;
            if (DEEP && waves && !a.ext) {
                size_t have = 0;
                if ((*rc = pool_scratch(a, waves * wave_bytes, &buf, &have)))
                    return true;
                waves = fit(have);
            }
            if (waves < 1)
                return false;
            // launches of equal length
            const int64_t nlaunch = rounds ? (items + waves * rounds - 1) / (waves * rounds) : 1;
            const int64_t per = (items + nlaunch - 1) / nlaunch;
            for (int64_t first = 0; first < items && *rc == GT355_OK; first += per) {
                const int64_t end = std::min(items, first + per);
                vadv_column_kernel<ST, CT, R, D, TL, NB, PARK, DEEP, MINK, WPE, CPOL_W>
                    <<<(int)std::min(waves, end - first), 64, 0, a.stream>>>((ST *)a.uts->origin,
                        (const ST *)a.us->origin, (const ST *)a.wc->origin, (const ST *)a.up->origin,
                        (const ST *)a.ut->origin, a.dtr, a.ni, a.nk, a.uts->stride[1], a.uts->stride[2],
                        a.wc->stride[1], a.wc->stride[2], strips_i, (int)first, (int)end, xcd_count(), (CT *)buf,
                        tail_rows);
                *rc = check_launch("gt355_vadv");
            }
            return true;
        }

        // Depths that fit registers: an instantiation per number of 8-level blocks below the top one, and per wavefronts
        // per SIMD and levels of load-ahead where the best of these depends on the number of strips.  Times below in us.
        template <class ST, class CT, int R, int MINK = R + 1>
        bool launch_column_blocks(const vadv_args<ST, CT> &a, int *rc) {
            constexpr bool F32 = sizeof(CT) == 4, S32 = sizeof(ST) == 4;
            constexpr int NB = R < 32 ? R : 32;
            // the most wavefronts per SIMD whose registers hold the column and its rings of 8 levels without spills (three
            // of FP64 up to 16 levels and of the mixed form at 17 to 24 spill: 1024x1024x9 FP64 110 against 90 of two,
            // 1024x1024x20 mixed 97 and 84)
            constexpr int WMAX = F32 ? (R <= 32 ? 3 : 2) : R <= (S32 ? 8 : 0) ? 3 : R <= (S32 ? 40 : 32) ? 2 : 1;
            constexpr int D = !F32 && R <= 32 && R > (S32 ? 24 : 16) ? 4 : 8;
            const int64_t items = (int64_t)((a.ni + 63) / 64) * a.nj, simds = (int64_t)cu_count() * 4;
            // Wavefronts per SIMD: a round of w takes about w times a round of one, so the fewest rounds times w, as many
            // as possible unless fewer save an eighth (400x400x40 FP64, 2.7 strips per SIMD: three rounds of one 50.9, two
            // of two 59.8; 400x400x40 FP32: one of three 26.2, three of one 29.5; 512x512x16 FP32, 4 strips per SIMD:
            // two of two 16, two of three 20).
            auto rounds = [&](int w) { return (items + simds * w - 1) / (simds * w); };
            int w = WMAX;
            for (int v = WMAX - 1; v >= 1; --v)
                if (rounds(v) * v * 8 < rounds(w) * w * 7)
                    w = v;
            // (FP64 of 9 to 16 levels over many rounds: one, which starts its next strip's loads sooner; 1400x1400x12 189
            // against 197 of two, over rotating fields 213 and 223, 1024x1024x9 87 and 90; 700x700x9, 7.5 strips per SIMD, 45 and 45)
            if (!S32 && R == 8 && MINK > 8 && items > simds * 12)
                w = 1;
            // A launch per round for large fields: over many rounds in one launch the wavefronts drift apart, and the
            // memory with them (one launch against one per round: 512x512x80 FP64 161 and 152, 1024x1024x80 744 and 686,
            // 1536x1536x80 mixed 938 and 824, FP32 925 and 836); smaller or shallower ones lose the wavefronts' overlap at
            // the rounds' ends (512x512x40 FP64 77.0 and 78.8; 900x900x80 mixed 294 and 307, but 1024x1024x80 356 and 346).
            const int64_t bytes = items * 64 * a.nk * (int64_t)sizeof(ST);
            // FP64 also where two launches have three quarters of the SIMDs or fewer each: one launch makes some wavefronts
            // solve two strips while others solve one, and all reads compete meanwhile (one launch against two: 300x300x80 65.6
            // and 58.7, over rotating fields 66.2 and 59.5, after hdiff 102 and 96; 256x350x56 45.8 and 40.9; 1600 strips
            // 256x400x80 70.5 and 68.9, 256x400x44 42.3 and 42.2; 1030 strips 64x1030x80 47.1 and 51.7)
            const bool halves = !S32 && R >= 40 && w == 1 && items * 8 >= simds * 9 && items * 2 <= simds * 3;
            const int per_launch =
                halves || (w < 3 && a.nk >= 32 && bytes >= ((F32 || !S32 ? 150LL : 300LL) << 20)) ? 1 : 0;
            // Where three wavefronts spill with 8 levels ahead, three with 4, which do not, if they run all strips in one round
            // (400x400x8 FP64 10.2 against 11.6 with 8 ahead, 14.1 of two wavefronts; 360x360x12 14.3, 17.2 and 17.7; 360x360x20 mixed
            // 13.5, 15.7 and 16.3)
            if constexpr (!F32 && WMAX == 2 && R <= (S32 ? 16 : 8))
                if (items > simds * 2 && items <= simds * 3)
                    return launch_column_as<ST, CT, R, 4, 0, NB, true, false, MINK, 3>(a, 0, rc);
            if constexpr (WMAX >= 3)
                if (w == 3)
                    return launch_column_as<ST, CT, R, D, 0, NB, true, false, MINK, 3>(a, per_launch, rc);
            if constexpr (WMAX >= 2)
                if (w == 2)
                    return launch_column_as<ST, CT, R, (R >= 40 ? 4 : D), 0, NB, true, false, MINK, 2>(
                        a, per_launch, rc);
            // FP32 storage, one wavefront per SIMD: 4 levels ahead keep the reads in flight below what the memory takes
            // where more than three of a CU's four SIMDs have one (256x256x80 mixed 20.4 against 22.0 with 8 ahead, 832
            // strips 18.7 and 20.1; 1536x1536x80 in rounds 824 against 843); 8 levels where fewer do (768 strips mixed 17.2
            // against 18.3, FP32 16.7 and 17.5, 256x160x80 FP32 15.3 and 17.3) and, a little, over two to four rounds
            // (512x512x80 79.6 against 80.3, 400x400x80 54.4 against 56.0).  FP64: 8 (64x64x80 on
            // one wavefront per strip 12.1 against 14.2).
            if constexpr (S32 && R >= 40)
                if (items * 4 > simds * 3 && (items <= simds || items > simds * 4))
                    return launch_column_as<ST, CT, R, 4, 0, NB, true, false, MINK, 1>(a, per_launch, rc);
            // FP64, all strips at once: the neighbours' lines are shared in flight, so wcon need not stay in the caches,
            // where other stencils' fields do (hdiff and this in turn, 256x256x80: 65.7 per pair with the default policy,
            // 60.4 non-temporal, each alone 22 and 38; several rounds: 512x512x80 153.9 and 155.3)
            if constexpr (!S32 && R >= 40)
                if (items <= simds)
                    return launch_column_as<ST, CT, R, D, 0, NB, true, false, MINK, 1, CPOL_NT>(a, 0, rc);
            // (the 4 levels of load-ahead of two wavefronts per SIMD are too few where half of the SIMDs or more have no strip:
            // 96x96x32 FP64 6.5 with 4, 6.1 with 8, over rotating fields 7.6 and 6.5; 200x200x32 12.1 and 12.2)
            if constexpr (!S32 && R == 24)
                if (items * 2 <= simds)
                    return launch_column_as<ST, CT, R, 8, 0, NB, true, false, MINK, 1>(a, 0, rc);
            return launch_column_as<ST, CT, R, D, 0, NB, true, false, MINK, 1>(a, per_launch, rc);
        }

        template <class ST, class CT>
        bool launch_column(const vadv_args<ST, CT> &a, int *rc) {
            const int nk = a.nk;
            // At most half as many strips as SIMDs: two wavefronts per strip, from 33 levels on (us, one against two: FP64
            // 64x64x40 7.3 and 6.6, 64x64x80 12.1 and 10.8, 256x128x80, 512 strips, 20.9 and 20.1, 192x160x137 34.7 and
            // 31.9; mixed 256x128x80 14.3 and 12.7, 128x128x137 24.4 and 19.6; FP32 256x128x80 14.2 and 11.6.  20 levels
            // FP64 256x128 6.4 and 6.9; 640 strips, 256x160x80 FP64, 27.2 and 31.9).
            if (nk > 32 && nk <= 144 && (int64_t)((a.ni + 63) / 64) * a.nj * 2 <= (int64_t)cu_count() * 4) {
                // (past 80 levels the pool is asked as by the other kernels, so that what a capture refuses does not
                // depend on the domain's size)
                void *buf;
                size_t have;
                if (nk > 80 && !a.ext && (*rc = pool_scratch(a, 0, &buf, &have)))
                    return true;
                constexpr auto duo = std::is_same_v<ST, CT> ? (sizeof(CT) == 8 ? vadv_duo_f64 : vadv_duo_f32)
                                                            : vadv_duo_mixed;
                *rc = duo(a.uts, a.us, a.wc, a.up, a.ut, a.dtr, a.ni, a.nj, nk, a.stream);
                return true;
            }
#define GT355_COLUMN_BLOCKS(R)                                                                                   \
    if (nk <= R + 8)                                                                                             \
        return launch_column_blocks<ST, CT, R>(a, rc)
            if (nk <= 8)
                return launch_column_blocks<ST, CT, 8, 2>(a, rc); // the block below the top one is left out at run time
            GT355_COLUMN_BLOCKS(8);
            GT355_COLUMN_BLOCKS(16);
            GT355_COLUMN_BLOCKS(24);
            GT355_COLUMN_BLOCKS(32);
            GT355_COLUMN_BLOCKS(40);
            GT355_COLUMN_BLOCKS(48);
            GT355_COLUMN_BLOCKS(56);
            GT355_COLUMN_BLOCKS(64);
            GT355_COLUMN_BLOCKS(72);
#undef GT355_COLUMN_BLOCKS
            // deeper: as many register levels as compile without spills
#define GT355_DEEP(R, D, TL, NB, PARK)                                                                           \
    return launch_column_as<ST, CT, R, D, TL, NB, PARK, true, 81, 1>(a, 0, rc)
            if constexpr (sizeof(CT) == 4) {
                if (nk <= 112)
                    GT355_DEEP(104, 8, 0, 32, true);
                GT355_DEEP(152, 8, 0, 32, true);
            } else if constexpr (sizeof(ST) == 4) {
                // u_pos parked while every level fits beside it
                if (nk <= 112)
                    GT355_DEEP(96, 8, 8, 32, true);
                GT355_DEEP(88, 8, 40, 16, false);
            } else {
                GT355_DEEP(88, 4, 40, 16, false);
            }
#undef GT355_DEEP
        }

        // ext_buf == nullptr: a path that needs ccol/dcol scratch takes it from the per-stream scratch pool.
        // Otherwise ext_buf (ext_bytes long) is used and nothing is allocated: the column sweep launches no more
        // wavefronts than it holds tails for, and vadv_scratch_kernel processes the rows in chunks whose ccol/dcol fit
        // it (columns are independent, so a chunked launch computes the same bits).
        template <class ST, class CT>
        int launch_vadv(const gt355_field *uts, const gt355_field *us, const gt355_field *wc, const gt355_field *up,
            const gt355_field *ut, double dtr_stage, int ni, int nj, int nk, hipStream_t stream,
            void *ext_buf = nullptr, size_t ext_bytes = 0) {
            int64_t sj = uts->stride[1], sk = uts->stride[2];
            GT355_CHECK(us->stride[1] == sj && us->stride[2] == sk && up->stride[1] == sj && up->stride[2] == sk &&
                            ut->stride[1] == sj && ut->stride[2] == sk,
                "gt355_vadv: utens_stage, u_stage, u_pos and utens must share one layout");
            // the reference keeps dtr_stage as a global_parameter of the storage type (vertical_advection_dycore.cpp:139)
            const CT dtr_c = CT(ST(dtr_stage));
            // the column sweep addresses fields through buffer descriptors with 32-bit byte offsets
            const int64_t span = std::max(((int64_t)(nk - 1) * sk + (int64_t)(nj - 1) * sj + ni) * (int64_t)sizeof(ST),
                ((int64_t)(nk - 1) * wc->stride[2] + (int64_t)(nj - 1) * wc->stride[1] + ni + 1) * (int64_t)sizeof(ST));
            const bool fits32 = span < (int64_t(1) << 32);
            int rc = GT355_OK;
            if (fits32 && nk <= 80) {
                // (a limit of the calls, not of this kernel, whose grid is one-dimensional: what it refuses stays refused)
                GT355_CHECK(nj <= 65535, "gt355_vadv: nj too large");
                if (launch_column<ST, CT>({uts, us, wc, up, ut, dtr_c, ni, nj, nk, stream, nullptr, 0, 0}, &rc))
                    return rc;
            }
            // ccol/dcol of levels 0..nk-2 for every column of a row
            const size_t row_bytes = sizeof(CT) * (size_t)ni * (size_t)(2 * nk - 1);
            GT355_CHECK(!ext_buf || row_bytes <= ext_bytes,
                "gt355_vadv_noalloc: ni = %d, nk = %d needs %zu bytes of ccol/dcol for one row of columns, more "
                "than the %zu-byte static scratch holds",
                ni, nk, row_bytes, ext_bytes);
            int rows = ext_buf ? (int)std::min<size_t>((size_t)nj, ext_bytes / row_bytes) : nj;
            GT355_CHECK((std::min(rows, nj) + 3) / 4 <= 65535, "gt355_vadv: nj too large");
            if (fits32 && nk > 80 &&
                launch_column<ST, CT>({uts, us, wc, up, ut, dtr_c, ni, nj, nk, stream, ext_buf, ext_bytes,
                                          row_bytes * (size_t)nj},
                    &rc))
                return rc;
            void *buf = ext_buf;
            if (!ext_buf) {
                size_t have = 0;
                if ((rc = scratch_for(stream, row_bytes * (size_t)nj, row_bytes * (size_t)nj, &buf, &have)))
                    return rc;
                // (less than every row's only while the stream is captured)
                rows = (int)std::min<size_t>((size_t)nj, have / row_bytes);
                if (rows < 1) {
                    set_error("gt355_vadv: a row of ni = %d, nk = %d needs %zu bytes of scratch, and the captured stream's "
                              "buffer has %zu; run the call once outside capture first",
                        ni, nk, row_bytes, have);
                    return GT355_EUNSUP;
                }
            }
            for (int j0 = 0; j0 < nj; j0 += rows) {
                const int nr = std::min(rows, nj - j0);
                dim3 grid((ni + 63) / 64, (nr + 3) / 4);
                vadv_scratch_kernel<ST, CT><<<grid, 256, 0, stream>>>((ST *)uts->origin + j0 * sj,
                    (const ST *)us->origin + j0 * sj, (const ST *)wc->origin + j0 * wc->stride[1],
                    (const ST *)up->origin + j0 * sj, (const ST *)ut->origin + j0 * sj, dtr_c, ni, nr, nk, sj, sk,
                    wc->stride[1], wc->stride[2], (CT *)buf, (int64_t)ni * nr);
                if ((rc = check_launch("gt355_vadv")))
                    return rc;
            }
            return GT355_OK;
        }
    } // namespace
} // namespace gt355
