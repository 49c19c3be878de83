// The hdiff register sweep of one wavefront (horizontal_diffusion.cpp:35-107): used by the single-domain hdiff
// kernel (hdiff.hip) and by the batching form's stencil phase (batch.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "functors.hpp"

namespace gt355 {
    // Register sweep: no LDS, no barriers.
    //
    // One wavefront owns 64 consecutive columns [i0, i0+64) of one k-level and sweeps JB output rows in j.
    // Rows of in live in registers (a three-row window), the i-neighbours of in and lap come from DPP
    // wavefront shifts, and the two lanes at the wave edges take their out-of-wave neighbour from a "side"
    // column the wave streams with scalar loads (columns i0-1 / i0+64, plus i0-2 / i0+65 for the side
    // laplacian): the DPP bound control keeps the destination's old value for a source lane outside
    // the wave, and that old value is exactly the side column.  Loads run P rows ahead through register
    // rings; all loads are unconditional (clamped to the valid box) so the load counter stays exact.
    // The wavefront's strip is columns [i0, i0+64) x rows [j0, j0+JB) of level k (i0, j0, k wave-uniform).  LAP also
    // stores the laplacian of every output point (the lap ij-cache value there) into `lap`, laid out like `out`.
    // PO / PI: the output and input pointer types (ST * and const ST * from kernel arguments; global-address-space
    // pointers when they come from a table in memory, so that accesses are global_* rather than flat_*).
    template <class ST, class CT, int JB, int P, bool LAP, class PO = ST *, class PI = const ST *>
    __device__ __forceinline__ void hdiff_sweep_wave(PO __restrict__ out, PI __restrict__ in, PI __restrict__ coeff,
        PO __restrict__ lap, int ni, int nj, int64_t osj, int64_t osk, int64_t isj, int64_t isk, int64_t csj,
        int64_t csk, int i0, int j0, int k) {
        constexpr int NR = JB + 4; // in rows j0-2 .. j0+JB+1
        const int lane = threadIdx.x & 63;
        const bool left = lane < 32;
        // columns, clamped to the readable box [-2, ni+2): own column per lane, side columns per wave
        const int ic = min(i0 + lane, ni + 1);
        const int ieL = i0 - 1, ifL = i0 - 2;
        const int ieR = min(i0 + 64, ni + 1), ifR = min(i0 + 65, ni + 1);
        const PI inp = in + (int64_t)k * isk;
        const PI cop = coeff + (int64_t)k * csk;
        auto row = [&](int t) { return (int64_t)min(j0 - 2 + t, nj + 1); }; // absolute row of ring step t

        ST rc[P], rk[P];                 // per-lane rings: own column, coeff
        ST reL[P], rfL[P], reR[P], rfR[P]; // wave-uniform rings: side columns (scalar loads)
        auto load = [&](int t) {
            const int64_t r = row(t);
            // in rows are re-read by the neighbouring strips (rim rows) and side columns: default cache policy
            rc[t % P] = inp[r * isj + ic];
            reL[t % P] = inp[r * isj + ieL];
            rfL[t % P] = inp[r * isj + ifL];
            reR[t % P] = inp[r * isj + ieR];
            rfR[t % P] = inp[r * isj + ifR];
            // coeff of the row that is output at ring step t, R-2 = j0-4+t (clamped into the interior; only
            // steps 4..NR-1 use it)
            const int64_t ro = min(max(j0 - 4 + t, 0), nj - 1);
            rk[t % P] = __builtin_nontemporal_load(cop + ro * csj + min(ic, ni - 1)); // read once
        };
#pragma clang loop unroll(full)
        for (int t = 0; t < P; ++t)
            load(t);

        CT c0 = 0, c1 = 0, c2 = 0;       // in rows R-2, R-1, R of the own column
        CT eL0 = 0, eL1 = 0, eL2 = 0;    // the same rows of column i0-1 (uniform)
        CT eR0 = 0, eR1 = 0, eR2 = 0;    // the same rows of column i0+64 (uniform)
        CT fL1 = 0, fR1 = 0;             // columns i0-2 and i0+65 of row R-1 (uniform)
        CT m1 = 0, p1 = 0;               // in(i-1), in(i+1) of row R-1
        CT m0 = 0, p0 = 0;               // in(i-1), in(i+1) of row R-2
        CT lap1 = 0, lap0 = 0;           // lap of rows R-1 and R-2 (own column)
        CT sl1 = 0, sl0 = 0;             // side laplacian of rows R-1 and R-2 (i0-1 on lane 0, i0+64 on lane 63)
        CT fly_m = 0;                    // fly of row R-3
        // output rows through buffer descriptors based at the strip's first point (wave-uniform): the row offset is
        // a scalar, the lane's column a vector offset, and the stores take the output cache policy
        const int64_t o0 = (int64_t)k * osk + (int64_t)j0 * osj + i0;
        const rsrc_t r_o = make_rsrc(wave_uniform((const void *)(out + o0)));
        const rsrc_t r_l = make_rsrc(wave_uniform((const void *)(LAP ? lap + o0 : out + o0)));
        const uint32_t ob = (uint32_t)(lane * sizeof(ST));
        const bool col_ok = i0 + lane < ni;
#pragma clang loop unroll(full)
        for (int t = 0; t < NR; ++t) {
            // shift the windows and take row R = j0 - 2 + t from the rings
            c0 = c1; c1 = c2; c2 = CT(rc[t % P]);
            eL0 = eL1; eL1 = eL2; eL2 = CT(reL[t % P]);
            eR0 = eR1; eR1 = eR2; eR2 = CT(reR[t % P]);
            const CT kout = CT(rk[t % P]); // coeff of row R-2
            const CT fL_r = CT(rfL[t % P]), fR_r = CT(rfR[t % P]);
            if (t + P < NR)
                load(t + P);
            // in(i-1), in(i+1) of row R: lane 0 keeps column i0-1, lane 63 keeps column i0+64
            const CT m2 = dpp_keep<DPP_WF_SR1>(eL2, c2), p2 = dpp_keep<DPP_WF_SL1>(eR2, c2);
            lap0 = lap1;
            sl0 = sl1;
            if (t >= 2) {
                // lap of row R-1 (lap_function, horizontal_diffusion.cpp:41-46): needs rows R-2..R
                lap1 = lap_f<CT>(c1, p1, c2, m1, c0);
                // side laplacian at i0-1 (left lanes) or i0+64 (right lanes); the own column is the i+1
                // neighbour on the left side and the i-1 neighbour on the right side
                const CT e0 = left ? eL0 : eR0, e1 = left ? eL1 : eR1, e2 = left ? eL2 : eR2;
                const CT ip = left ? c1 : fR1, im = left ? fL1 : c1;
                sl1 = lap_f<CT>(e1, ip, e2, im, e0);
            }
            if (t >= 4) {
                // output row R-2: flx, flx[i-1], fly, fly[j-1], out (horizontal_diffusion.cpp:56-60, 70-74, 86-90)
                const CT lm = dpp_keep<DPP_WF_SR1>(sl0, lap0), lp = dpp_keep<DPP_WF_SL1>(sl0, lap0);
                const CT flx_c = flux_f<CT>(lp, lap0, p0, c0);
                const CT flx_m = flux_f<CT>(lap0, lm, c0, m0);
                const CT fly_c = flux_f<CT>(lap1, lap0, c1, c0);
                const CT res = c0 - kout * (((flx_c - flx_m) + fly_c) - fly_m);
                fly_m = fly_c;
                const int r_out = j0 + t - 4;
                if (col_ok && r_out < nj) {
                    const uint32_t rb = (uint32_t)((t - 4) * osj * (int64_t)sizeof(ST));
                    bstore<ST, CPOL_OUT>(r_o, static_cast<ST>(res), ob, rb);
                    if constexpr (LAP)
                        bstore<ST, CPOL_OUT>(r_l, static_cast<ST>(lap0), ob, rb);
                }
            } else if (t == 3) {
                // fly of row j0-1, the fly[j-1] of the first output row
                fly_m = flux_f<CT>(lap1, lap0, c1, c0);
            }
            // rows move down one: (R-1) -> R-2 for the next step's output, R -> R-1 for its laplacian
            m0 = m1;
            p0 = p1;
            m1 = m2;
            p1 = p2;
            fL1 = fL_r;
            fR1 = fR_r;
        }
    }

    // Column-pair register sweep: the register sweep above with two adjacent columns per lane, so one wavefront
    // covers 128 columns [i0, i0+128) and every row load is one 2-element vector per lane (8 bytes per lane for
    // FP32 storage: 512-byte wavefront requests, the size at which the FP64 sweep streams best; measured at
    // 256x256x80 FP32 storage: 14.2 us against 16.5 us for one column per lane).  Lane l owns columns
    // a = i0+2l and b = a+1: the i-neighbours inside a lane are the other column of the pair, across lanes they
    // come from DPP shifts (a's i-1 is the b column of lane l-1, b's i+1 the a column of lane l+1), and lanes
    // 0 / 63 keep the side columns i0-1 / i0+128 (and i0-2 / i0+129 for the side laplacian), streamed with
    // scalar loads.  flx at b-1 is flx at a, so each lane evaluates three x-fluxes, not four.  Lanes past the
    // domain load the last pair (clamped) and store nothing; since ni is even, the lane after the last valid
    // one loads exactly columns ni and ni+1, the right neighbours the last valid lane needs.  The launcher uses
    // it for even ni with 2-element-aligned rows (origin and j/k strides); other shapes take the flat sweep below (FP32
    // storage) or the one-column sweep (FP64).
    // The wavefront's strip is columns [i0, i0+128) x rows [j0, j0+JB) of level k (wave-uniform); LAP also stores the
    // laplacian of every output point into `lap`, laid out like `out`.  PO / PI as for hdiff_sweep_wave.
    template <class ST, class CT, int JB, int P, bool LAP, class PO = ST *, class PI = const ST *>
    __device__ __forceinline__ void hdiff_pair_wave(PO __restrict__ out, PI __restrict__ in, PI __restrict__ coeff,
        PO __restrict__ lap, int ni, int nj, int64_t osj, int64_t osk, int64_t isj, int64_t isk, int64_t csj,
        int64_t csk, int i0, int j0, int k) {
        typedef ST vec2 __attribute__((ext_vector_type(2)));
        // vector pointers in the address space of the field pointers
        using VCP = decltype((const vec2 *)(PI)nullptr);
        constexpr int NR = JB + 4; // in rows j0-2 .. j0+JB+1
        const int lane = threadIdx.x & 63;
        const bool left = lane < 32;
        const int ca = i0 + 2 * lane;
        // pair starts, clamped: in is readable on [-2, ni+2), coeff on [0, ni); ni is even
        const int pin_ = min(ca, ni), pco = min(ca, ni - 2);
        const int ieL = i0 - 1, ifL = i0 - 2;
        const int ieR = min(i0 + 128, ni + 1), ifR = min(i0 + 129, ni + 1);
        const PI inp = in + (int64_t)k * isk;
        const PI cop = coeff + (int64_t)k * csk;
        auto row = [&](int t) { return (int64_t)min(j0 - 2 + t, nj + 1); };

        vec2 rc[P], rk[P];
        ST reL[P], rfL[P], reR[P], rfR[P];
        auto load = [&](int t) {
            const int64_t r = row(t);
            rc[t % P] = *(VCP)(inp + r * isj + pin_);
            reL[t % P] = inp[r * isj + ieL];
            rfL[t % P] = inp[r * isj + ifL];
            reR[t % P] = inp[r * isj + ieR];
            rfR[t % P] = inp[r * isj + ifR];
            const int64_t ro = min(max(j0 - 4 + t, 0), nj - 1);
            rk[t % P] = __builtin_nontemporal_load((VCP)(cop + ro * csj + pco)); // read once
        };
#pragma clang loop unroll(full)
        for (int t = 0; t < P; ++t)
            load(t);

        CT a0 = 0, a1 = 0, a2 = 0, b0 = 0, b1 = 0, b2 = 0; // in rows R-2, R-1, R of columns a and b
        CT eL0 = 0, eL1 = 0, eL2 = 0, eR0 = 0, eR1 = 0, eR2 = 0;
        CT fL1 = 0, fR1 = 0;
        CT ma1 = 0, ma0 = 0; // in(a-1) of rows R-1, R-2
        CT pb1 = 0, pb0 = 0; // in(b+1) of rows R-1, R-2
        CT la1 = 0, la0 = 0, lb1 = 0, lb0 = 0; // lap of rows R-1, R-2 at a and b
        CT sl1 = 0, sl0 = 0;                  // side laplacian (i0-1 on lane 0, i0+128 on lane 63)
        CT flya_m = 0, flyb_m = 0;            // fly of row R-3
        const int64_t o0 = (int64_t)k * osk + (int64_t)j0 * osj + i0;
        const rsrc_t r_o = make_rsrc(wave_uniform((const void *)(out + o0)));
        const rsrc_t r_l = make_rsrc(wave_uniform((const void *)(LAP ? lap + o0 : out + o0)));
        const uint32_t ob = (uint32_t)(2 * lane * sizeof(ST));
        const bool col_ok = ca < ni; // ni even: b = a+1 is inside too
#pragma clang loop unroll(full)
        for (int t = 0; t < NR; ++t) {
            const vec2 v = rc[t % P];
            a0 = a1; a1 = a2; a2 = CT(v.x);
            b0 = b1; b1 = b2; b2 = CT(v.y);
            eL0 = eL1; eL1 = eL2; eL2 = CT(reL[t % P]);
            eR0 = eR1; eR1 = eR2; eR2 = CT(reR[t % P]);
            const vec2 kv = rk[t % P];
            const CT ka = CT(kv.x), kb = CT(kv.y);
            const CT fL_r = CT(rfL[t % P]), fR_r = CT(rfR[t % P]);
            if (t + P < NR)
                load(t + P);
            const CT ma2 = dpp_keep<DPP_WF_SR1>(eL2, b2), pb2 = dpp_keep<DPP_WF_SL1>(eR2, a2);
            la0 = la1;
            lb0 = lb1;
            sl0 = sl1;
            if (t >= 2) {
                // lap of row R-1 at a and b (lap_function, horizontal_diffusion.cpp:41-46)
                la1 = lap_f<CT>(a1, b1, a2, ma1, a0);
                lb1 = lap_f<CT>(b1, pb1, b2, a1, b0);
                const CT e0 = left ? eL0 : eR0, e1 = left ? eL1 : eR1, e2 = left ? eL2 : eR2;
                const CT ip = left ? a1 : fR1, im = left ? fL1 : b1;
                sl1 = lap_f<CT>(e1, ip, e2, im, e0);
            }
            if (t >= 4) {
                // output row R-2 (horizontal_diffusion.cpp:56-60, 70-74, 86-90)
                const CT lam = dpp_keep<DPP_WF_SR1>(sl0, lb0), lbp = dpp_keep<DPP_WF_SL1>(sl0, la0);
                const CT flx_a = flux_f<CT>(lb0, la0, b0, a0);
                const CT flx_am = flux_f<CT>(la0, lam, a0, ma0);
                const CT flx_b = flux_f<CT>(lbp, lb0, pb0, b0);
                const CT fly_a = flux_f<CT>(la1, la0, a1, a0);
                const CT fly_b = flux_f<CT>(lb1, lb0, b1, b0);
                const CT ra = a0 - ka * (((flx_a - flx_am) + fly_a) - flya_m);
                const CT rb = b0 - kb * (((flx_b - flx_a) + fly_b) - flyb_m);
                flya_m = fly_a;
                flyb_m = fly_b;
                const int r_out = j0 + t - 4;
                if (col_ok && r_out < nj) {
                    const uint32_t rbo = (uint32_t)((t - 4) * osj * (int64_t)sizeof(ST));
                    bstore_pair<ST, CPOL_OUT>(r_o, static_cast<ST>(ra), static_cast<ST>(rb), ob, rbo);
                    if constexpr (LAP)
                        bstore_pair<ST, CPOL_OUT>(r_l, static_cast<ST>(la0), static_cast<ST>(lb0), ob, rbo);
                }
            } else if (t == 3) {
                // fly of row j0-1, the fly[j-1] of the first output row
                flya_m = flux_f<CT>(la1, la0, a1, a0);
                flyb_m = flux_f<CT>(lb1, lb0, b1, b0);
            }
            ma0 = ma1;
            pb0 = pb1;
            ma1 = ma2;
            pb1 = pb2;
            fL1 = fL_r;
            fR1 = fR_r;
        }
    }

    // Flat column-pair sweep: two adjacent columns per lane and JB rows of one level, as hdiff_pair_wave, but with the
    // lanes taken from one list over every (level, row block, column pair) instead of from 128-column strips.
    //
    // The list of a row block is its pairs from column -2 to ni+1 (one rim pair on each side), padded to NP entries
    // (a multiple of 4, so that rows of outputs start on whole 32-byte sectors); row blocks follow each other, then
    // levels.  A wavefront takes 62 consecutive entries (lanes 62 and 63 repeat the pattern unused) and outputs those of
    // lanes 1..60, so consecutive wavefronts overlap by two rim entries.  A lane's neighbours i-1 and i+2 are always in
    // the next lanes (DPP shifts): there are no side columns, no scalar loads, no side laplacian and no selects between
    // sides, and a lane's flx at its left edge is the left lane's flx (a shift instead of a fourth flux).  Rows of any
    // width fill their lanes, and an odd ni or unaligned rows need no more than the last pair's handling below (a
    // request only needs element alignment).
    // What bounds it: ~28 vector instructions per point against ~78 of the one-column sweep (mixed form), so not those but
    // what is in flight: all JB + 4 rows (JB 4, 2 or 1) are loaded ahead, so a wavefront waits for memory once, and has
    // nothing in flight while it computes and stores; 7 wavefronts per SIMD cover for that in part (387x251x61 mixed 4.4
    // TB/s, like the aligned 256x256x80 on strips; about 5 us of it a launch's ramp and drain).  A wavefront's rows start
    // anywhere, five lines where an aligned 128-column strip has four: full strips stay with hdiff_pair_wave
    // (512x512x80 FP64 82 us against 85 here, 1536x1536x80 mixed 382 against 394) and ragged widths come here (mixed, us,
    // strips / flat: 387x251x61 19.6 / 16.2, 130x400x137 26.2 / 19.7, 101x203x60 8.3 / 5.9).
    // Rows: block b covers output rows b*JB.., moved up to end at nj (j0 = min(b*JB, nj - JB), nj >= JB); rows that the
    // block before owns are computed but not stored, so every row has one writer.  Addresses are buffer descriptors
    // plus a lane offset and one scalar offset per row (the launcher checks that every field spans less than 4 GiB).
    // Odd ni (ODD): the rim pair on the right starts at ni+1 and would read ni+2, so it is loaded one column to the
    // left and its a column taken from the second element; the last pair (ni-1, ni) loads coeff one column to the left
    // and stores its a column alone.
    constexpr int FLAT_OW = 60, FLAT_ALIGN = 4;
    struct hdiff_flat_args {
        int ni, nj, np, blocks;                // np: list entries per row block; blocks: row blocks per level
        uint32_t osj, osk, isj, isk, csj, csk; // strides in bytes
        int total;                             // list entries
    };
    // list entries per row block
    __host__ __device__ inline int flat_entries(int ni) { return ((ni + 1) / 2 + 2 + FLAT_ALIGN - 1) / FLAT_ALIGN * FLAT_ALIGN; }
    template <class ST, class CT, int JB, int P, bool LAP, bool ODD>
    __device__ __forceinline__ void hdiff_flat_wave(
        rsrc_t r_out, rsrc_t r_in, rsrc_t r_co, rsrc_t r_lap, const hdiff_flat_args &g, int w) {
        constexpr int NR = JB + 4; // in rows j0-2 .. j0+JB+1
        static_assert(P <= NR, "rows in flight");
        constexpr uint32_t S = sizeof(ST);
        const int lane = threadIdx.x & 63;
        // entry w*OW + lane as (level k, row block b, pair p): the wavefront's first entry by uniform divisions, a
        // lane's own by carrying over
        constexpr int OW = FLAT_OW;
        const int v0 = w * OW;
        const int q0 = v0 / g.np;
        int p = v0 - q0 * g.np + lane, k = q0 / g.blocks, b = q0 - k * g.blocks;
        while (__any(p >= g.np)) {
            if (p >= g.np) {
                p -= g.np;
                if (++b == g.blocks)
                    b = 0, ++k;
            }
        }
        // the wavefront's last lanes may lie past the list: they repeat its last entry, a rim pair
        const bool inside = v0 + lane < g.total;
        if (!inside) {
            p = g.np - 1;
            b = g.blocks - 1;
            k = (g.total / g.np) / g.blocks - 1;
        }
        const int pairs = (g.ni + 1) / 2;      // pairs with an output column
        const int a = 2 * (min(p, pairs + 1) - 1); // the lane's first column (padding entries repeat the rim pair)
        const int j0 = min(b * JB, g.nj - JB), skip = b * JB - j0;
        const bool odd_rim = ODD && a > g.ni;       // starts at ni + 1
        const bool odd_last = ODD && a == g.ni - 1; // its b column is ni
        const uint32_t vi = (uint32_t)k * g.isk + (uint32_t)j0 * g.isj + (uint32_t)(a + 2 - (odd_rim ? 1 : 0)) * S;
        // coeff and the outputs exist on [0, ni) only: rim lanes take the nearest pair and store nothing
        const int ac = min(max(a, 0), 2 * (pairs - 1));
        const uint32_t vc =
            (uint32_t)k * g.csk + (uint32_t)j0 * g.csj + (uint32_t)(ac - (ODD && ac == g.ni - 1 ? 1 : 0)) * S;
        const uint32_t vo = (uint32_t)k * g.osk + (uint32_t)j0 * g.osj + (uint32_t)ac * S;
        const bool own = inside && lane >= 1 && lane <= OW && p >= 1 && p <= pairs;

        two<ST> rc[P], rk[P];
        auto load = [&](int t) {
            rc[t % P] = bload2<ST>(r_in, vi, (uint32_t)t * g.isj); // rim rows are re-read: default cache policy
            if (t >= 4)
                rk[t % P] = bload2<ST, CPOL_NT>(r_co, vc, (uint32_t)(t - 4) * g.csj);
        };
#pragma clang loop unroll(full)
        for (int t = 0; t < P; ++t)
            load(t);

        // rows R-2, R-1, R: columns a and b, in(a-1) and in(b+1); laplacians and fly of the previous rows
        CT a0 = 0, a1 = 0, a2 = 0, b0 = 0, b1 = 0, b2 = 0, ma1 = 0, pb1 = 0, pb0 = 0;
        CT la1 = 0, la0 = 0, lb1 = 0, lb0 = 0, flya_m = 0, flyb_m = 0;
#pragma clang loop unroll(full)
        for (int t = 0; t < NR; ++t) {
            const two<ST> v = rc[t % P], kv = rk[t % P];
            const ST va = odd_rim ? v.b : v.a;
            if (t + P < NR)
                load(t + P);
            a0 = a1; a1 = a2; a2 = CT(va);
            b0 = b1; b1 = b2; b2 = CT(v.b);
            const CT ma2 = CT(dpp_any<DPP_WF_SR1>(v.b)), pb2 = CT(dpp_any<DPP_WF_SL1>(va));
            la0 = la1;
            lb0 = lb1;
            if (t >= 2) {
                // lap of row R-1 at a and b (lap_function, horizontal_diffusion.cpp:41-46)
                la1 = lap_f<CT>(a1, b1, a2, ma1, a0);
                lb1 = lap_f<CT>(b1, pb1, b2, a1, b0);
            }
            if (t >= 4) {
                // output row R-2 (horizontal_diffusion.cpp:56-60, 70-74, 86-90)
                const CT lbp = dpp_any<DPP_WF_SL1>(la0);
                const CT flx_a = flux_f<CT>(lb0, la0, b0, a0);
                const CT flx_b = flux_f<CT>(lbp, lb0, pb0, b0);
                const CT flx_am = dpp_any<DPP_WF_SR1>(flx_b);
                const CT fly_a = flux_f<CT>(la1, la0, a1, a0);
                const CT fly_b = flux_f<CT>(lb1, lb0, b1, b0);
                const CT ka = CT(ODD && odd_last ? kv.b : kv.a), kb = CT(kv.b);
                const CT ra = a0 - ka * (((flx_a - flx_am) + fly_a) - flya_m);
                const CT rb = b0 - kb * (((flx_b - flx_a) + fly_b) - flyb_m);
                flya_m = fly_a;
                flyb_m = fly_b;
                if (own && t - 4 >= skip) {
                    const uint32_t so = (uint32_t)(t - 4) * g.osj;
                    if (!ODD || !odd_last) {
                        bstore_pair<ST, CPOL_OUT>(r_out, ST(ra), ST(rb), vo, so);
                        if constexpr (LAP)
                            bstore_pair<ST, CPOL_OUT>(r_lap, ST(la0), ST(lb0), vo, so);
                    } else {
                        bstore<ST, CPOL_OUT>(r_out, ST(ra), vo, so);
                        if constexpr (LAP)
                            bstore<ST, CPOL_OUT>(r_lap, ST(la0), vo, so);
                    }
                }
            } else if (t == 3) {
                // fly of row j0-1, the fly[j-1] of the first output row
                flya_m = flux_f<CT>(la1, la0, a1, a0);
                flyb_m = flux_f<CT>(lb1, lb0, b1, b0);
            }
            ma1 = ma2;
            pb0 = pb1;
            pb1 = pb2;
        }
    }

} // namespace gt355
