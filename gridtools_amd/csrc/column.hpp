// The vertical advection of one wavefront's 64 columns (one per lane) at any depth: ccol/dcol of the first R levels
// in registers, of the next TL levels in LDS, of the levels beyond in the wavefront's scratch.
//
// What bounds it: a column's forward sweep needs five reads per level and its backward sweep ccol, dcol and u_pos of
// every level again, in reverse.  One wavefront per SIMD owns 512 registers and a quarter of the CU's LDS (40 KiB),
// which together hold ccol/dcol of R + TL levels; u_pos of those levels fits beside them only in part, so:
//   PARK: u_pos of the register levels is parked in LDS during the forward sweep (FP32 storage, TL = 16);
//   otherwise the backward sweep re-reads u_pos (default cache policy: the Infinity Cache holds what the forward
//   sweep read), NB levels ahead.
// The sweep keeps every load unconditional with its level clamped to the top, as vadv_onchip_kernel does, so the
// load counter stays exact; formulas at the top level are chosen by value.  Loops over register levels are unrolled
// (their ccol/dcol need static registers), loops over the tail run in blocks of D levels with static ring slots.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "functors.hpp"

namespace gt355 {

    // The fields as buffer descriptors (origins at grid point (0,0,0)) and their level strides in bytes.
    struct column_src {
        rsrc_t uts, us, wc, up, ut;
        uint32_t skb, wskb;
        int nk;
    };

    template <class ST, class CT, int R, int D, int TL, int NB, bool PARK>
    struct column_sweep {
        static_assert(R % D == 0 && TL % D == 0 && NB <= R, "tail blocks start on a ring slot");
        static constexpr int CPOL_UP = PARK ? CPOL_NT : 0;
        // per-lane rings of the forward sweep, level L in slot L % D: u_stage and wcon at i and i+1 (consumed at step
        // L-1), utens_stage, u_pos and utens (consumed at step L); us0: u_stage of level 0
        ST a_us[D], a_wi[D], a_wip[D], b_uts[D], b_up[D], b_ut[D], us0;

        static __device__ __forceinline__ uint32_t lvl(const column_src &f, int L) {
            return (uint32_t)min(L, f.nk - 1);
        }
        // opaque strides and depth: a step's loads, its level's clamped offset and its top-level test exist from that
        // step on (otherwise the compiler hoists all of them, out of the loop over strips too, and spills)
        static __device__ __forceinline__ void pin(column_src &f) {
            asm volatile("" : "+s"(f.skb));
            asm volatile("" : "+s"(f.wskb));
            asm volatile("" : "+s"(f.nk));
        }
        __device__ __forceinline__ void load_a(const column_src &f, int L, int s, uint32_t cb, uint32_t wb) {
            a_us[s] = bload<ST, CPOL_NT>(f.us, cb, lvl(f, L) * f.skb);
            // default policy: the neighbouring strip reads the column-64 line of this one from L2
            const two<ST> w = bload2<ST>(f.wc, wb, lvl(f, L) * f.wskb);
            a_wi[s] = w.a;
            a_wip[s] = w.b;
        }
        __device__ __forceinline__ void load_b(const column_src &f, int L, int s, uint32_t cb) {
            const uint32_t o = lvl(f, L) * f.skb;
            b_uts[s] = bload<ST, CPOL_NT>(f.uts, cb, o);
            b_up[s] = bload<ST, CPOL_UP>(f.up, cb, o);
            b_ut[s] = bload<ST, CPOL_NT>(f.ut, cb, o);
        }
        // the first D levels of the column at byte offsets cb (wcon: wb)
        __device__ __forceinline__ void prologue(column_src &f, uint32_t cb, uint32_t wb) {
            pin(f);
            us0 = bload<ST, CPOL_NT>(f.us, cb, 0);
#pragma clang loop unroll(full)
            for (int L = 0; L < D; ++L) {
                load_b(f, L, L, cb);
                load_a(f, L + 1, (L + 1) % D, cb, wb);
            }
        }

        // The sweep of one column per lane, after its prologue.  s_up: R x 64 parked u_pos (PARK); s_tail: TL x 2 x 64
        // ccol/dcol; sc: the wavefront's scratch, 2 x 64 values per level past R + TL.  next() is called once, NB
        // levels before the end of the backward sweep, when no load of this column is left to issue: it may start
        // the next column's prologue, in flight during the last NB steps.
        template <class NEXT>
        __device__ __forceinline__ void sweep(column_src &f, CT dtr, uint32_t cb, uint32_t wb, ST (*s_up)[64],
            CT *s_tail, rsrc_t sc, NEXT &&next) {
            const int lane = threadIdx.x & 63;
            const int nk = f.nk;
            CT c[R], d[R];
            CT us_m = CT(0), us_c = CT(us0), w_c_i = CT(0), w_c_ip = CT(0), cm = CT(0), dm = CT(0);
            // forward step of level k: slots s = k % D and s1 = (k + 1) % D, refilled with levels k + D and k + 1 + D
            auto step = [&](int k, int s, int s1, bool first) {
                const CT v_uts = CT(b_uts[s]), v_up = CT(b_up[s]), v_ut = CT(b_ut[s]);
                // top level: the k+1 wind taken as zero reproduces last_level exactly (see vadv_onchip_kernel)
                const bool at_top = k == f.nk - 1;
                const CT us_p = at_top ? us_c : CT(a_us[s1]);
                const CT w_p_i = at_top ? CT(0) : CT(a_wi[s1]);
                const CT w_p_ip = at_top ? CT(0) : CT(a_wip[s1]);
                pin(f);
                load_b(f, k + D, s, cb);
                load_a(f, k + 1 + D, s1, cb, wb);
                fwd_out<CT> r =
                    first ? forward_first<CT>(dtr, w_p_i, w_p_ip, us_c, us_p, v_up, v_ut, v_uts)
                          : forward_body<CT>(dtr, w_c_i, w_c_ip, w_p_i, w_p_ip, us_m, us_c, us_p, v_up, v_ut, v_uts,
                                cm, dm, at_top);
                asm volatile("" : "+v"(r.c), "+v"(r.d)); // keeps the chain at its step (no sinking)
                cm = r.c;
                dm = r.d;
                us_m = us_c;
                us_c = us_p;
                w_c_i = w_p_i;
                w_c_ip = w_p_ip;
            };
#pragma clang loop unroll(full)
            for (int k = 0; k < R; ++k) {
                if constexpr (PARK)
                    s_up[k][lane] = b_up[k % D];
                step(k, k % D, (k + 1) % D, k == 0);
                c[k] = cm;
                d[k] = dm;
                __builtin_amdgcn_sched_barrier(0);
            }
            const uint32_t lb = (uint32_t)(lane * sizeof(CT));
            constexpr uint32_t ROW = 64 * sizeof(CT);
            const int lds_end = min(nk, R + TL);
            if constexpr (TL > 0) {
                for (int kb = R; kb < lds_end; kb += D) {
#pragma clang loop unroll(full)
                    for (int s = 0; s < D; ++s) {
                        step(kb + s, s, (s + 1) % D, false);
                        CT *t = s_tail + (kb - R + s) * 128 + lane;
                        t[0] = cm;
                        t[64] = dm;
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            for (int kb = R + TL; kb < nk; kb += D) {
#pragma clang loop unroll(full)
                for (int s = 0; s < D; ++s) {
                    step(kb + s, s, (s + 1) % D, false);
                    const uint32_t o = (uint32_t)(kb - R - TL + s) * 2 * ROW;
                    bstore<CT>(sc, cm, lb, o);
                    bstore<CT>(sc, dm, lb, o + ROW);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }

            // backward sweep (vertical_advection_dycore.cpp:110-121), top level first
            CT data = CT(0);
            auto back = [&](int k, CT cc, CT dd, CT v_up) {
                const CT dt = dd - cc * data;
                const CT nd = k == f.nk - 1 ? dd : dt;
                data = nd;
                // a step above the top writes a value that the top's own step overwrites later in program order
                bstore<ST, CPOL_OUT>(f.uts, ST(dtr * (nd - v_up)), cb, lvl(f, k) * f.skb);
            };
            ST r_up[NB]; // u_pos of the register levels, NB levels ahead (level L in slot L % NB)
            if constexpr (!PARK) {
                pin(f);
#pragma clang loop unroll(full)
                for (int s = 0; s < NB; ++s)
                    r_up[(R - 1 - s) % NB] = bload<ST, CPOL_UP>(f.up, cb, lvl(f, R - 1 - s) * f.skb);
            }
            if (nk > R) {
                // the tail, in blocks of D levels; rings one block deep: u_pos, and ccol/dcol from scratch or LDS
                const int last = R + (nk - 1 - R) / D * D;
                ST rp[D];
                CT rc[D], rd[D];
#pragma clang loop unroll(full)
                for (int s = 0; s < D; ++s)
                    rp[s] = bload<ST, CPOL_UP>(f.up, cb, lvl(f, last + s) * f.skb);
                int kb = last;
                if (kb >= R + TL) {
                    auto fetch = [&](int k, int s) {
                        const uint32_t o = (uint32_t)max(k - R - TL, 0) * 2 * ROW;
                        rc[s] = bload<CT>(sc, lb, o);
                        rd[s] = bload<CT>(sc, lb, o + ROW);
                    };
#pragma clang loop unroll(full)
                    for (int s = 0; s < D; ++s)
                        fetch(kb + s, s);
                    for (; kb >= R + TL; kb -= D) {
#pragma clang loop unroll(full)
                        for (int s = D - 1; s >= 0; --s) {
                            back(kb + s, rc[s], rd[s], CT(rp[s]));
                            pin(f);
                            rp[s] = bload<ST, CPOL_UP>(f.up, cb, lvl(f, kb + s - D) * f.skb);
                            fetch(kb + s - D, s);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
                if constexpr (TL > 0) {
                    auto fetch = [&](int k, int s) {
                        const CT *t = s_tail + max(k - R, 0) * 128 + lane;
                        rc[s] = t[0];
                        rd[s] = t[64];
                    };
#pragma clang loop unroll(full)
                    for (int s = 0; s < D; ++s)
                        fetch(kb + s, s);
                    for (; kb >= R; kb -= D) {
#pragma clang loop unroll(full)
                        for (int s = D - 1; s >= 0; --s) {
                            back(kb + s, rc[s], rd[s], CT(rp[s]));
                            pin(f);
                            rp[s] = bload<ST, CPOL_UP>(f.up, cb, lvl(f, kb + s - D) * f.skb);
                            fetch(kb + s - D, s);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
            constexpr int UA = 4; // parked u_pos read ahead of its use
            ST l_up[UA];
            if constexpr (PARK) {
#pragma clang loop unroll(full)
                for (int s = 0; s < UA; ++s)
                    l_up[(R - 1 - s) % UA] = s_up[R - 1 - s][lane];
            }
#pragma clang loop unroll(full)
            for (int k = R - 1; k >= 0; --k) {
                if (k == NB - 1)
                    next();
                CT v_up;
                if constexpr (PARK) {
                    v_up = CT(l_up[k % UA]);
                    pin(f);
                    if (k - UA >= 0)
                        l_up[k % UA] = s_up[k - UA][lane];
                } else {
                    v_up = CT(r_up[k % NB]);
                    pin(f);
                    if (k - NB >= 0)
                        r_up[k % NB] = bload<ST, CPOL_UP>(f.up, cb, lvl(f, k - NB) * f.skb);
                }
                back(k, c[k], d[k], v_up);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

} // namespace gt355
