// The vertical advection of one wavefront's 64 columns (one per lane) at any depth: ccol/dcol of the topmost 8 levels
// and of the first R below them in registers, of the next TL levels in LDS, of the levels beyond in the wavefront's
// scratch.
//
// What bounds it: a column's forward sweep needs five reads per level and its backward sweep ccol, dcol and u_pos of
// every level again, in reverse.  One wavefront per SIMD owns 512 registers and a quarter of the CU's LDS (40 KiB),
// which together hold ccol/dcol of R + 8 + TL levels; u_pos of those levels fits beside them only in part, so:
//   PARK: u_pos is parked in LDS during the forward sweep;
//   otherwise the backward sweep re-reads u_pos (default cache policy: the Infinity Cache holds what the forward
//   sweep read), NB levels ahead.
// A wavefront alone on its SIMD issues one instruction at a time, so below the memory's rate the time is its
// instruction count: ~51 per forward level (mixed form) and ~9 per backward level, next to 67 and 17 of a sweep that
// evaluates every functor operation and clamps and selects at every level.  Hence:
//   * levels run in blocks of BLK, unrolled, the block that holds the top level last, with the top's selects and clamps;
//     no level past it is ever run and no other block selects or clamps.  Where the depth may end in several blocks
//     (EXIT), each of those can be left for the one copy of the top block: the rings of all exits meet there, which
//     costs register moves and a wait for what is in flight.  Depths that fit the registers therefore have an
//     instantiation per block count instead, without exits;
//   * what a level shares with the one below it is taken from there (see `step`);
//   * level offsets are carried along, one addition per layout and level.
// Loads stay D levels ahead in register rings with static slots (level L in slot L % D).  A block is only entered from
// the one before it, so the wait before a slot covers that slot's own loads and no younger ones.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "common.hpp"
#include "functors.hpp"

namespace gt355 {

    // The fields as buffer descriptors (origins at grid point (0,0,0)) and their level strides in bytes.
    struct column_src {
        rsrc_t uts, us, wc, up, ut;
        uint32_t skb, wskb;
        int nk;
    };

    // f(integral_constant 0..N-1) until one returns false: an unrolled loop whose index is a constant from the start,
    // so that arrays indexed with it go to registers
    template <class F, int... I>
    __device__ __forceinline__ bool each_until(F &&f, std::integer_sequence<int, I...>) {
        return (f(std::integral_constant<int, I>()) && ...);
    }
    template <int N, class F>
    __device__ __forceinline__ bool each_until(F &&f) {
        return each_until(f, std::make_integer_sequence<int, N>());
    }

    // The levels below the top block are R in registers, then TL in LDS, then scratch.  MINK: the smallest depth; one that
    // ends in the block after the R + TL levels, R + TL < nk <= R + TL + 8, is the only one unless DEEP.  CPOL_W: the cache
    // policy of wcon, whose column-64 line a strip shares with its neighbour: the default policy keeps it in L2 for a
    // neighbour that runs later, the non-temporal one leaves the Infinity Cache to other fields.
    template <class ST, class CT, int R, int D, int TL, int NB, bool PARK, bool DEEP, int MINK = R + TL + 1,
        int CPOL_W = 0>
    struct column_sweep {
        static constexpr int BLK = 8;
        static constexpr bool EXIT = MINK <= R + TL;
        static_assert(R % BLK == 0 && TL % BLK == 0 && NB % BLK == 0 && NB <= R && (BLK % D == 0 || !(EXIT || DEEP)),
            "whole blocks; ring slots that every exit agrees on");
        static_assert(PARK || (NB & (NB - 1)) == 0, "the u_pos ring's slots are level mod NB");
        static constexpr int CPOL_UP = PARK ? CPOL_NT : 0;
        // per-lane rings of the forward sweep, level L in slot L % D: u_stage and wcon at i and i+1 (consumed at step
        // L-1), utens_stage, u_pos and utens (consumed at step L); us0: u_stage of level 0
        ST a_us[D], a_wi[D], a_wip[D], b_uts[D], b_up[D], b_ut[D], us0;

        static __device__ __forceinline__ uint32_t lvl(const column_src &f, int L) {
            return (uint32_t)min(L, f.nk - 1);
        }
        // opaque strides and depth: a step's loads, its level's offset and the depth tests exist from that step on
        // (otherwise the compiler hoists all of them, out of the loop over strips too, and spills)
        static __device__ __forceinline__ void pin(column_src &f) {
            asm volatile("" : "+s"(f.skb));
            asm volatile("" : "+s"(f.wskb));
            asm volatile("" : "+s"(f.nk));
        }
        __device__ __forceinline__ void load_a(
            const column_src &f, int s, uint32_t cb, uint32_t wb, uint32_t o, uint32_t ow) {
            a_us[s] = bload<ST, CPOL_NT>(f.us, cb, o);
            const two<ST> w = bload2<ST, CPOL_W>(f.wc, wb, ow);
            a_wi[s] = w.a;
            a_wip[s] = w.b;
        }
        __device__ __forceinline__ void load_b(const column_src &f, int s, uint32_t cb, uint32_t o) {
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
                load_b(f, L, cb, lvl(f, L) * f.skb);
                load_a(f, (L + 1) % D, cb, wb, lvl(f, L + 1) * f.skb, lvl(f, L + 1) * f.wskb);
            }
        }

        // The sweep of one column per lane, after its prologue.  s_up: (R + TL) x 64 parked u_pos (PARK); s_tail: TL x 2
        // x 64 ccol/dcol; sc: the wavefront's scratch, 2 x 64 values per level past R + TL below the top block.  next() is
        // called once, at the NB lowest levels of the backward sweep, when no load of this column is left to issue: it
        // may start the next column's prologue, in flight during those levels.
        template <class NEXT>
        __device__ __forceinline__ void sweep(column_src &f, CT dtr, uint32_t cb, uint32_t wb, ST (*s_up)[64],
            CT *s_tail, rsrc_t sc, NEXT &&next) {
            using std::false_type;
            using std::true_type;
            const int lane = threadIdx.x & 63;
            CT c[R], d[R];
            CT us_c = CT(us0), cm = CT(0), dm = CT(0), g_m = CT(0), t_m = CT(0);
            // byte offsets of the level loaded last into the a ring, clamped to the top (the b ring: the level below)
            uint32_t oa = lvl(f, D) * f.skb, ow = lvl(f, D) * f.wskb;
            const uint32_t oa_top = (uint32_t)(f.nk - 1) * f.skb, ow_top = (uint32_t)(f.nk - 1) * f.wskb;
            // Forward step of level k, slots s = k % D and s1 = (k + 1) % D, refilled with levels k + D and k + 1 + D
            // where ld_b / ld_a ask for it.  TOP: the block that holds the top level; first: level 0 (run-time there).
            // The functors' operations (forward_first / forward_body), with what level k shares with level k-1 taken
            // from there.  Level k's gav is minus level k-1's gcv, so a = as = -g_m with g = gcv * BET_P, and
            // -as (us_m - us_c) = g_m (us_m - us_c) = -t_m with t = cs (us_p - us_c): negation commutes with rounding,
            // and where us_m == us_c the two zeros differ in sign only, which no output sees (a sum with a nonzero term
            // or with +0 drops it; where the whole right-hand side is -0, u_pos is -0 too and data - u_pos is +0).
            // Level 0 takes the same form with zero g_m, t_m, cm and dm: x + 0 and x - 0 keep every nonzero x.
            auto step = [&](auto top_c, int k, int s, int s1, bool ld_b, bool ld_a) {
                constexpr bool TOP = decltype(top_c)::value;
                // (with exits, the top block and the next register block start alike: without values of its own the
                // compiler would evaluate what they share, and wait for it, before the branch between them)
                if constexpr (TOP && EXIT)
                    asm volatile(""
                                 : "+v"(b_uts[s]), "+v"(b_up[s]), "+v"(b_ut[s]), "+v"(a_us[s1]), "+v"(a_wi[s1]),
                                 "+v"(a_wip[s1]));
                const CT v_uts = CT(b_uts[s]), v_up = CT(b_up[s]), v_ut = CT(b_ut[s]);
                const CT us_p = CT(a_us[s1]), w_i = CT(a_wi[s1]), w_ip = CT(a_wip[s1]);
                pin(f);
                if (ld_b)
                    load_b(f, s, cb, oa);
                if (ld_a) {
                    // (oa + skb may wrap past 4 GiB only above the top, where any level's values do)
                    oa = min(oa + f.skb, oa_top);
                    ow = min(ow + f.wskb, ow_top);
                    load_a(f, s1, cb, wb, oa, ow);
                }
                // top level: zero k+1 winds and no k+1 correction term reproduce last_level exactly (forward_body)
                const bool at_top = TOP && k == f.nk - 1;
                const CT w_sum = at_top ? CT(0) : w_ip + w_i;
                const CT g = (CT(.25) * w_sum) * CT(BET_P);
                const CT t = g * (us_p - us_c);
                const CT b = (dtr + g_m) - g;
                const CT corr = -t_m - (at_top ? CT(0) : t);
                const CT rhs = ((dtr * v_up + v_ut) + v_uts) + corr;
                const CT divided = CT(1) / (b + cm * g_m);
                cm = g * divided;
                dm = (rhs + dm * g_m) * divided;
                asm volatile("" : "+v"(cm), "+v"(dm)); // keeps the chain at its step (no sinking)
                g_m = g;
                t_m = t;
                us_c = us_p;
            };
            const uint32_t lb = (uint32_t)(lane * sizeof(CT));
            constexpr uint32_t ROW = 64 * sizeof(CT);
            // the blocks on chip below the one that holds the top level; kb: the first level of that one
            int kb = EXIT ? 0 : R + TL;
            const bool past = each_until<(R + TL) / BLK>([&](auto n) {
                constexpr int k0 = decltype(n)::value * BLK;
                if constexpr (k0 + BLK >= MINK) {
                    pin(f);
                    if (k0 + BLK >= f.nk)
                        return false;
                }
#pragma clang loop unroll(full)
                for (int s = 0; s < BLK; ++s) {
                    const int k = k0 + s;
                    if constexpr (PARK)
                        s_up[k][lane] = b_up[k % D];
                    // (without exits the loads past the top block are left out)
                    step(false_type(), k, k % D, (k + 1) % D, EXIT || DEEP || k + D < R + TL + BLK,
                        EXIT || DEEP || k + 1 + D < R + TL + BLK);
                    if constexpr (k0 < R) {
                        c[k0 + s] = cm;
                        d[k0 + s] = dm;
                    } else {
                        s_tail[(k0 - R + s) * 128 + lane] = cm;
                        s_tail[(k0 - R + s) * 128 + 64 + lane] = dm;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (EXIT)
                    kb = k0 + BLK;
                return true;
            });
            if constexpr (DEEP) {
                if (past) {
                    for (; kb + BLK < f.nk; kb += BLK) { // the levels in scratch
#pragma clang loop unroll(full)
                        for (int s = 0; s < BLK; ++s) {
                            step(false_type(), kb + s, s % D, (s + 1) % D, true, true);
                            const uint32_t o = (uint32_t)(kb - R - TL + s) * 2 * ROW;
                            bstore<CT>(sc, cm, lb, o);
                            bstore<CT>(sc, dm, lb, o + ROW);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
            // the block of the top level: levels kb..kb+7, the top among them
            CT ct[BLK], dt[BLK], upt[BLK];
#pragma clang loop unroll(full)
            for (int s = 0; s < BLK; ++s) {
                if constexpr (EXIT)
                    asm volatile("" : "+v"(b_up[s % D]));
                constexpr int T0 = EXIT || DEEP ? 0 : R + TL; // the block's first level, as far as slots go
                upt[s] = CT(b_up[(T0 + s) % D]);
                step(true_type(), kb + s, (T0 + s) % D, (T0 + s + 1) % D, s + D < BLK, s + 1 + D < BLK);
                ct[s] = cm;
                dt[s] = dm;
                __builtin_amdgcn_sched_barrier(0);
            }

            // Backward sweep (vertical_advection_dycore.cpp:110-121), top level first: the recurrence of a block's
            // levels, then its outputs.
            // u_pos of the levels on chip, NB levels ahead (level L in slot L % NB): first the NB levels below kb, or below
            // the scratch levels
            ST r_up[PARK ? 1 : NB];
            if constexpr (!PARK) {
                pin(f);
                const int base = min(kb, R + TL) - NB;
#pragma clang loop unroll(full)
                for (int q = 0; q < NB; ++q)
                    r_up[q] = bload<ST, CPOL_UP>(f.up, cb, (uint32_t)max(base + ((q - base) & (NB - 1)), 0) * f.skb);
            }
            CT data = CT(0);
            {
                CT x[BLK];
#pragma clang loop unroll(full)
                for (int s = BLK - 1; s >= 0; --s) {
                    const CT v = dt[s] - ct[s] * data;
                    data = kb + s == f.nk - 1 ? dt[s] : v;
                    x[s] = data;
                }
                pin(f);
#pragma clang loop unroll(full)
                for (int s = BLK - 1; s >= 0; --s)
                    // a level above the top writes to the top a value that the top's own store, later in program order,
                    // replaces
                    bstore<ST, CPOL_OUT>(f.uts, ST(dtr * (x[s] - upt[s])), cb, lvl(f, kb + s) * f.skb);
                __builtin_amdgcn_sched_barrier(0);
            }
            uint32_t so = (uint32_t)(kb - 1) * f.skb; // byte offset of the level stored next
            if constexpr (DEEP) {
                if (kb > R + TL) {
                    // the blocks in scratch; rings one block deep
                    ST rp[BLK];
                    CT rc[BLK], rd[BLK];
                    auto fetch = [&](int k, int s) {
                        const uint32_t o = (uint32_t)(k - R - TL) * 2 * ROW;
                        rp[s] = bload<ST, CPOL_UP>(f.up, cb, (uint32_t)k * f.skb);
                        rc[s] = bload<CT>(sc, lb, o);
                        rd[s] = bload<CT>(sc, lb, o + ROW);
                    };
                    auto back_block = [&](auto more_c) {
#pragma clang loop unroll(full)
                        for (int s = BLK - 1; s >= 0; --s) {
                            data = rd[s] - rc[s] * data;
                            pin(f);
                            bstore<ST, CPOL_OUT>(f.uts, ST(dtr * (data - CT(rp[s]))), cb, so);
                            so -= f.skb;
                            if constexpr (decltype(more_c)::value)
                                fetch(kb + s - BLK, s);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    };
                    kb -= BLK;
#pragma clang loop unroll(full)
                    for (int s = 0; s < BLK; ++s)
                        fetch(kb + s, s);
                    for (; kb > R + TL; kb -= BLK)
                        back_block(true_type());
                    back_block(false_type());
                }
            }
            // the blocks on chip below kb
            each_until<(R + TL) / BLK>([&](auto n) {
                constexpr int k0 = R + TL - BLK - decltype(n)::value * BLK;
                if constexpr (k0 == NB - BLK)
                    next();
                pin(f);
                if (k0 + BLK < MINK || k0 < kb) {
                    ST v_up[BLK];
                    CT x[BLK], cc[BLK], dd[BLK];
#pragma clang loop unroll(full)
                    for (int s = BLK - 1; s >= 0; --s) {
                        if constexpr (k0 < R) {
                            cc[s] = c[k0 + s];
                            dd[s] = d[k0 + s];
                        } else {
                            cc[s] = s_tail[(k0 - R + s) * 128 + lane];
                            dd[s] = s_tail[(k0 - R + s) * 128 + 64 + lane];
                        }
                        if constexpr (PARK) {
                            v_up[s] = s_up[k0 + s][lane];
                        } else {
                            v_up[s] = r_up[(k0 + s) % NB];
                            if (k0 + s - NB >= 0)
                                r_up[(k0 + s) % NB] =
                                    bload<ST, CPOL_UP>(f.up, cb, (uint32_t)(k0 + s - NB) * f.skb);
                        }
                    }
#pragma clang loop unroll(full)
                    for (int s = BLK - 1; s >= 0; --s) {
                        data = dd[s] - cc[s] * data;
                        x[s] = data;
                    }
                    pin(f);
#pragma clang loop unroll(full)
                    for (int s = BLK - 1; s >= 0; --s) {
                        bstore<ST, CPOL_OUT>(f.uts, ST(dtr * (x[s] - CT(v_up[s]))), cb, so);
                        so -= f.skb;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                return true;
            });
        }
    };

} // namespace gt355
