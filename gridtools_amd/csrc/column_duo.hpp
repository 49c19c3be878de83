// The vertical advection of 64 columns (one per lane) by two wavefronts, for domains with fewer strips than SIMDs.
//
// What bounds such a domain: one wavefront alone on its SIMD issues an instruction every four cycles, ~60 per level,
// whatever the memory could do (column.hpp), and half of the SIMDs or more have none.  So the level's work is split
// over two SIMDs of a CU:
//   * the coefficient wavefront loads the fields and evaluates what does not depend on the level below (gcv, b and the
//     right-hand side), a block of BLK levels ahead; in the backward sweep it turns the solution into outputs, with
//     u_pos kept in its registers;
//   * the recurrence wavefront runs the chain: the division, ccol and dcol (in registers up to RREG levels, then LDS),
//     and the backward substitution.
// Blocks pass through LDS, double buffered, one barrier per block: a wavefront refills a buffer only after the
// barrier that follows the other's last read of it.  Same operations in the same order as column.hpp: the same bits.
// The block count is a template parameter: everything is unrolled, no level past the block of the top one is run.
// What bounds it now: the recurrence's chain of dependent operations, the division's among them (FP64 64x64: 6.6 us at
// 40 levels, 10.8 at 80, so ~105 ns per level against ~120 of one wavefront; 128x128x137 19.7 us against 26.4).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "column.hpp"
#include "common.hpp"
#include "functors.hpp"

namespace gt355 {

    template <class ST, class CT, int NBLK>
    struct column_duo {
        static constexpr int BLK = 8, N = NBLK * BLK, D = BLK;
        // levels of ccol/dcol in the recurrence wavefront's registers; those beyond in LDS
        static constexpr int RREG = sizeof(CT) == 8 ? (N < 104 ? N : 104) : N;
        struct shared {
            CT g[2][BLK][64], b[2][BLK][64], rhs[2][BLK][64]; // forward: a block's coefficients
            CT x[2][BLK][64];                                 // backward: a block's solution
            CT c[N - RREG > 0 ? N - RREG : 1][64], d[N - RREG > 0 ? N - RREG : 1][64];
        };

        // what was written to LDS before is visible to the other wavefront after; loads from memory stay in flight
        static __device__ __forceinline__ void meet() {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        }

        static __device__ __forceinline__ void coefficients(
            column_src f, CT dtr, uint32_t cb, uint32_t wb, shared &sh, int lane) {
            ST a_us[D], a_wi[D], a_wip[D], b_uts[D], b_ut[D], up[N];
            auto pin = [&]() {
                asm volatile("" : "+s"(f.skb));
                asm volatile("" : "+s"(f.wskb));
                asm volatile("" : "+s"(f.nk));
            };
            auto lvl = [&](int L) { return (uint32_t)min(L, f.nk - 1); };
            auto load_a = [&](int L) {
                a_us[L % D] = bload<ST, CPOL_NT>(f.us, cb, lvl(L) * f.skb);
                // default policy: the neighbouring strip reads the column-64 line of this one from L2
                const two<ST> w = bload2<ST>(f.wc, wb, lvl(L) * f.wskb);
                a_wi[L % D] = w.a;
                a_wip[L % D] = w.b;
            };
            pin();
            const ST us0 = bload<ST, CPOL_NT>(f.us, cb, 0);
            CT us_c = CT(0), g_m = CT(0), t_m = CT(0);
            // forward: block n from the rings, whose slots are refilled for block n + 1
            each_until<NBLK + 1>([&](auto nc) {
                constexpr int n = decltype(nc)::value - 1;
                if constexpr (n == 0)
                    us_c = CT(us0);
#pragma clang loop unroll(full)
                for (int s = 0; s < BLK; ++s) {
                    const int k = n * BLK + s, L = k + BLK; // the level evaluated, the level loaded
                    if constexpr (n >= 0) {
                        const bool at_top = n == NBLK - 1 && k == f.nk - 1;
                        const CT us_p = CT(a_us[(k + 1) % D]);
                        const CT w_sum = at_top ? CT(0) : CT(a_wip[(k + 1) % D]) + CT(a_wi[(k + 1) % D]);
                        const CT g = (CT(.25) * w_sum) * CT(BET_P);
                        const CT t = g * (us_p - us_c);
                        const CT corr = -t_m - (at_top ? CT(0) : t);
                        sh.g[n & 1][s][lane] = g;
                        sh.b[n & 1][s][lane] = (dtr + g_m) - g;
                        sh.rhs[n & 1][s][lane] = ((dtr * CT(up[k]) + CT(b_ut[s])) + CT(b_uts[s])) + corr;
                        g_m = g;
                        t_m = t;
                        us_c = us_p;
                    }
                    if constexpr (n + 1 < NBLK) {
                        pin();
                        b_uts[s] = bload<ST, CPOL_NT>(f.uts, cb, lvl(L) * f.skb);
                        up[L] = bload<ST, CPOL_NT>(f.up, cb, lvl(L) * f.skb);
                        b_ut[s] = bload<ST, CPOL_NT>(f.ut, cb, lvl(L) * f.skb);
                        load_a(L + 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (n >= 0)
                    meet();
                return true;
            });
            // backward: the outputs of a block, top block first (vertical_advection_dycore.cpp:110-121)
            each_until<NBLK>([&](auto nc) {
                constexpr int n = NBLK - 1 - decltype(nc)::value;
                meet();
                pin();
#pragma clang loop unroll(full)
                for (int s = BLK - 1; s >= 0; --s) {
                    const int k = n * BLK + s;
                    // a level above the top writes to the top a value that the top's own store, later in program order,
                    // replaces
                    bstore<ST, CPOL_OUT>(f.uts, ST(dtr * (sh.x[n & 1][s][lane] - CT(up[k]))), cb,
                        (n == NBLK - 1 ? lvl(k) : (uint32_t)k) * f.skb);
                }
                __builtin_amdgcn_sched_barrier(0);
                return true;
            });
        }

        static __device__ __forceinline__ void recurrence(int nk, CT dtr, shared &sh, int lane) {
            CT c[RREG], d[RREG], cm = CT(0), dm = CT(0), g_m = CT(0);
            each_until<NBLK>([&](auto nc) {
                constexpr int n = decltype(nc)::value;
                meet();
                CT g[BLK], b[BLK], rhs[BLK];
#pragma clang loop unroll(full)
                for (int s = 0; s < BLK; ++s) {
                    g[s] = sh.g[n & 1][s][lane];
                    b[s] = sh.b[n & 1][s][lane];
                    rhs[s] = sh.rhs[n & 1][s][lane];
                }
#pragma clang loop unroll(full)
                for (int s = 0; s < BLK; ++s) {
                    const CT divided = CT(1) / (b[s] + cm * g_m);
                    cm = g[s] * divided;
                    dm = (rhs[s] + dm * g_m) * divided;
                    g_m = g[s];
                    if constexpr (n * BLK < RREG) {
                        c[n * BLK + s] = cm;
                        d[n * BLK + s] = dm;
                    } else {
                        sh.c[n * BLK + s - RREG][lane] = cm;
                        sh.d[n * BLK + s - RREG][lane] = dm;
                    }
                }
                return true;
            });
            CT data = CT(0);
            each_until<NBLK>([&](auto nc) {
                constexpr int n = NBLK - 1 - decltype(nc)::value;
#pragma clang loop unroll(full)
                for (int s = BLK - 1; s >= 0; --s) {
                    const int k = n * BLK + s;
                    CT cc, dd;
                    if constexpr (n * BLK < RREG) {
                        cc = c[k];
                        dd = d[k];
                    } else {
                        cc = sh.c[k - RREG][lane];
                        dd = sh.d[k - RREG][lane];
                    }
                    const CT v = dd - cc * data;
                    data = n == NBLK - 1 && k == nk - 1 ? dd : v;
                    sh.x[n & 1][s][lane] = data;
                }
                meet();
                return true;
            });
        }
    };

} // namespace gt355
