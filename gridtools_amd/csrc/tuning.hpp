// Tile choices of the tiled kernels and the table the autotuner fills.
#pragma once

#include <cstdint>

namespace gt355 {

    // Every tile shape instantiated for hdiff: X(TI, TJ, KC).  TI*TJ must be a multiple of 256.
#define GT355_HDIFF_TILES(X)                                                                                     \
    X(64, 4, 4) X(64, 4, 5) X(64, 4, 8) X(64, 4, 10) X(64, 4, 16)                                                  \
    X(64, 8, 4) X(64, 8, 5) X(64, 8, 8) X(64, 8, 10) X(64, 8, 16)                                                  \
    X(64, 16, 5) X(64, 16, 8)                                                                                      \
    X(128, 2, 8) X(128, 2, 10) X(128, 4, 5) X(128, 4, 8)                                                           \
    X(256, 1, 8) X(256, 1, 16)                                                                                     \
    X(32, 8, 8) X(32, 16, 8)

    // Every register-sweep shape instantiated for hdiff: X(JB, P).
#define GT355_HDIFF_SWEEPS(X) X(4, 4) X(8, 4) X(16, 4) X(16, 8) X(32, 4) X(32, 8)

    // Every column-pair sweep shape instantiated for hdiff: X(JB, P).
#define GT355_HDIFF_SWEEPS2(X) X(4, 4) X(8, 4) X(8, 8) X(16, 4) X(16, 8)

    // Every flat column-pair sweep shape instantiated for hdiff: X(JB, P), none of them among the strips above.
#define GT355_HDIFF_FLATS(X) X(4, 8) X(2, 6)

    // One hdiff launch configuration: impl 0 = LDS tile (a, b, c) = (TI, TJ, KC); impl 1 = register sweep
    // (a, b) = (JB, P); impl 2 = column-pair register sweep (a, b) = (JB, P) over 128-column strips, or with c = 1
    // over the flat list of pairs.
    struct hdiff_cfg {
        int impl, a, b, c;
    };
    // whether a configuration is a flat column-pair sweep (c = 1 with any other shape means its strips, as ever)
    inline bool hdiff_is_flat(const hdiff_cfg &c) {
#define GT355_IS_FLAT(JB, P) || (c.a == JB && c.b == P)
        return c.impl == 2 && c.c == 1 && (false GT355_HDIFF_FLATS(GT355_IS_FLAT));
#undef GT355_IS_FLAT
    }

    // The configuration for an hdiff launch, in this order: environment overrides (GT355_TUNE_hdiff_*), the entry
    // the autotuner recorded for (storage size, compute size, ni, nj, nk), the measured default for the storage type.
    hdiff_cfg hdiff_cfg_for(int st_size, int ct_size, int ni, int nj, int nk);
    // the measured default configuration for a storage size and domain (no tuned entry, no knob)
    hdiff_cfg hdiff_default_cfg(int st_size, int ni, int nj, int nk);
    // whether a configuration is one of the instantiated ones (hdiff.hip)
    bool hdiff_cfg_instantiated(hdiff_cfg cfg);
    void record_hdiff_cfg(int st_size, int ct_size, int ni, int nj, int nk, hdiff_cfg cfg, double us);

    // A batch's launch configuration, as the batch tuner records it for one list of domains (its signature).
    struct batch_cfg {
        int hjb;     // stencil phase: 8, 16 or 32 for 1, 2 or 4 rows per wavefront
        int hw;      // stored and returned as ever (2, 4, 8); the stencil phase has one wavefront per piece of work
        int w;       // vertical phase (or the single-launch forms): the persistent grid's setting (1..4)
        int deep_nk; // stored and returned as ever; the vertical phase chooses its register levels by depth alone
    };
    bool find_batch_cfg(uint64_t sig, int st_size, int ct_size, int impl, batch_cfg *out);
    void record_batch_cfg(uint64_t sig, int st_size, int ct_size, int impl, batch_cfg cfg, double us);

    // A named integer tuning knob: the environment variable GT355_TUNE_<name> if set, otherwise dflt.  The
    // environment is read once per process; tune_env_refresh (gt355_tune_env_refresh) reads it again.
    int tune_param(const char *name, int dflt);
    void tune_env_refresh();

} // namespace gt355
