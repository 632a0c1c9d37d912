// knobs.hpp — a renderer's speed knobs (prh_tuning) and what a frame makes of
// them.  A knob nobody set is a state of its own, not the default's value:
// only there a rule on the frame's size decides.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "../../include/prh.h"

namespace prh {

constexpr int32_t ITEM_PRIMS = 2048;     // prh_tuning.item_prims' default
constexpr int32_t MAIN_DIRECT_MAX = 48;  // and main_direct_max'
// The main view's triangles of at most so many pixel centres are drawn by the
// setup; with the knob never set, 16 in a frame of its own of at most 2^19
// triangles (2048 workgroups, 8 a CU).  48 -> 16: 480x270 of 197 k triangles
// 148 -> 138 us on the device and back, 1001x701 of 310 k 147 -> 134, 512x512 of
// 104 k 69 -> 64; 1.04 M triangles 414 -> 422 and a 64-view batch 2254 -> 2457,
// which are bound by the work and keep 48.  The line is where 1920x1080 without
// AO crosses (one stream, 16 against 48: 439 k triangles 176 / 180, 535 k 192 /
// 192, 823 k 228 / 224); smaller frames still gain a little past it (1001x701 of
// 679 k 167 / 179), 3840x2160 is within 1 % either way.
constexpr int32_t MAIN_DIRECT_FEW = 16, LATENCY_TRIS = 1 << 19;
// overlap_shadows is 1 from so many pixels.  A frame that has it so by default
// still takes one stream with at most LATENCY_TRIS triangles, whose setups
// leave the chip room and whose fork and joins cost more than they hide:
// 1001x701 of 310 k triangles 131 -> 122 us on the device and back, 1600x900 146
// -> 135, 3840x2160 314 -> 302, a textured 1600x1200 one 235 -> 224; 1.04 M
// triangles 1001x701 195 against 200 on one stream, 1920x1080 with AO 400
// against 417.  With AO 1920x1080 crosses there too (48 centres, one stream
// against two: 439 k triangles 320 / 318, 535 k 338 / 336, 823 k 381 / 372).
// With AO and 2^22 pixels the AO beside the shading is worth the fork (3840x2160
// of 116 k triangles 602 against 614).
constexpr size_t OVERLAP_PIXELS = 1 << 19, OVERLAP_AO_PIXELS = 1 << 22;

struct Knobs : prh_tuning {
    bool direct_set, overlap_set;  // main_direct_max, overlap_shadows: by a caller
};

inline Knobs default_knobs(size_t pixels) {
    Knobs k{};
    k.raster_wg_per_cu = 8, k.item_prims = ITEM_PRIMS;
    k.shadow_direct_max = 64, k.main_direct_max = MAIN_DIRECT_MAX;
    k.overlap_shadows = pixels >= OVERLAP_PIXELS ? 1 : 0;
    k.raster_tile = 16;
    return k;
}
inline bool valid_knobs(const prh_tuning& t) {
    const bool pow2 = t.item_prims > 0 && (t.item_prims & (t.item_prims - 1)) == 0;
    return t.raster_wg_per_cu >= 1 && t.raster_wg_per_cu <= 16 && pow2 && t.item_prims >= 64 && t.item_prims <= 8192 &&
           t.shadow_direct_max >= 0 && t.shadow_direct_max <= 256 && t.main_direct_max >= 0 && t.main_direct_max <= 256 &&
           (t.overlap_shadows == 0 || t.overlap_shadows == 1) &&
           (t.raster_tile == 8 || t.raster_tile == 16 || t.raster_tile == 32);
}
// A caller's setting (prh_set_tuning): every knob.  `ms` stays.
inline void set_knobs(Knobs& k, const prh_tuning& t) {
    const float ms = k.ms;
    static_cast<prh_tuning&>(k) = t;
    k.ms = ms;
    k.direct_set = k.overlap_set = true;
}

// What a frame of n_tris triangles uses.  wide: one of a batch's wide launches.
inline int32_t direct_centres(const Knobs& k, int64_t n_tris, bool wide) {
    return !k.direct_set && !wide && n_tris <= LATENCY_TRIS ? MAIN_DIRECT_FEW : k.main_direct_max;
}
inline bool two_streams(const Knobs& k, size_t pixels, int64_t n_tris, bool ao) {
    return k.overlap_shadows && (k.overlap_set || n_tris > LATENCY_TRIS || (ao && pixels >= OVERLAP_AO_PIXELS));
}

}  // namespace prh
