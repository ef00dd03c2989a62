/*
 * snh_layout.h -- which element-pass layout a mesh can be launched in.  Plain
 * C, so that the rules can be checked on the host.
 */
#ifndef SNH_LAYOUT_H
#define SNH_LAYOUT_H

#include <stdint.h>

#include "../../include/snac_hip.h"

/* A row of doubles read with a scalar base and a 32-bit byte offset (ld_row)
   holds at most 2^29 of them. */
#define ROW_MOST 536870912
/* Tet per lane places a lane in the ten tets' rows of a component, so ten
   times its elements have to fit a row.  Its rows of nodes then fit too: a
   mesh has at most eight nodes per element. */
#define LANE_MOST_ELEMENTS (ROW_MOST / 10)

/* The layout that a context of N nodes and E elements runs when `variant` is
   chosen.  Beyond a layout's rows another takes its place: tet per wave for
   tet per lane, and element per lane, whose addresses have 64 bits, for tet
   per wave (a column one or two elements across reaches 2^29 nodes while its
   stress still fits the device's memory).  All give the same bits. */
static inline int32_t elem_layout(int32_t variant, int64_t N, int64_t E) {
    if (variant == SNH_ELEM_TET_PER_LANE && E > LANE_MOST_ELEMENTS) variant = SNH_ELEM_TET_PER_WAVE;
    if (variant == SNH_ELEM_TET_PER_WAVE && (N > ROW_MOST || E > ROW_MOST)) variant = SNH_ELEM_ELEMENT_PER_LANE;
    return variant;
}

/* The element-pass layout of a context that is not autotuned.  Tet per wave
   fills its loads, tet per lane starts more and smaller blocks and lets fewer
   tets wait for one that yields.  Measured (us, tet per lane / per wave):
   elastic 9.5 / 10.7 at 8112 elements, 14.2 / 12.0 at 16384, 52 / 38 at
   127000; Maxwell 11.1 / 12.9, 16.5 / 14.2, 65 / 50; Mohr-Coulomb extension
   98 / 102 at 256000, 177 / 179 at 441000, 397 / 364 at 885000, and yielding
   throughout 106 / 136, 199 / 236, 430 / 424; visco-plastic 111 / 117,
   197 / 209, 473 / 429.  In rows of few elements a wave's 64 span several
   rows of a Mohr-Coulomb model, whose yielding follows its planes and walls,
   and more waves wait: yielding throughout 392 / 619 at 8x64x1600, 456 / 487
   at 16x64x800, 404 / 466 at 32x40x640 and 411 / 433 at 48x40x430, against
   463 / 401 at 64x50x250; from 1.5e6 elements on rows of any length take tet
   per wave (1270 / 1206 at 16x64x2000). */
static inline int32_t default_elem_variant(int plastic, int viscoplastic, int64_t EI, int64_t E) {
    int64_t least = 12000;
    if (plastic || viscoplastic) least = 700000;
    if (plastic && EI < 64) least = 1500000;
    return E >= least ? SNH_ELEM_TET_PER_WAVE : SNH_ELEM_TET_PER_LANE;
}

/* whether a mesh can be a member of a batched launch: its element pass runs
   tet per lane or tet per wave, its node pass reads rows of E and N */
static inline int batch_addressable(int64_t N, int64_t E) {
    return E <= LANE_MOST_ELEMENTS && N <= ROW_MOST;
}

#endif
