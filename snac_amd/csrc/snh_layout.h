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

/* whether a mesh can be a member of a batched launch: its element pass runs
   tet per lane or tet per wave, its node pass reads rows of E and N */
static inline int batch_addressable(int64_t N, int64_t E) {
    return E <= LANE_MOST_ELEMENTS && N <= ROW_MOST;
}

#endif
