// Which decode steps are one launch (step_kernel), of one or of several workgroups per group, which are two or three, and which are
// scoring + selection and attention in launches of their own; where an attention's workgroups count their arrivals.  Host code only.
#pragma once
#include <stdint.h>

#include "../../include/retro_mi355.h"

// Heads of a group as the kernels pad them.
static inline int gs_pad_of(int gs) { return gs <= 4 ? 4 : (gs <= 8 ? 8 : 16); }

// Groups that an attention launch gives one workgroup each: few rows (fewer the more heads share their arithmetic), or no
// compute unit left for a second one.
static inline bool attend_alone(int64_t rows, int gs, int BG) { return rows * gs_pad_of(gs) <= 384 * 4 || BG > 128; }

// Words between the arrival counters of a launch's waves, eight to a group of more than one workgroup, which up to 128 groups
// have (attend_common.h).  Every arrival is an atomic at the memory side, where those on one line wait for each other: counters have
// lines of their own while there is room.  Four counters to 64 bytes / one to a line of 128, us: 2 groups of 8 heads, 15100 rows
// 13.8 / 12.4, 1 of 8, 40000 18.0 / 16.5, 8 of 8, 20000 21.2 / 19.3, 6 of 8, 3000 9.4 / 9.1; half a line the same.
static constexpr int attend_counter_pitch(int BG) { return BG <= 16 ? 32 : BG <= 32 ? 16 : BG <= 64 ? 8 : 4; }

#define STEP_CLUSTERS 512
// Selection and attention in one launch, and the scoring too up to STEP_CLUSTERS: what step.hip's kernels hold.  (A probe per
// thread; 512 threads, or wide 1024, whose registers do not hold sixteen heads; up to 32 clusters a thread; with sixteen heads
// 32 KB of LDS are left for the tables, of which those of up to 512 clusters take 8; without sizes and first rows there are none.  A
// workgroup that scores has a compute unit to itself: 264 groups of 4 heads, 512 clusters, a captured layer 33.2 us in two launches, 36.4 in one.)
static inline bool step_is_wide(const ri_decode_step_t* s) {
  return s->gs <= 8 && s->np <= 1024 && (s->nc > 8192 || s->np > 512);
}
static inline bool step_is_joined(const ri_decode_step_t* s) {
  if (!s->cluster_size_i32 || !s->cluster_start) return false;
  if (s->nc <= STEP_CLUSTERS) return s->BG <= 256;
  if (s->nc > 16384) return false;
  return step_is_wide(s) || (s->np <= 512 && (s->gs <= 8 || 3 * s->np + s->es <= 8000));
}

// Who sums the scores of a step that is scored before: dist_kernel, which then hands keys over, or the workgroups that select, from
// the logits.  dist_kernel / the selecting workgroups, captured layers with their appends, us:
//  * Up to six heads dist_kernel past 4096 clusters: 32 groups of 4 heads, 8192 44.8 / 47.6, 5632 36.1 / 38.7, 4096 29.5 / 29.2; 8 of 4, 5632
//    24.3 / 26.5; of 1, 32 of 8192 42.9 / 44.0; 16 of 5, 2560 20.8 / 20.8, 128 of 6, 3104 52.8 / 52.4.
//  * Seven and eight heads past 2048 in up to 64 groups: 12 of 7, 1920 23.0 / 22.0, 32 of 8, 2048 25.7 / 24.7; 8 of 7, 2304 19.6 / 20.4, 8 of 8,
//    3328 21.6 / 22.3, 32 of 8, 2816 24.9 / 25.7; 56 of 7, 2304 27.7 / 28.1, 3840 34.7 / 35.5, 64 of 7, 2304 28.9 / 29.5, 3328 36.4 / 37.0, 64 of
//    8, 2304 29.8 / 30.4, 3840 37.4 / 38.2.  In more groups they fill the chip with selecting workgroups, and the second launch is made up
//    for no longer: 80 of 7, 2304 33.1 / 33.7, 3328 40.4 / 40.0, 72 of 8, 3840 41.6 / 41.6, 96 of 7, 2816 45.1 / 45.0, of 8 42.9 / 42.7, 112 of
//    7 47.9 / 47.3, 128 of 8 52.3 / 52.0, 3840 59.9 / 59.5, 192 of 7, 3328 78.9 / 78.4, 256 of 8, 2816 90.8 / 90.0, 3840 111.3 / 110.4.
//  * More heads past 2048 in any number of groups: 8 of 16, 2048 26.0 / 25.9, 64 of 16, 1024 28.8 / 27.6; 56 of 9, 2304 30.6 / 33.7, of 12, 2816
//    37.1 / 40.8, of 16, 4096 43.0 / 46.7, 72 of 9, 4096 47.1 / 48.5, of 16, 2816 43.7 / 47.0, 128 of 9, 2304 47.6 / 49.3, of 12, 3328 63.0 /
//    65.5, of 16, 4096 78.0 / 80.0.  (Eight clusters of sixteen heads to a thread are 157 registers and 118 KB of LDS.)
static inline bool step_sums_apart(int gs, int BG, int nc) {
  return nc > (gs > 8 ? 2048 : gs > 6 && BG <= 64 ? 2048 : 4096);
}

// Steps that score for themselves, of up to eight heads (step_kernel).  Up to 128 groups several workgroups per group make them.
// Captured layers with their appends, us, one / several: 8 groups of 4 heads, 512 clusters 13.85 / 13.35; of 1, 104 11.65 / 11.40; of 8, 256
// 13.30 / 12.90; 88 of 1, 120 12.10 / 11.85; 16 of 4, 256 12.35 / 12.10; 32 of 4, 496 13.75 / 13.40; 128 of 4, 496 15.20 / 14.90, of 8, 256
// 14.10 / 13.70; 1 of 4, 320 11.90 / 11.60.  Past 128 there is no second one, and where the usual 16 tokens to a cluster make no more than STEP_ROWS
// rows the kernel's form for one, which knows of no other, makes them: form for several / for one 136 groups of 4 heads, 96 clusters 12.4 / 12.3,
// 256 13.35 / 13.15, of 8, 512 17.7 / 17.6; 192 of 8, 256 15.4 / 15.1; 256 of 4, 256 15.65 / 15.4, of 8, 512 22.6 / 22.4.
#define STEP_ROWS 448
static inline bool step_is_one(const ri_decode_step_t* s, int static_len) {
  return s->BG > 128 && step_is_joined(s) && s->nc <= STEP_CLUSTERS && s->gs <= 8 &&
         static_len + (int64_t)s->np * 16 + s->es <= STEP_ROWS;
}

// Rows up to which one of several workgroups attends them all and the others leave (step_kernel looks behind the selection, where
// a captured step's length and what the clusters hold are known).  Earlier kernels' captured layers with their appends, us, by the rows, several
// that all work / that leave: 8 groups of 4 heads, 192 clusters 161 16.0 / 14.8, 281 16.2 / 15.6, 411 16.0 / 16.1; 8 of 8, 320 223 16.9 / 15.8,
// 343 16.9 / 16.7; 32 of 4, 512 331 17.4 / 17.6.  With two workgroups per group only: 128 groups of 4 heads, 512 331 20.1 / 18.9, 581 22.4 /
// 22.3, of 8 331 21.0 / 19.9, 581 23.0 / 22.9.
static inline int step_alone_rows(int BG) { return BG > 64 ? 640 : 336; }
