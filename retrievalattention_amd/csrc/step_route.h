// Which decode steps one workgroup per group makes in one launch (step_kernel), which several do, and which are scoring +
// selection and attention in launches of their own; where an attention's workgroups count their arrivals.  Host code only.
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

// Short: what one workgroup may have to itself (step_is_alone: and does).  It scores for itself (select.hip), and usually (16
// tokens per retrieved cluster) has no more rows than it attends as fast as two launches do (figures of both, before
// step_is_joined): 8 groups of 8 heads 424 rows 14.6 us against 15.5, 488: 14.8 / 15.7, 552: 15.9 /
// 15.5; of 4 heads 488: 13.8 / 15.0, 552: 15.4 / 14.8; one group of 8 heads 488: 14.5 / 15.0, 552: 15.6 / 14.9.
// The rows are not known here when the kernel reads the zone's length from the device, as a captured step does until the
// zone is full, and never what the retrieved clusters hold:
//  * Where the attention by itself would be one workgroup per group all the same, one launch is faster whatever they turn
//    out to be.  8 groups of 4 heads captured with 331 rows: then 12.3 us against 14.2, at 1354 rows 22.3 / 24.4, with 512
//    tokens in each of 9 clusters 53.6 / 55.6; 128 groups 13.9 / 16.3 and 25.7 / 27.8.
//  * Elsewhere the other route has more workgroups, so the rows that the zone can hold decide, and those of the clusters are
//    bounded by the page limit and the store.  8 groups of 8 heads captured with 331 rows: then 13.1 us against 15.5, at 458
//    rows 15.0 / 15.5, but at 762 18.1 / 16.6, 962: 20.1 / 17.8, 1354: 24.4 / 18.8; with 64 tokens in each of 9 clusters (763
//    rows) 18.5 / 16.8, with 512: 64.9 / 28.5.  At twice the limit the most crowded clusters cost what usual ones save.
#define STEP_CLUSTERS 512
#define STEP_ROWS 448
#define STEP_ROWS_CROWDED (2 * STEP_ROWS)
static inline bool step_is_short(const ri_decode_step_t* s, int static_len) {
  if (s->nc > STEP_CLUSTERS || s->gs > 8 || s->BG > 256 || !s->cluster_size_i32 || !s->cluster_start) return false;
  const int64_t usual = (int64_t)s->np * 16 + s->es;
  if (static_len + usual > STEP_ROWS) return false;
  if (attend_alone(static_len + usual, s->gs, s->BG)) return true;
  const int64_t zone = s->static_len_dev ? s->steady_stride : static_len;
  const int64_t pages = (int64_t)s->max_pages * s->page, held = pages < s->store_stride ? pages : s->store_stride;
  return zone + usual <= STEP_ROWS && zone + s->es + held <= STEP_ROWS_CROWDED;
}

// Selection and attention in one launch, and the scoring too up to STEP_CLUSTERS: what step.hip's kernels hold.  (A probe per
// thread; 512 threads, or wide 1024, whose registers do not hold sixteen heads; up to 32 clusters a thread; with sixteen heads
// 32 KB of LDS are left for the tables; without sizes and first rows there are none.  A workgroup that scores has a compute unit
// to itself: 264 groups of 4 heads, 512 clusters 32.5 us in two launches, 37.3 in one.)
static inline bool step_is_wide(const ri_decode_step_t* s) {
  return s->gs <= 8 && s->np <= 1024 && (s->nc > 8192 || s->np > 512);
}
static inline bool step_is_joined(const ri_decode_step_t* s) {
  if (!s->cluster_size_i32 || !s->cluster_start) return false;
  if (s->nc <= STEP_CLUSTERS) return s->gs <= 8 && s->BG <= 256;
  if (s->nc > 16384) return false;
  return step_is_wide(s) || (s->np <= 512 && (s->gs <= 8 || 3 * s->np + s->es <= 8000));
}

// Of the short steps those that one workgroup per group makes as fast as several, which take the same at any length (us, one /
// several).  8 groups of 8 heads 225 rows 13.4 / 14.2, 321: 14.1 / 14.2, 353: 14.5 / 14.2, 417: 15.1 / 14.2; of 4 heads 225: 12.7
// / 13.5, 321: 13.4 / 13.5, 353: 13.7 / 13.5, with 512 clusters 331: 13.9 / 13.8 (a step, 15.2 either way), 523: 16.0 / 13.8; of 1 head 321: 13.0 / 13.1; 32
// groups of 4 heads 321: 14.2 / 14.2, 417: 15.3 / 14.6.  With two workgroups per group only: 128 groups of 4 heads 417: 16.4 / 17.7,
// of 8 heads, 512 clusters 587: 21.0 / 21.1; past 128 there is no second one.  (Several workgroups that find fewer rows than
// the line leave them to one: step_kernel.)
// A captured step starts at the length at hand and ends at the zone's, and may grow past the line.  One wins at first, several
// later; from sixteen groups on every workgroup more shows in the start of the launch.  Zones of 323 rows, us a layer at the
// first length, on average and at the last, several | one: 16 groups of 4 heads, up to 508 rows 15.2, 17.0, 18.2 | 15.2, 16.8,
// 18.4; 32 of 4, 508 16.4, 17.6, 18.3 | 16.0, 17.5, 18.9; 64 of 4, 477 15.9, 17.2, 18.2 | 15.6, 17.1, 18.5; 32 of 8, 446 16.2,
// 17.7, 18.4 | 16.0, 17.5, 19.0; 40 of 2, 477 15.3, 16.5, 17.4 | 15.2, 16.7, 18.5.  Past the line 24 of 4, 531 16.6, 17.4, 18.1 |
// 16.2, 17.7, 19.1; 64 of 4, 554 17.1, 18.2, 18.7 | 16.5, 18.3, 19.9; 8 of 4, 477 14.1, 15.3, 16.3 | 14.2, 15.5, 17.1.
static inline int step_alone_rows(int BG) { return BG > 64 ? 640 : 336; }
static inline int step_alone_end(int BG) { return BG > 64 ? 800 : BG >= 16 ? 512 : 420; }
static inline bool step_is_alone(const ri_decode_step_t* s, int static_len) {
  if (s->BG > 128) return true;
  const int64_t usual = (int64_t)s->np * 16 + s->es, zone = s->static_len_dev ? s->steady_stride : static_len;
  return static_len + usual <= step_alone_rows(s->BG) && zone + usual <= step_alone_end(s->BG);
}
