// conv_dwx.h — what the host side (conv_dw.hip) and the kernel instances (conv_dwx_inst.hip) of
// the three-part weight gradient share.
#pragma once
#include "common.h"

namespace tdh {

// filter rows x 4 (channel blocks x shares) waves
constexpr int dwx_threads(int RW) { return 64 * 4 * RW; }
// 4-pixel words of a staged row: the taps of the last 16-pixel group reach two 16-byte words past
// its start, and rows are an odd number of 16-byte words
constexpr int dwx_words(int TC, int S) { return (TC + 8) / 4; }

struct DwxArgs {
  const float *x, *dy;
  float *partial;     // [slices*tiles_x][Kc][C*R*S]
  float *partial_db;  // [slices*tiles_x][Kc], or null
  int batch, C, Kc, H, W, OH, OW, ph, pw, R, RS;
  int pwa;            // staged X column 0 is image column x0 - pwa
  int tiles_x, co_tiles, ci_tiles, fy_groups;
  int chunks_per_image, chunks_total, chunks_per_slice;  // chunks of 64/TC output rows
};

struct DwxPlan {
  bool ok;
  int tc, cob, cib, shift, slices, workgroups;
  size_t lds_bytes;
  DwxArgs args;
};

int dwx_launch_3_vec(const DwxPlan &p);
int dwx_launch_3_scalar(const DwxPlan &p);
int dwx_launch_5_scalar(const DwxPlan &p);

}  // namespace tdh
