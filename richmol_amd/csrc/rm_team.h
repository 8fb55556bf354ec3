// richmol_amd: several workgroups on each of a few wavepackets with real
// operators on domains of up to TEAM_MAX_ROWS rows (rm_team.hip).
#pragma once

#include "rm_block.h"

constexpr int TEAM_MAX_ROWS = 3840;   // 4 rows of the full vectors per lane

// Workgroups per wavepacket for these long domains side by side on n_cu
// compute units (max_grid at most, if > 0), 0: a domain does not fit, or
// (unless forced) the block kernel is as good.
int team_size(const std::vector<LongItem>& items, int n_cu, int32_t max_grid, bool forced);
// One cooperative launch for all items (team: team_size).
int team_run(void** ws, size_t* ws_bytes, const SubOp* d_ops, const SubOp* op0, const int4* d_items,
             const std::vector<LongItem>& items, int team, int32_t kcap, int32_t fixed_m, int32_t maxorder, double tol,
             int n_cu, hipStream_t s, int32_t abort_preset);
