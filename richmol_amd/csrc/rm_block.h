// richmol_amd: one workgroup per wavepacket on domains of up to BLK_MAX_ROWS
// rows (rm_block.hip).
#pragma once

#include "rm_common.h"

// pairs of entries a lane holds in registers (1024 threads leave 128 vector
// registers; a pair takes 5 in FP64, 3 in FP32, 9 and 5 for complex operators,
// FP32 ones two more while they are multiplied: 20 FP32 pairs were slower, 28
// against 20 us a step)
constexpr int BLK_PAIRS(bool f32, bool real) { return real ? 12 : f32 ? 8 : 6; }
constexpr int BLK_MAX_ROWS = 4096;

// The launch variant of a domain of nslices slices: 0 when it does not fit;
// otherwise the same for every launch of that domain.
int blk_variant(int64_t nslices, bool real);
// Pairs of entries per lane of a domain of nslices slices, the longest of
// maxpairs: its launch keeps them in registers up to BLK_PAIRS.
int blk_part_pairs(int64_t nslices, int64_t maxpairs);
// Launches items [first, first + count) of one variant (by falling ppairs) on s; ws: workspace grown in place;
// pre_bytes: what operators formed ahead for all wavepackets of a job may take.
int blk_run(void** ws, size_t* ws_bytes, const SubOp* d_ops, const SubOp* op0, const int4* d_items,
            const std::vector<LongItem>& items, size_t first, size_t count, int variant, int32_t kcap, int32_t fixed_m,
            int32_t maxorder, double tol, bool f32, int n_cu, size_t pre_bytes, hipStream_t s);
