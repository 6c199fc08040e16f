// The bf16 tiles that pb_linear hands plain launches over many rows to (pb_linear_tiles.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "pb_common.h"

int pcb_linear_tiles(const pcb_linear_args& a, hipStream_t stream);
// two products of the same rows in one grid: the tiles for it where that is the better, else -1
int pcb_linear_tiles_pair_shape(const pcb_linear_args& a, const pcb_linear_args& b);
int pcb_linear_tiles_pair(const pcb_linear_args& a, const pcb_linear_args& b, int shape, hipStream_t stream);
// ... and those over some tens or hundreds of rows (pb_linear_waves.hip): which launches whose rows can be read in 16-byte chunks it is the better for
int64_t pcb_linear_waves_tiles(const pcb_linear_args& a);
bool pcb_linear_waves_fits(const pcb_linear_args& a);
int pcb_linear_waves(const pcb_linear_args& a, hipStream_t stream);
// ... and those in fp32 of so many tiles that splitting their operands may pay, with what such a launch takes (pb_linear_split.hip)
bool pcb_linear_split_fits(const pcb_linear_args& a);
float pcb_linear_split_us(const pcb_linear_args& a);
int pcb_linear_split_shape(const pcb_linear_args& a);
int pcb_linear_split(const pcb_linear_args& a, hipStream_t stream);
