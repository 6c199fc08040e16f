// The bf16 tiles that pb_linear hands plain launches over many rows to (pb_linear_tiles.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "pb_common.h"

int pcb_linear_tiles(const pcb_linear_args& a, hipStream_t stream);
