// What is measured of the device: integer-VALU rates, and which streams run
// side by side (probe.hip).
#pragma once

#include "field.h"
#include "runtime.h"

namespace nkr {

// v_mad_u64_u32 per second over the whole device, and this library's Fr
// Montgomery products per second (two independent chains per lane).
void valu_probe(int device, double *mad_per_s, double *fr_mul_per_s);

// Two non-blocking streams of the current device whose kernels overlap, where
// the process has such a pair.  Sets what it created as it goes (null before
// the call), so that a caller that cleans up after an exception can.
void create_overlapping_streams(hipStream_t *main, hipStream_t *side);

}  // namespace nkr
