// The layers of a decode step of one row as one resident launch (decode_resident.hip).
#pragma once

#include "../../include/logismos_decode.h"

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace lg {

// Bytes of the step's workspace that the launch uses: 0 where the geometry is not one of its own.
size_t decode_resident_bytes(const logismos_decode_config_t& c);

// Whether a step of one row is better there than operator by operator.
bool decode_resident_pays(const logismos_decode_config_t& c);

// Whether a step of t rows over these operands can run there.
bool decode_resident_applies(const logismos_decode_config_t& c, const logismos_decode_layer_t* layers,
                             const logismos_decode_batch_t& b, int t);

// What tests set (0: what a step takes).
struct ResidentLimits {
    int workgroups;  // launched (fewer than the work is cut for do the same work with the same result)
    int polls;       // of a wave, after which it gives up
    int tickets;     // with which the step is closed: the workgroups without one leave
};

// All layers: residual stream in and out in b.hidden_f32, K/V rows into the pools.
hipError_t decode_resident_launch(const logismos_decode_config_t& c, const logismos_decode_layer_t* layers,
                                  const logismos_decode_batch_t& b, void* region, hipStream_t st,
                                  const ResidentLimits& limits = {});

}  // namespace lg
