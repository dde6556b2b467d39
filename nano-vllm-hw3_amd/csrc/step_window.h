// What a buffer load to LDS of step `t` of a walk over `steps` steps of `step` bytes is given, where the walk asks for steps past its
// last one (its wait counter is positional: the loads are issued, and read nothing): the resource's bytes and the uniform offset.
// A raw buffer load is in range if its lane's offset is below the resource's bytes less the uniform offset.  That difference may not
// go below zero: with an empty resource beside the offset of a step it is nearly 2^32, and what lies past the activations was read.
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define STEP_WINDOW_FN __host__ __device__ __forceinline__
#else
#define STEP_WINDOW_FN inline
#endif

struct StepWindow { unsigned bytes, at; };

STEP_WINDOW_FN StepWindow step_window(int t, int steps, unsigned step, unsigned bytes) {
    const bool there = t < steps;
    return {there ? bytes : 0u, there ? (unsigned)t * step : 0u};
}
