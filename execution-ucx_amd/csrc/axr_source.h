// Plans made straight from a sequence of framework tensors.  Shared by the planner and by
// lib/_axr_torch; not part of the C ABI.
#ifndef AXR_SOURCE_H_
#define AXR_SOURCE_H_

#include <stddef.h>
#include <stdint.h>

#include "axon_rocm.h"

extern "C" {

// Tensors that are described a few at a time while the plan is made of them, instead of all of them
// into an array first: for 65,536 tensors that array is 4 MB, written and read once, and giving such blocks
// back makes malloc return the heap to the system, so that every call pages its memory in again.
struct axr_tensor_source {
  size_t count;
  // Fills out[0, n) for the tensors first, first + 1, ...; nonzero gives the plan up.  Called with ascending
  // `first` and without a gap.  Shapes and strides have to stay where they are until the next call.
  int (*describe)(axr_tensor_source* self, size_t first, size_t n, axr_tensor_t* out);
};

// axr_plan_create and axr_plan_from_header_bind for such a source.  The second one does not copy the
// header: it has to stay where it is for as long as the plan lives.
typedef int axr_plan_create_from_fn(axr_tensor_source* tensors, uint32_t align, axr_plan_t** plan);
typedef int axr_plan_bind_from_fn(const void* header, size_t length, axr_tensor_source* tensors, axr_plan_t** plan);
AXR_API axr_plan_create_from_fn axr_plan_create_from;
AXR_API axr_plan_bind_from_fn axr_plan_bind_from;

}  // extern "C"

#endif  // AXR_SOURCE_H_
