// Device to host copies of whole fields.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace lbm {

// Copies `bytes` from the device to host memory behind the work enqueued on
// `s`, and returns when they have arrived.
hipError_t read_back(void* dst, const void* src, size_t bytes, hipStream_t s);

// Copies the `take` most recent of `written` force records (6 doubles each)
// from a device ring of `cap`, oldest first.
hipError_t read_records(double* out, const double* ring, size_t cap, unsigned long long written, size_t take,
                        hipStream_t s);

// The pinned staging of read_back lives from the first large copy until the
// last user lets go of it.
void read_back_retain();
void read_back_release();

}  // namespace lbm
