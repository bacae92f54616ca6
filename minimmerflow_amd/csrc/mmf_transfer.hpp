// mmf_transfer.hpp -- large device-to-host copies into pageable memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace mmf {

// dst[0, bytes) = src, after everything enqueued on s; returns with dst
// complete.  From TRANSFER_MIN bytes the copy goes through pinned chunks that
// worker threads move on while the next ones arrive; smaller ones, and every
// copy while another thread holds the chunks, are a plain hipMemcpy.
hipError_t copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t s);

// rows[N][5] on the host from the planes soa (field stride fs), after everything
// enqueued on s, and back, into a second set of planes too (copy, or nullptr);
// both through scratch, 5 N doubles on the device.
// Below a few thousand cells the host forms them: a launch and its wait cost
// more than its loop (see the figures in mmf_transfer.cpp).  The planes are
// filled on s, which may still run when the call returns; rows is free by then.
hipError_t planes_to_rows(double *rows, const double *soa, int64_t N, int64_t fs, double *scratch, hipStream_t s);
hipError_t rows_to_planes(const double *rows, double *soa, double *copy, int64_t N, int64_t fs, double *scratch,
                          hipStream_t s);

// The pinned chunks are shared by every context of the process, allocated by
// the first large copy and released with the last context.
void transfer_attach();
void transfer_detach();

}  // namespace mmf
