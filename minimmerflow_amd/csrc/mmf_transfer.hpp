// mmf_transfer.hpp -- large device-to-host copies into pageable memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace mmf {

// dst[0, bytes) = src, after everything enqueued on s; returns with dst
// complete.  From TRANSFER_MIN bytes the copy goes through pinned chunks that
// worker threads move on while the next ones arrive; smaller ones, and every
// copy while another thread holds the chunks, are a plain hipMemcpy.
hipError_t copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t s);

// The pinned chunks are shared by every context of the process, allocated by
// the first large copy and released with the last context.
void transfer_attach();
void transfer_detach();

}  // namespace mmf
