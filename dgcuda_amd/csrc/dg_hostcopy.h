// Copies between the caller's pageable host arrays and device memory through
// pinned blocks.
#pragma once
#include "dg_solver.h"

namespace dgmi {

// A pinned block of the copies' pool, which kernels reach at its host address:
// a small array is read or written there by the kernel that converts it.  The
// work that uses it is waited for before the block is given back.
constexpr size_t PINNED_BLOCK_BYTES = size_t(1) << 20;
class PinnedBlock {
   public:
    Status take();
    ~PinnedBlock();
    double* data() const { return static_cast<double*>(p); }

   private:
    void* p = nullptr;
};

// The first two wait for the copy.  The device side is ready (copy_to_host) or free to
// be overwritten (copy_to_device) once the work queued on `st` has finished.
Status copy_to_host(void* dst, const void* src_dev, size_t bytes, hipStream_t st);
Status copy_to_device(void* dst_dev, const void* src, size_t bytes, hipStream_t st);
// copy_to_device; a small array is only queued, as a wait for each of a
// set-up's arrays costs more than its copy: the caller waits for `st` before
// it lets the array go
Status upload_small(void* dst_dev, const void* src, size_t bytes, hipStream_t st);

}  // namespace dgmi
