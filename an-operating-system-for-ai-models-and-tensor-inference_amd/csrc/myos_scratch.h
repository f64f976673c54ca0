// Device scratch for the op tier's calls, kept between calls.
//
// hipMallocAsync + hipFreeAsync cost 10.5 us of host time per pair, from any
// pool, and a default pool also unmaps at every synchronisation (a gemm_bf16 of
// 2048 x 3584 x 18944 waited for alone: 1218 us against 596 among others). A
// block here is held by one call at a time and belongs to the stream that made
// it; a call on that stream takes it after hipStreamWaitEvent on the event its
// last holder recorded (4 us for both). The event, not the stream's handle, is
// what makes reuse safe: a handle that a later stream reuses waits for the
// earlier stream's work.
//
// Bounded: at most kScratchBlocks blocks and kScratchBytes per device. At a bound, a
// block that no call has taken for kScratchIdle calls (its stream is gone, or its
// shapes are) makes room: it is freed in stream order behind its event. With none,
// under stream capture, and where a block cannot be had, a call takes hipMallocAsync
// / hipFreeAsync. op_scratch_trim (myos_scratch_trim, and a closing model) gives idle
// blocks back.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace myos {

class OpScratch {
 public:
  OpScratch(size_t bytes, hipStream_t s);
  ~OpScratch();
  OpScratch(const OpScratch &) = delete;
  OpScratch &operator=(const OpScratch &) = delete;
  bool ok() const { return !bytes_ || p_; }
  void *get() const { return p_; }
  // after the call's last launch; the block is the next call's from here on
  hipError_t done();

 private:
  size_t bytes_;
  hipStream_t s_;
  void *p_ = nullptr;
  void *block_ = nullptr;  // the kept block, null for a plain allocation
};

// frees the current device's blocks that no call holds, waiting for their last work
void op_scratch_trim();

}  // namespace myos
