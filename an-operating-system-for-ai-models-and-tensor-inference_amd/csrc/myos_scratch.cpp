// The op tier's kept scratch blocks (myos_scratch.h).
#include "myos_scratch.h"

#include <stdint.h>

#include <mutex>
#include <vector>

namespace myos {
namespace {

constexpr size_t kScratchBytes = 256ull << 20;  // per device
constexpr int kScratchBlocks = 8;               // per device
constexpr size_t kGrain = 1ull << 20;
constexpr uint64_t kScratchIdle = 256;  // calls on the device: far more than live streams take turns over

struct Block {
  void *p = nullptr;
  size_t size = 0;
  int dev = 0;
  hipStream_t owner = nullptr;
  hipEvent_t ev = nullptr;  // recorded after the last holder's launches
  uint64_t last = 0;        // the call that took it last
  bool used = false;        // ev has been recorded
  bool held = false;
};

std::mutex g_mu;
uint64_t g_calls = 0;
// never destroyed: a call may come from another static's destructor
std::vector<Block *> &blocks() {
  static std::vector<Block *> *v = new std::vector<Block *>();
  return *v;
}

// a failed call here is no error of the caller's: the launches that follow read
// hipGetLastError
bool good(hipError_t e) {
  if (e != hipSuccess) (void)hipGetLastError();
  return e == hipSuccess;
}

void unlist(Block *b) {
  auto &v = blocks();
  for (size_t i = 0; i < v.size(); i++)
    if (v[i] == b) {
      v.erase(v.begin() + i);
      break;
    }
}

// b's memory back to the pool, on s behind b's last work
bool give_back(Block *b, hipStream_t s) {
  if (b->used && !good(hipStreamWaitEvent(s, b->ev, 0))) return false;
  if (!good(hipFreeAsync(b->p, s))) return false;
  unlist(b);
  (void)good(hipEventDestroy(b->ev));
  delete b;
  return true;
}

// The block of stream s that fits, grown or made where the bounds allow; null:
// the caller allocates for itself. Called with g_mu held; only stream-ordered
// calls on s, so a capture on another stream goes on undisturbed.
Block *take(size_t bytes, hipStream_t s) {
  int dev = 0;
  if (!good(hipGetDevice(&dev))) return nullptr;
  const uint64_t now = ++g_calls;
  Block *small = nullptr;
  size_t total = 0;
  int count = 0;
  for (Block *b : blocks()) {
    if (b->dev != dev) continue;
    total += b->size;
    count++;
    if (b->held || b->owner != s) continue;
    if (b->size >= bytes) {
      if (b->used && !good(hipStreamWaitEvent(s, b->ev, 0))) return nullptr;
      b->held = true;
      b->last = now;
      return b;
    }
    small = b;
  }
  if (bytes > kScratchBytes) return nullptr;
  const size_t size = (bytes + kGrain - 1) / kGrain * kGrain;
  if (small) {  // too small for this stream's calls: replaced
    total -= small->size;
    count--;
  }
  while (count >= kScratchBlocks || total + size > kScratchBytes) {
    Block *idle = nullptr;
    for (Block *b : blocks())
      if (b->dev == dev && !b->held && b != small && now - b->last > kScratchIdle &&
          (!idle || b->last < idle->last))
        idle = b;
    if (!idle) return nullptr;
    const size_t was = idle->size;
    if (!give_back(idle, s)) return nullptr;
    total -= was;
    count--;
  }
  if (small && !give_back(small, s)) return nullptr;
  Block *b = new Block();
  b->size = size;
  b->dev = dev;
  b->owner = s;
  b->last = now;
  b->held = true;
  if (!good(hipEventCreateWithFlags(&b->ev, hipEventDisableTiming))) {
    delete b;
    return nullptr;
  }
  if (!good(hipMallocAsync(&b->p, size, s))) {
    (void)good(hipEventDestroy(b->ev));
    delete b;
    return nullptr;
  }
  blocks().push_back(b);
  return b;
}

}  // namespace

OpScratch::OpScratch(size_t bytes, hipStream_t s) : bytes_(bytes), s_(s) {
  if (!bytes) return;
  // a captured graph may be replayed while another call holds the block
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (good(hipStreamIsCapturing(s, &cap)) && cap == hipStreamCaptureStatusNone) {
    std::lock_guard<std::mutex> lock(g_mu);
    if (Block *b = take(bytes, s)) {
      block_ = b;
      p_ = b->p;
      return;
    }
  }
  if (hipMallocAsync(&p_, bytes, s) != hipSuccess) p_ = nullptr;
}

hipError_t OpScratch::done() {
  if (!p_) return hipSuccess;
  hipError_t e;
  if (Block *b = (Block *)block_) {
    e = hipEventRecord(b->ev, s_);
    std::lock_guard<std::mutex> lock(g_mu);
    b->used = true;
    // without its event nothing says when the block is free again: it stays held
    b->held = e != hipSuccess;
  } else {
    e = hipFreeAsync(p_, s_);
  }
  p_ = nullptr;
  return e;
}

OpScratch::~OpScratch() { (void)done(); }

void op_scratch_trim() {
  int cur = 0;
  if (!good(hipGetDevice(&cur))) return;
  std::vector<Block *> idle;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    for (Block *b : blocks())
      if (!b->held && b->dev == cur) idle.push_back(b);
    for (Block *b : idle) unlist(b);
  }
  // out of the list nobody else sees them: the waits hold up no other call
  for (Block *b : idle) {
    if ((b->used && !good(hipEventSynchronize(b->ev))) || !good(hipFree(b->p))) {
      std::lock_guard<std::mutex> lock(g_mu);
      blocks().push_back(b);
      continue;
    }
    (void)good(hipEventDestroy(b->ev));
    delete b;
  }
}

}  // namespace myos
