// The op tier's kept scratch blocks (myos_scratch.h).
#include "myos_scratch.h"

#include <mutex>
#include <vector>

namespace myos {
namespace {

constexpr size_t kScratchBytes = 256ull << 20;  // per device
constexpr int kScratchBlocks = 8;               // per device
constexpr size_t kGrain = 1ull << 20;

struct Block {
  void *p = nullptr;
  size_t size = 0;
  int dev = 0;
  hipStream_t owner = nullptr;
  hipEvent_t ev = nullptr;  // recorded after the last holder's launches
  bool used = false;        // ev has been recorded
  bool held = false;
};

std::mutex g_mu;
// never destroyed: a call may come from another static's destructor
std::vector<Block *> &blocks() {
  static std::vector<Block *> *v = new std::vector<Block *>();
  return *v;
}

void drop(Block *b) {
  auto &v = blocks();
  for (size_t i = 0; i < v.size(); i++)
    if (v[i] == b) {
      v.erase(v.begin() + i);
      break;
    }
  (void)hipEventDestroy(b->ev);
  delete b;
}

// The block of stream s that fits, grown or made where the bounds allow; null:
// the caller allocates for itself. Called with g_mu held; only stream-ordered
// calls on s, so a capture on another stream goes on undisturbed.
Block *take(size_t bytes, hipStream_t s) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  Block *small = nullptr;
  size_t total = 0;
  int count = 0;
  for (Block *b : blocks()) {
    if (b->dev != dev) continue;
    total += b->size;
    count++;
    if (b->held || b->owner != s) continue;
    if (b->size >= bytes) {
      if (b->used && hipStreamWaitEvent(s, b->ev, 0) != hipSuccess) return nullptr;
      b->held = true;
      return b;
    }
    small = b;
  }
  if (bytes > kScratchBytes) return nullptr;
  const size_t size = (bytes + kGrain - 1) / kGrain * kGrain;
  if (total - (small ? small->size : 0) + size > kScratchBytes) return nullptr;
  if (small) {  // too small for this stream's calls: replaced
    if (small->used && hipStreamWaitEvent(s, small->ev, 0) != hipSuccess) return nullptr;
    if (hipFreeAsync(small->p, s) != hipSuccess) return nullptr;
    drop(small);
  } else if (count >= kScratchBlocks) {
    return nullptr;
  }
  Block *b = new Block();
  b->size = size;
  b->dev = dev;
  b->owner = s;
  b->held = true;
  if (hipEventCreateWithFlags(&b->ev, hipEventDisableTiming) != hipSuccess) {
    delete b;
    return nullptr;
  }
  if (hipMallocAsync(&b->p, size, s) != hipSuccess) {
    (void)hipEventDestroy(b->ev);
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
  if (hipStreamIsCapturing(s, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone) {
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
  std::lock_guard<std::mutex> lock(g_mu);
  int cur = 0;
  if (hipGetDevice(&cur) != hipSuccess) return;
  for (size_t i = blocks().size(); i-- > 0;) {
    Block *b = blocks()[i];
    if (b->held || b->dev != cur) continue;
    if (b->used && hipEventSynchronize(b->ev) != hipSuccess) continue;
    if (hipFree(b->p) != hipSuccess) continue;
    drop(b);
  }
}

}  // namespace myos
