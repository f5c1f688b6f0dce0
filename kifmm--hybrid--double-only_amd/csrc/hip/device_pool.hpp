/*
 * device_pool.hpp -- what handles and tree builds take from the device: idle
 * streams, and memory carved from few allocations.
 *
 * A program that rebuilds its tree every step creates and destroys both each
 * time, and at 131 thousand points that cost more than the work: 283 hipMallocs
 * (each new 2 MB of the runtime's own pool takes 0.3 ms, 4.8 ms in all; the
 * frees take as long, when the last event that refers to the memory goes) and
 * three streams whose hardware queue went with the last of them (3 ms to take
 * down, in stream and event destruction, and set up again).  With both kept,
 * uploads staged (dev_upload) and downloads queued (Down, kifmm_gpu_tree.hip)
 * a step of that size, tree to potentials, went from 18.0 to 10.5 ms.
 */
#ifndef KIFMM_DEVICE_POOL_HPP
#define KIFMM_DEVICE_POOL_HPP
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <new>
#include <utility>
#include <vector>

namespace kifmm_dev {

/* What is idle between owners: non-blocking streams of default priority, at
 * most STREAMS_KEPT in the whole process and over all devices (the hardware has
 * four queues per process), and blocks of device arenas, BLOCKS_KEPT bytes at
 * most.  A stream beyond those, or one that did not end its work cleanly, is
 * destroyed.  An idle stream holds no user data.  The blocks go back to the
 * runtime when an arena's allocation fails, and with the streams by
 * kifmm_gpu_release_idle.
 * hipDeviceReset destroys all of it.  So a device's idle things count as long
 * as its mark does, a small allocation made with the first of them: an
 * allocation's buffer id names no other one later, whatever its address.
 * After a reset they are forgotten, not used and not freed. */
constexpr size_t STREAMS_KEPT = 4;
constexpr size_t BLOCKS_KEPT = (size_t)128 << 20;
struct Block {
  int dev;
  void* p;
  size_t bytes;
};
struct IdlePool {
  struct Mark {
    int dev;
    void* p;
    unsigned long long id;
  };
  std::mutex m;
  std::vector<std::pair<int, hipStream_t>> streams;
  std::vector<Block> blocks;
  size_t bytes = 0; /* of blocks */
  std::vector<Mark> marks;

  static bool buffer_id(void* p, unsigned long long* id) {
    *id = 0;
    if (hipPointerGetAttribute(id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, (hipDeviceptr_t)p) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
  }
  /* whether what is idle of dev can be used; m is held, here and below */
  bool alive(int dev) {
    for (size_t k = 0; k < marks.size(); k++) {
      if (marks[k].dev != dev) continue;
      unsigned long long id;
      if (buffer_id(marks[k].p, &id) && id == marks[k].id) return true;
      forget(dev);
      return false;
    }
    return false; /* nothing of dev is idle */
  }
  /* before something of dev is put away; false: it cannot be kept */
  bool mark(int dev) {
    if (alive(dev)) return true;
    int cur = -1;
    Mark k{dev, nullptr, 0};
    if (hipGetDevice(&cur) != hipSuccess || cur != dev) return false;
    if (hipMalloc(&k.p, 1) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    if (buffer_id(k.p, &k.id)) try {
        marks.push_back(k);
        return true;
      } catch (const std::bad_alloc&) {
      }
    (void)hipFree(k.p);
    return false;
  }
  void forget(int dev) {
    streams.erase(std::remove_if(streams.begin(), streams.end(), [&](const auto& e) { return e.first == dev; }),
                  streams.end());
    for (const Block& b : blocks)
      if (b.dev == dev) bytes -= b.bytes;
    blocks.erase(std::remove_if(blocks.begin(), blocks.end(), [&](const Block& b) { return b.dev == dev; }),
                 blocks.end());
    marks.erase(std::remove_if(marks.begin(), marks.end(), [&](const Mark& k) { return k.dev == dev; }), marks.end());
  }
  void free_blocks() {
    for (size_t k = blocks.size(); k-- > 0;) {
      if (k >= blocks.size() || !alive(blocks[k].dev)) continue; /* forgotten */
      (void)hipFree(blocks[k].p);
      bytes -= blocks[k].bytes;
      blocks.erase(blocks.begin() + (long)k);
    }
  }
};
inline IdlePool& idle_pool() {
  alignas(IdlePool) static char at[sizeof(IdlePool)];
  static IdlePool* const p = new (at) IdlePool; /* never destroyed: the runtime may be gone by then */
  return *p;
}
/* a stream of device dev, the current one */
inline hipError_t take_stream(int dev, hipStream_t* s) {
  *s = nullptr;
  {
    IdlePool& p = idle_pool();
    std::lock_guard<std::mutex> lock(p.m);
    if (p.alive(dev))
      for (size_t k = 0; k < p.streams.size(); k++)
        if (p.streams[k].first == dev) {
          *s = p.streams[k].second;
          p.streams.erase(p.streams.begin() + (long)k);
          break;
        }
  }
  return *s ? hipSuccess : hipStreamCreateWithFlags(s, hipStreamNonBlocking);
}
/* waits for the stream's work first */
inline void give_stream(int dev, hipStream_t s) {
  if (!s) return;
  if (hipStreamSynchronize(s) == hipSuccess) {
    IdlePool& p = idle_pool();
    std::lock_guard<std::mutex> lock(p.m);
    if (p.streams.size() < STREAMS_KEPT && p.mark(dev)) try {
        p.streams.emplace_back(dev, s);
        return;
      } catch (const std::bad_alloc&) {
      }
  }
  (void)hipStreamDestroy(s);
}
inline void* take_block(int dev, size_t bytes) {
  IdlePool& p = idle_pool();
  std::lock_guard<std::mutex> lock(p.m);
  if (!p.alive(dev)) return nullptr;
  for (size_t k = 0; k < p.blocks.size(); k++)
    if (p.blocks[k].dev == dev && p.blocks[k].bytes == bytes) {
      void* const q = p.blocks[k].p;
      p.blocks.erase(p.blocks.begin() + (long)k);
      p.bytes -= bytes;
      return q;
    }
  return nullptr;
}
/* false: not kept */
inline bool give_block(const Block& b) {
  IdlePool& p = idle_pool();
  std::lock_guard<std::mutex> lock(p.m);
  if (p.bytes + b.bytes > BLOCKS_KEPT || !p.mark(b.dev)) return false;
  try {
    p.blocks.push_back(b);
  } catch (const std::bad_alloc&) {
    return false;
  }
  p.bytes += b.bytes;
  return true;
}
inline void drop_blocks() {
  IdlePool& p = idle_pool();
  std::lock_guard<std::mutex> lock(p.m);
  p.free_blocks();
}
inline void drop_idle() {
  IdlePool& p = idle_pool();
  std::lock_guard<std::mutex> lock(p.m);
  p.free_blocks();
  while (!p.marks.empty()) {
    const IdlePool::Mark k = p.marks.back();
    if (!p.alive(k.dev)) continue; /* forgotten, the mark with it */
    for (const auto& s : p.streams)
      if (s.first == k.dev) (void)hipStreamDestroy(s.second);
    (void)hipFree(k.p);
    p.forget(k.dev);
  }
}

/* hipMalloc, with the idle blocks given back if it needs their memory; what
 * failed is returned and not left for a later launch check to find */
inline hipError_t device_malloc(void** p, size_t bytes) {
  hipError_t e = hipSuccess;
  for (int k = 0; k < 2; k++) {
    *p = nullptr;
    if ((e = hipMalloc(p, bytes)) == hipSuccess) return e;
    (void)hipGetLastError();
    if (k == 0) drop_blocks();
  }
  *p = nullptr;
  return e;
}

/* Device memory of one owner: pieces of up to OWN bytes are cut from blocks of
 * 8, 16, 32, then 64 MB, larger ones are allocations of their own.  No two
 * owners share a block at a time; a block changes hands only when its owner's
 * work has ended (stream, or the owner's word for it), with what the owner wrote
 * in it. */
class DeviceArena {
 public:
  static constexpr size_t OWN = (size_t)8 << 20, MOST = (size_t)64 << 20, ALIGN = 256;

  /* st: the stream whose work uses the memory; null when the owner waits for
   * it before free() */
  explicit DeviceArena(hipStream_t st = nullptr) : st_(st) {}
  DeviceArena(const DeviceArena&) = delete;
  DeviceArena& operator=(const DeviceArena&) = delete;
  ~DeviceArena() { free(); }

  /* of the current device; null when there is no memory; aligned to ALIGN */
  void* get(size_t bytes) {
    bytes = (std::max<size_t>(bytes, 1) + ALIGN - 1) / ALIGN * ALIGN;
    if (bytes > OWN) {
      own_.reserve(own_.size() + 1); /* a throw here loses nothing */
      void* p;
      if (device_malloc(&p, bytes) == hipSuccess) own_.push_back(p);
      return p;
    }
    if (bytes > left_) {
      int dev = 0;
      if (hipGetDevice(&dev) != hipSuccess) return nullptr;
      blocks_.reserve(blocks_.size() + 1);
      size_t size = next_;
      void* p = take_block(dev, size);
      if (!p && device_malloc(&p, size) != hipSuccess && device_malloc(&p, size = bytes) != hipSuccess)
        return nullptr; /* (the second: the last of the memory) */
      blocks_.push_back({dev, p, size});
      at_ = (char*)p;
      left_ = size;
      next_ = std::min(2 * next_, MOST);
    }
    void* const p = at_;
    at_ += bytes;
    left_ -= bytes;
    return p;
  }
  /* a piece that no queued work uses: an allocation of its own is freed, a
   * cut piece stays with its block */
  void release(void* p) {
    const auto it = std::find(own_.begin(), own_.end(), p);
    if (it == own_.end()) return;
    (void)hipFree(p);
    own_.erase(it);
  }
  bool is_own(const void* p) const { return std::find(own_.begin(), own_.end(), p) != own_.end(); }
  /* ended: the work that used the memory has, as far as the owner knows */
  void free(bool ended = true) {
    if (own_.empty() && blocks_.empty()) return;
    if (st_ && hipStreamSynchronize(st_) != hipSuccess) ended = false;
    for (void* p : own_) (void)hipFree(p);
    for (const Block& b : blocks_)
      if (!ended || b.bytes < OWN || !give_block(b)) (void)hipFree(b.p);
    own_.clear();
    blocks_.clear();
    at_ = nullptr;
    left_ = 0;
  }

 private:
  hipStream_t st_;
  std::vector<void*> own_;
  std::vector<Block> blocks_;
  char* at_ = nullptr;
  size_t left_ = 0, next_ = OWN;
};

}  // namespace kifmm_dev

#endif
