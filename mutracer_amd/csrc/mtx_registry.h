// Handle registry: uint64 handles (monotonic, never reused) to resident objects.
#pragma once
#include <atomic>
#include <memory>
#include <mutex>
#include <unordered_map>

#include "mtx_scene.h"

namespace mtx {

struct Context;
struct Server;

struct Registry {
  std::mutex m;
  std::atomic<uint64_t> nextHandle{1};
  std::unordered_map<uint64_t, std::shared_ptr<Blas>> blas;
  std::unordered_map<uint64_t, std::shared_ptr<Accel>> accel;
  std::unordered_map<uint64_t, std::shared_ptr<Context>> contexts;
  std::unordered_map<uint64_t, std::shared_ptr<Server>> servers;
  uint64_t next();
  std::shared_ptr<Blas> get_blas(uint64_t h) {
    std::lock_guard<std::mutex> g(m);
    auto it = blas.find(h);
    if (it == blas.end()) throw Error(MTX_INVALID_HANDLE, "unknown BLAS handle");
    return it->second;
  }
  std::shared_ptr<Accel> get_accel(uint64_t h) {
    std::lock_guard<std::mutex> g(m);
    auto it = accel.find(h);
    if (it == accel.end()) throw Error(MTX_INVALID_HANDLE, "unknown acceleration handle");
    return it->second;
  }
};

Registry &registry();
uint32_t trace_grid();

// The spill memory of a stream's traversal stacks (ptr), held while a render
// enqueues its launches: no other thread's launches on the stream grow (free)
// it in between. A render whose launches run on a stream of its own in place
// of the null stream (which cannot be recorded) calls enter() before them: the
// memory is the null stream's, and two such streams do not follow one another
// by themselves.
struct StreamScratch;
class SpillLease {
 public:
  SpillLease(hipStream_t s, uint32_t blocks, uint32_t blockThreads);
  void enter(const std::shared_ptr<OwnStream> &own);
  int32_t *ptr = nullptr;

 private:
  std::shared_ptr<StreamScratch> scratch;
  std::unique_lock<std::mutex> lock;
};

}  // namespace mtx
