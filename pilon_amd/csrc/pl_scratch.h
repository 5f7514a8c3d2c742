// pl_scratch.h — device memory of passes that need scratch for one call (VCF,
// tracks, K-mers, uploads), kept by the lane for its next call.  Mem allocates
// and frees it (device memory, or the CPU tests' own).
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <vector>

#define PL_SCRATCH_KEEP ((size_t)2 << 30)   // most a lane keeps between calls

template <class Mem> class Scratch;

// The lanes' scratch of the process.  What an idle lane keeps is given back
// when an allocation anywhere in the library finds no memory, so keeping it
// never makes a call fail.
template <class Mem> class ScratchRegistry {
 public:
  static ScratchRegistry& get() { static ScratchRegistry* r = new ScratchRegistry; return *r; }   // (outlives every lane)
  std::mutex mu;                        // of the list, and of which scratch is in use
  std::vector<Scratch<Mem>*> all;
  bool give_back() {
    std::lock_guard<std::mutex> lk(mu);
    bool any = false;
    for (Scratch<Mem>* s : all)
      if (!s->top && !s->blocks.empty()) { s->release(); any = true; }
    return any;
  }
};

// Mem::alloc, a second time once idle scratch has been given back
template <class Mem> bool alloc_or_give_back(void** p, size_t n) {
  return Mem::alloc(p, n) || (ScratchRegistry<Mem>::get().give_back() && Mem::alloc(p, n));
}

// Blocks handed out by bumping an offset and taken back when the call ends
// (ScratchCall), kept up to PL_SCRATCH_KEEP.  A call's hipMalloc and hipFree
// of its dozen buffers took longer than its kernels on small batches.
template <class Mem> class Scratch {
 public:
  Scratch() {
    std::lock_guard<std::mutex> lk(reg().mu);
    reg().all.push_back(this);
  }
  ~Scratch() {
    std::lock_guard<std::mutex> lk(reg().mu);
    release();
    reg().all.erase(std::find(reg().all.begin(), reg().all.end(), this));
  }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  // gives the blocks back now (the lane ends)
  void drop() {
    std::lock_guard<std::mutex> lk(reg().mu);
    release();
  }

 private:
  template <class M> friend class ScratchRegistry;
  template <class M> friend class ScratchCall;
  struct Block { uint8_t* p; size_t n; bool held; };   // held: part of it is handed out
  std::vector<Block> blocks;
  size_t at = 0, used = 0;         // the block in use and how much of it
  size_t want = 0;                 // size of the next first block
  void* top = nullptr;             // the innermost ScratchCall alive
  static ScratchRegistry<Mem>& reg() { return ScratchRegistry<Mem>::get(); }

  bool take(size_t bytes, void** out) {
    bytes = (std::max<size_t>(bytes, 1) + 255) & ~(size_t)255;
    while (at < blocks.size() && bytes > blocks[at].n - used) { at++; used = 0; }
    if (at == blocks.size()) {
      Block b{nullptr, std::max(bytes, blocks.empty() && want ? want : (size_t)1 << 20), false};
      if (!Mem::alloc((void**)&b.p, b.n)) {
        // blocks that were too small for this call, then idle lanes' scratch
        for (Block& x : blocks)
          if (!x.held && x.p) { Mem::free(x.p); x.p = nullptr; x.n = 0; }
        b.n = bytes;
        if (!alloc_or_give_back<Mem>((void**)&b.p, b.n)) return false;
      }
      blocks.push_back(b);
      used = 0;
    }
    *out = blocks[at].p + used;
    blocks[at].held = true;
    used += bytes;
    return true;
  }
  void back_to(size_t a, size_t u) {
    at = a;
    used = u;
    for (size_t k = u ? a + 1 : a; k < blocks.size(); k++) blocks[k].held = false;
  }
  void release() {
    for (Block& b : blocks) if (b.p) Mem::free(b.p);
    blocks.clear();
    at = used = 0;
  }
  // nothing in use any more: many blocks become one next time, and none is
  // kept above the bound
  void settle() {
    size_t t = 0;
    for (const Block& b : blocks) t += b.n;
    at = used = 0;
    blocks.erase(std::remove_if(blocks.begin(), blocks.end(), [](const Block& b) { return !b.p; }), blocks.end());
    if (t > PL_SCRATCH_KEEP) { want = 0; release(); }
    else if (blocks.size() > 16) { want = t; release(); }
  }
};

// Device buffers of one call, given back on every exit: to the lane's
// scratch (calls nest, so the last one begun is the first to end), or freed
// when they were allocated while a call begun later was still using it.
template <class Mem> class ScratchCall {
 public:
  explicit ScratchCall(Scratch<Mem>& scratch) : s(scratch) {
    std::lock_guard<std::mutex> lk(s.reg().mu);
    at = s.at;
    used = s.used;
    outer = s.top;
    s.top = this;
  }
  ~ScratchCall() {
    for (void* x : own) Mem::free(x);
    std::lock_guard<std::mutex> lk(s.reg().mu);
    s.top = outer;
    s.back_to(at, used);
    if (!outer) s.settle();
  }
  ScratchCall(const ScratchCall&) = delete;
  ScratchCall& operator=(const ScratchCall&) = delete;
  bool take(size_t n, void** out) {
    if (s.top == this) return s.take(n, out);
    if (!alloc_or_give_back<Mem>(out, n ? n : 1)) return false;
    own.push_back(*out);
    return true;
  }

 private:
  Scratch<Mem>& s;
  size_t at, used;
  void* outer;
  std::vector<void*> own;
};
