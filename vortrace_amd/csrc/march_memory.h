// Device memory of the march (march.h).  All of it is optional: without it every
// ray runs in the ray engine.  So it is taken only where there is room, and given
// back when an allocation that a call cannot do without fails.
//
//  * Lists and boxes (280 B per cell) belong to their cloud and are built by the
//    first calls that are worth it.
//  * Rows (up to 4.5 GiB while a call marches) belong to no cloud: a call leases a
//    block and returns it when it has been waited for.  One block per device is
//    kept between calls, until its last cloud goes.
//
// Calls on different clouds may run in several threads.  MarchMemory's lock
// guards the blocks at rest and the set of clouds with lists; a call marks its
// cloud's lists as in use, which keeps other threads from dropping them.
// (Included by vt_hip.hip alone, inside no namespace.)
#pragma once

namespace {

// Device memory that is free, for requests of `want` bytes; small ones need not
// ask.
size_t free_for(size_t want) {
  size_t avail = 0, total = 0;
  if (want < ((size_t)256 << 20)) return SIZE_MAX / 2;
  return hipMemGetInfo(&avail, &total) == hipSuccess ? avail : 0;
}

struct MarchLists {
  enum : int { kNone = 0, kIdle = 1, kUsed = 2 };
  std::atomic<int> state{kNone};
  void *p = nullptr;  // one allocation, which N points into
  size_t bytes = 0;
  vt::NbLists N{};
  bool ready() const { return state.load() != kNone; }
  // Lists stay for their cloud's life, so they may take half of what is free.
  bool alloc(size_t want) {
    if (p && bytes >= want) return true;  // (from a build that failed half way)
    if (p) (void)hipFree(p);
    bytes = 0;
    if (want > free_for(want) / 2 || hipMalloc(&p, want) != hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
      return false;
    }
    bytes = want;
    return true;
  }
  // Frees them unless a call uses them.  They count as used meanwhile, so that a
  // call of their cloud neither takes nor builds them.  (What a build that failed
  // half way left, its own cloud's calls alone free.)
  bool drop() {
    int was = kIdle;
    if (!state.compare_exchange_strong(was, kUsed) && was == kUsed) return false;
    const bool freed = p != nullptr;
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
    state.store(kNone);
    return freed;
  }
};

struct MarchMemory {
  struct Block {
    void *p = nullptr;
    size_t bytes = 0;
  };
  std::mutex mu;
  std::map<int, Block> rows;      // the block at rest, per device
  std::map<int, int> clouds;      // uploaded clouds, per device
  std::set<vt_cloud *> listed;    // clouds with lists
  bool drop_rows(int dev) {
    Block &b = rows[dev];
    if (!b.p) return false;
    (void)hipFree(b.p);
    b = Block{};
    return true;
  }
};

// (Never destroyed: nothing is freed after the HIP runtime has gone.)
MarchMemory &march_memory() {
  static MarchMemory *m = new MarchMemory;
  return *m;
}

void leave_march_memory(vt_cloud *c);

// A cloud's lists, for the time a call marches; empty when it has none.
struct ListLease {
  MarchLists &l;
  const bool held;
  ListLease(MarchLists &lists, bool wanted) : l(lists), held(wanted && take(lists)) {}
  ListLease(const ListLease &) = delete;
  ~ListLease() {
    if (held) l.state.store(MarchLists::kIdle);
  }
  explicit operator bool() const { return held; }
  static bool take(MarchLists &l) {
    int idle = MarchLists::kIdle;
    return l.state.compare_exchange_strong(idle, MarchLists::kUsed);
  }
};

// A call's block of rows.  A call that ends before idle() may still have work on
// its stream, which is waited for.
struct RowLease {
  hipStream_t st;
  int dev = -1;
  MarchMemory::Block b;
  bool busy = true;
  explicit RowLease(hipStream_t stream) : st(stream) {}
  RowLease(const RowLease &) = delete;
  void *data() const { return b.p; }
  size_t bytes() const { return b.bytes; }
  void idle() { busy = false; }
  // A block of `want` bytes, or of at least `least` where there is room for no
  // more (a quarter of what is free, so that a program's own allocations find
  // the rest).
  bool take(int device, size_t want, size_t least) {
    MarchMemory &m = march_memory();
    std::lock_guard<std::mutex> lk(m.mu);
    MarchMemory::Block &rest = m.rows[device];
    if (rest.bytes < want) {
      const size_t room = (free_for(want) + rest.bytes) / 4;
      size_t get = std::min(want, std::max(room, least));
      if (rest.bytes < least || get > rest.bytes + rest.bytes / 4) {
        (void)m.drop_rows(device);
        void *p = nullptr;
        while (hipMalloc(&p, get) != hipSuccess) {
          (void)hipGetLastError();
          p = nullptr;
          if (get == least) return false;
          get = std::max(least, get / 2);
        }
        rest = MarchMemory::Block{p, get};
      }
    }
    b = rest;
    rest = MarchMemory::Block{};
    dev = device;
    return true;
  }
  // Makes the block at least `want` bytes up to its `tail` of `size` bytes, whose
  // first `keep` are kept (it may move); false when there is no room.  The call
  // has been waited for.
  bool grow(size_t want, uint32_t *&tail, size_t size, size_t keep) {
    if ((size_t)(reinterpret_cast<char *>(tail) - static_cast<char *>(b.p)) >= want) return true;
    void *p = nullptr;
    if (want + size > free_for(want + size) / 4 || hipMalloc(&p, want + size) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    uint32_t *moved = reinterpret_cast<uint32_t *>(static_cast<char *>(p) + want);
    const bool ok = hipMemcpyAsync(moved, tail, keep, hipMemcpyDeviceToDevice, st) == hipSuccess &&
                    hipStreamSynchronize(st) == hipSuccess;
    if (!ok) {
      (void)hipGetLastError();
      (void)hipFree(p);
      return false;
    }
    (void)hipFree(b.p);
    b = MarchMemory::Block{p, want + size};
    tail = moved;
    return true;
  }
  ~RowLease() {
    if (!b.p) return;
    if (busy) (void)hipStreamSynchronize(st);
    MarchMemory &m = march_memory();
    std::lock_guard<std::mutex> lk(m.mu);
    MarchMemory::Block &rest = m.rows[dev];
    if (rest.bytes < b.bytes) std::swap(rest, b);
    if (b.p) (void)hipFree(b.p);
  }
};

}  // namespace
