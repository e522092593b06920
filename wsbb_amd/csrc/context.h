// Library-private state behind the wsbb_ctx handle.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/wsbb_amd.h"
#include "device.h"
#include "instance.h"

struct wsbb_ctx;

namespace wsbb {

void set_error(const std::string& msg);
int hip_fail(hipError_t e, const char* what);

// Grow-only device buffer owned by a context.
struct DevBuf {
  void* ptr = nullptr;
  size_t bytes = 0;
  hipError_t reserve(size_t need) {
    if (need <= bytes) return hipSuccess;
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
    hipError_t e = hipMalloc(&ptr, need);
    if (e == hipSuccess) bytes = need;
    return e;
  }
  void release() {
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
  }
  template <class T>
  T* as(size_t byte_offset = 0) const {
    return reinterpret_cast<T*>(static_cast<char*>(ptr) + byte_offset);
  }
};

// Pinned host memory that kernels read and write in place.
struct HostBuf {
  char* ptr = nullptr;  // as the host sees it
  char* dev = nullptr;  // as kernels do
  size_t bytes = 0;
  // false: no pinned memory to be had (the caller stages by copies)
  bool reserve(size_t need) {
    if (need <= bytes) return true;
    release();
    void *h = nullptr, *d = nullptr;
    if (hipHostMalloc(&h, need, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    if (hipHostGetDevicePointer(&d, h, 0) != hipSuccess) {
      (void)hipGetLastError();
      (void)hipHostFree(h);
      return false;
    }
    ptr = static_cast<char*>(h);
    dev = static_cast<char*>(d);
    bytes = need;
    return true;
  }
  void release() {
    if (ptr) (void)hipHostFree(ptr);
    ptr = dev = nullptr;
    bytes = 0;
  }
};

struct SearchState;    // search.hip
struct SelectorState;  // selector.hip

struct Launch {
  int groups = 1;
  int grid_cap = 0;  // 0: automatic
  int int16 = 1;     // two nodes per lane in int16 halves: 0 never, 1 for
                     // large batches, 2 whenever the instance fits
};

}  // namespace wsbb

struct wsbb_ctx {
  int device = 0;
  int num_cus = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev_start = nullptr, ev_stop = nullptr;
  wsbb::Instance inst;
  wsbb::DevTables T{};
  wsbb::DevBuf tables;  // every instance table in one allocation
  wsbb::DevBuf batch;   // staging for host-buffer batch calls
  wsbb::HostBuf pinned; // and for small ones while another call holds the device's
  wsbb::Launch launch;
  int pool_capacity = 1 << 24;  // device node-pool capacity (nodes)
  int profile_every = 0;         // time every k-th round's bound launch in wsbb_solve
  bool search_graph = false;     // replay search rounds from a captured hipGraph
  int rounds_per_sync = 4;       // rounds queued between host status checks
  wsbb_trace_fn trace_fn = nullptr;  // per-round search trace (one round per sync)
  void* trace_user = nullptr;
  // autotuned shapes by batch size class (log2 of tiles), -1 = not tuned: of
  // the scans, and of the matrix-core form
  int tuned_groups[32], tuned_waves[32];
  wsbb::SearchState* search = nullptr;
  wsbb::SelectorState* selector = nullptr;

  int grid_cap() const {
    if (launch.grid_cap > 0) return launch.grid_cap;
    return num_cus * 16;  // 16 blocks per CU: a 2^20-node batch, one per four tiles
  }
  int groups_for(int N) const;
  // a caller who asks for the int16 form gets it
  int mfma_for() const { return T.mf != nullptr && launch.int16 != 2; }
  // A large batch of few pairs is nearly all heads and tails, which the scans
  // run with less work (from 2^18 nodes on two nodes a lane), while a pair
  // costs the matrix cores whole tiles: the scans are faster where pairs x
  // jobs is small against the jobs that the tiles leave empty, counted from
  // the sizes at which they stop to be (20 and 29 of one row tile, 56 of two,
  // 116 of three; 230 at 95 and 96 jobs, whose fourth column block costs the
  // kernel a wave per SIMD).  With more than 96 jobs a block's four waves
  // share heads and tails, and the matrix cores win.  us, scan / matrix cores:
  // 2^20 nodes, 11 jobs 3 machines 33 / 41, 5 machines 44 / 47, 6 machines 52 /
  // 52; 33 jobs 4 machines 105 / 123, 6 machines 146 / 143; 65 jobs 5 machines
  // 290 / 321, 6 machines 355 / 347; 90 jobs 3 machines 294 / 347, 5 machines
  // 421 / 380; 96 jobs 5 machines 446 / 556; 100 jobs 3 machines 389 / 361.
  // 300 000 nodes, 11 jobs 3 machines 17 / 18, 4 machines 19 / 19; 65 jobs 3
  // machines 90 / 93, 5 machines 130 / 104.  131 072 nodes, 11 jobs 3 machines
  // 10.1 / 10.4, 96 jobs 5 machines 73 / 78.  65 536 nodes, 8 jobs 3 machines
  // 7.4 / 8.1, 33 jobs 3 machines 16 / 12, 96 jobs 3 machines 41 / 40.
  bool few_pairs(int N) const {
    const int n = T.n, P = T.P, simds = 4 * num_cus;
    if (n > 96) return false;
    const int empty = (n <= 20 ? 20 : n <= 32 ? 29 : n <= 64 ? 56 : n <= 94 ? 116 : 230) - n;
    if (N >= 256 * simds) {
      if (T.steps16 == nullptr || !int16_for(N)) return false;
      return N >= 512 * simds ? P <= 28 && P * n < 14 * empty : 2 * P * n <= 9 * empty;
    }
    return N >= (n <= 10 ? 48 : 96) * simds && (n > 94 ? P <= 10 : P <= 3 && 2 * P * n <= 9 * empty);
  }
  static int size_class(int N) {
    const int tiles = (N + 63) / 64;
    int cls = 0;
    while ((1 << (cls + 1)) <= tiles && cls < 31) ++cls;
    return cls;
  }
  // the split a caller asked for, or the launch's own
  void johnson_args(wsbb::BoundArgs& A) const {
    A.mfma = mfma_for();
    A.num_cus = num_cus;
    A.waves = launch.groups > 1 ? launch.groups : 0;
  }
  // the same for a batch of A.N nodes, with the tuned split of its size.  A
  // search round is not one: A.N is its capacity, and its live children,
  // often far fewer, are not the batch that was tuned.
  void johnson_batch_args(wsbb::BoundArgs& A) const {
    johnson_args(A);
    A.mfma = A.mfma && !few_pairs(A.N);
    const int tuned = tuned_waves[size_class(A.N)];
    if (A.waves == 0 && tuned > 0) A.waves = tuned;
  }
  // two nodes per lane pays once a batch gives every SIMD two 128-node tiles;
  // smaller launches are latency-bound and prefer more wavefronts
  int int16_for(long long N) const {
    if (launch.int16 == 2) return 1;
    return launch.int16 == 1 && N >= 2LL * 128 * 4 * num_cus;
  }
};
