// LB2 on the matrix cores (johnson.hip): operands and launchers.
#pragma once
#include <algorithm>

#include "device.h"

namespace wsbb {

// x_k = lag + p_a is split as lo + kXBase hi, both in a signed byte
constexpr int kXBase = 127;
// 32-wide column blocks of n jobs and the two constants
__host__ __device__ inline int column_blocks(int n) { return (n + 33) >> 5; }
// register arrays over machines: 8, 12, 16, 20 or 24
inline int padded_machines(int m) { return m <= 8 ? 8 : (m + 3) & ~3; }
constexpr int kXMax = kXBase * kXBase + kXBase - 1;

// Couples of pairs of m machines (k_johnson walks two pairs of one first
// machine at a time): machine a has ceil((m - 1 - a) / 2).
__host__ __device__ inline int johnson_first_couple(int m, int a) {
  // sum over i < a of ceil((m - 1 - i) / 2)
  const int up = (m - 1 + 1) / 2, dn = (m - 1) / 2;  // of machines 0 and 1
  const int k = a >> 1;
  // two machines further each takes one couple less
  return k * (up + dn) - k * (k - 1) + ((a & 1) ? up - k : 0);
}
__host__ __device__ inline int johnson_couples(int m) { return johnson_first_couple(m, m - 1); }
// Entries of the pair table, with those that a wave may read past the last
// couple, and its bytes: one KiB per entry, 32 rows and 32 columns.
__host__ __device__ inline int johnson_entries(int m) { return 2 * (johnson_couples(m) + 4); }
inline size_t johnson_bytes(int n, int m) {
  return static_cast<size_t>(johnson_entries(m)) * ((n + 31) >> 5) * column_blocks(n) * 1024;
}
inline size_t johnson_time_bytes(int n) { return static_cast<size_t>(column_blocks(n)) * 1024; }

// How a launch is laid out over waves and LDS (set by the launcher).
struct JohnsonShape {
  int rts;         // 32-row tiles of a pair
  int groups;      // waves that split the pairs of one tile and row tile
  int tpb;         // tiles per block
  int tile_bytes;  // LDS of one tile
  int first_block; // of this launch
  int list_rows;   // 64-word rows of a tile's pair list
  int wide;        // tiles of 128 nodes, not 64
  const int* list; // the children to bound, or null: all of them
};

// The layout for N nodes; waves: ways to split the pairs, or 0 (chosen).
JohnsonShape johnson_shape(int n, int P, int N, int waves, bool subset, int num_cus);
inline int johnson_block_nodes(const JohnsonShape& H) { return (H.wide ? 128 : 64) * H.tpb; }
// How many of 1, 2 and 4 waves can split the pairs of one tile of n jobs.
inline int johnson_splits(int n) { return n <= 32 ? 3 : n <= 64 ? 2 : 1; }
// Instances of one class share a kernel: equal padded machines, row tiles and
// column blocks.
int johnson_class(int n, int m);

// Fills mf (johnson_bytes), pf (johnson_time_bytes) and pr (32 n bytes) from
// T's step table and times.
hipError_t build_johnson(const DevTables& T, int4* mf, int4* pf, int4* pr, hipStream_t stream);

// Plain LB2 of every node, or (children with tile_sel) LB2 over each tile's
// pairs.  Children need their parents' state.
hipError_t launch_johnson(const DevTables& T, const BatchSource& src, const BoundArgs& A,
                          int grid_cap, hipStream_t stream);
hipError_t launch_johnson(const DevTables& T, const ChildSource& src, const BoundArgs& A,
                          int grid_cap, hipStream_t stream);
// Nodes of several instances of one class; T: the class's largest n and P, A.N
// its nodes; every block holds at most johnson_block_nodes of one instance.
hipError_t launch_johnson(const DevTables& T, const MultiSource& src, const BoundArgs& A, int blocks,
                          int grid_cap, hipStream_t stream);
hipError_t launch_johnson(const DevTables& T, const ListSource& src, const BoundArgs& A,
                          int grid_cap, hipStream_t stream);

}  // namespace wsbb
