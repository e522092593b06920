// The Johnson two-machine bound LB2 on the matrix cores.
//
// For a machine pair (a, b) and a node with free jobs F, the scan of
// heuristiqueCmax (bound_flowshop.cpp:64-77) is a maximum over the free jobs:
// with d_j = p_a(j) - p_b(j), x_j = lag(j) + p_a(j) and "before" the pair's
// Johnson order,
//   t1 = rem(b) + max(start(b), start(a) + max_{k in F} Z_k),
//   Z_k = x_k + sum over j in F before k of d_j.
// Z is linear in the node's 0/1 vector of free jobs, so all rows k of a pair
// for 32 nodes are one matrix product: rows are jobs (in job order, whatever
// the pair's Johnson order), columns are nodes, and the accumulator starts at
// 0 for a free job's row and at -2^28 for a scheduled one's, which takes the
// row out of the maximum.  The two columns after the last job hold x_k as
// x_k = lo + 127 hi against the constants 1 and 127.  Every operand is a
// whole number in eight bits and every sum is exact in 32, as the scan's.
//
// The rest of a pair is a maximum over the 16 rows a lane holds, one
// three-way add and a maximum; the terms start(b) + rem(b) + tail(b) and the
// one-machine terms start(a) + rem(a) + tail(a) of cmaxFin (92-100, 146-148)
// do not depend on the pair and are taken once per node.  The remaining work
// rem(k) of every machine is one more product with the same right operand.
#include "johnson.h"

#include <hip/hip_ext.h>

#include <type_traits>

namespace wsbb {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// bytes of a job's row of times: one per machine, padded to 16
__host__ __device__ constexpr int row_bytes(int m) { return m <= 16 ? 16 : 32; }
constexpr int kOut = -(1 << 28);  // a scheduled job's row

__device__ __forceinline__ v16i mfma_i8(v4i a, v4i b, v16i c) {
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// the largest of the first NR rows a lane holds
template <int NR>
__device__ __forceinline__ int max_rows(const v16i& z) {
  int t = z[0];
#pragma unroll
  for (int i = 1; i + 1 < NR; i += 2) t = max(max(t, z[i]), z[i + 1]);
  return NR & 1 ? t : max(t, z[NR - 1]);
}

// Rows to jobs: a pair's n jobs are split evenly over its row tiles and a
// tile's over the two lane halves, so that every lane's rows are its first
// few registers: register i of half h in tile rt is row 8 (i / 4) + 4 h +
// i % 4 of the product and job rt jobs + h per + i.
struct RowMap {
  int jobs, per;
  __device__ __host__ RowMap(int n, int rts)
      : jobs((n + rts - 1) / rts), per((jobs + 1) / 2) {}
  // the job of register i, half h, or -1
  __device__ __forceinline__ int job(int rt, int h, int i, int n) const {
    const int j = h * per + i;
    return i < per && j < jobs && rt * jobs + j < n ? rt * jobs + j : -1;
  }
};

// Pairs are walked in couples (a, b), (a, b + 1) of one machine a, in
// lexicographic order; the last couple of a machine with an odd number of
// pairs holds its last pair twice, which changes no maximum.
__device__ __forceinline__ void next_couple(int m, int& a, int& b) {
  b += 2;
  if (b >= m) {
    a = min(a + 1, m - 2);
    b = a + 1;
  }
}

// ---- the instance's operands, built once per context ----------------------
// Fragment
// (s, rt, kb): lane h * 32 + r holds columns 32 kb + 16 h .. + 15 of row r
// of row tile rt, one byte each.
__global__ __launch_bounds__(256) void k_johnson_tables(DevTables T, int4* mf, int4* pf,
                                                             int4* pr) {
  __shared__ int s_pos[kMaxJobs], s_d[kMaxJobs], s_x[kMaxJobs];
  // block 0: the times; then one block per entry of the pair table
  const int n = T.n, m = T.m, at_s = static_cast<int>(blockIdx.x) - 1;
  // entry 2 d + i holds pair (a, b + i) of couple d = (a, b), or the pair
  // before it again where b + i = m; entries past the last couple repeat it
  int s = 0;
  {
    int a = 0, b = 1;
    for (int d = 0; d < at_s >> 1; ++d) next_couple(m, a, b);
    b = min(b + (at_s & 1), m - 1);
    s = a * m - a * (a + 1) / 2 + b - a - 1;
  }
  const int rts = (n + 31) >> 5, kbs = column_blocks(n);
  const RowMap rm(n, rts);
  if (at_s < 0) {
    for (int u = threadIdx.x; u < kbs * 64; u += blockDim.x) {
      const int kb = u >> 6, k = u & 31, c0 = 32 * kb + 16 * ((u >> 5) & 1);
      uint32_t w[4] = {0u, 0u, 0u, 0u};
      for (int i = 0; i < 16; ++i)
        if (c0 + i < n && k < m)
          w[i >> 2] |= static_cast<uint32_t>(T.p[k * n + c0 + i]) << (8 * (i & 3));
      pf[u] = make_int4(w[0], w[1], w[2], w[3]);
    }
    // job-major rows of 16 or 32 bytes
    const int rs = row_bytes(m);
    for (int u = threadIdx.x; u < n * rs / 16; u += blockDim.x) {
      const int j = 16 * u / rs, k0 = 16 * u % rs;
      uint32_t w[4] = {0u, 0u, 0u, 0u};
      for (int i = 0; i < 16; ++i)
        if (k0 + i < m)
          w[i >> 2] |= static_cast<uint32_t>(T.p[(k0 + i) * n + j]) << (8 * (i & 3));
      pr[u] = make_int4(w[0], w[1], w[2], w[3]);
    }
    return;
  }
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const int4 st = T.steps[static_cast<size_t>(s) * T.n4 + k];
    s_pos[st.x] = k;
    s_d[st.x] = st.y - st.z;
    s_x[st.x] = st.w - kBias - st.z + st.y;  // lag + p_a
  }
  __syncthreads();
  for (int u = threadIdx.x; u < rts * kbs * 64; u += blockDim.x) {
    const int lane = u & 63, kb = (u >> 6) % kbs, rt = (u >> 6) / kbs;
    const int row = lane & 31, c0 = 32 * kb + 16 * (lane >> 5);
    const int r = rm.job(rt, (row >> 2) & 1, 4 * (row >> 3) + (row & 3), n);
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    if (r >= 0)
      for (int i = 0; i < 16; ++i) {
        const int c = c0 + i;
        int v = 0;
        if (c < n) v = s_pos[c] < s_pos[r] ? s_d[c] : 0;
        else if (c == n) v = s_x[r] % kXBase;
        else if (c == n + 1) v = s_x[r] / kXBase;
        w[i >> 2] |= static_cast<uint32_t>(v & 0xff) << (8 * (i & 3));
      }
    mf[static_cast<size_t>(at_s) * rts * kbs * 64 + u] = make_int4(w[0], w[1], w[2], w[3]);
  }
}

// ---- heads and tails -------------------------------------------------------
// a job's times in LDS, one byte per machine (every time is at most 127):
// rows of 16 or 32 bytes, machines m.. zero
template <int MM>
__device__ __forceinline__ void byte_row(const uint8_t* rows, int j, int (&pk)[MM]) {
  constexpr int RS = row_bytes(MM);
  const uint32_t* q = reinterpret_cast<const uint32_t*>(rows + j * RS);
  uint32_t w[MM / 4];
#pragma unroll
  for (int i = 0; i < MM / 4; ++i) w[i] = q[i];
#pragma unroll
  for (int k = 0; k < MM; ++k) pk[k] = (w[k >> 2] >> (8 * (k & 3))) & 0xff;
}

// the jobs a prefix or suffix holds, W words of 32
template <int W>
struct JobSet {
  unsigned long long lo = 0, hi = 0;
  __device__ __forceinline__ void add(int j) {
    if constexpr (W == 1) {
      lo |= 1u << j;
    } else if constexpr (W == 2) {
      lo |= 1ull << j;
    } else {
      const unsigned long long b = 1ull << (j & 63);
      lo |= j < 64 ? b : 0ull;
      hi |= j < 64 ? 0ull : b;
    }
  }
  __device__ __forceinline__ uint32_t word(int w) const {
    return static_cast<uint32_t>((w < 2 ? lo : hi) >> (32 * (w & 1)));
  }
};

// exclusive sums of 128 LDS counters by one wave, in place
__device__ __forceinline__ void wave_exscan128(int* h) {
  const int lane = threadIdx.x & 63;
  const int a = h[2 * lane], b = h[2 * lane + 1];
  int t = a + b;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(t, d, 64);
    if (lane >= d) t += u;
  }
  h[2 * lane] = t - a - b;
  h[2 * lane + 1] = t - b;
}

// the child at place k: all of them, or the listed ones
__device__ __forceinline__ int index_of(const JohnsonShape& H, int k, int count) {
  k = min(k, count - 1);
  return H.list ? H.list[k] : k;
}

// LDS of a block, in bytes from the start: the tiles, what the waves of a
// tile combine, the sort, the times
struct Layout {
  int comb, sort, rows, total;
  __host__ __device__ Layout(int tpb, int tile_bytes, int waves, int nodes, int n, int rs) {
    comb = tpb * tile_bytes;
    sort = comb + waves * (nodes / tpb) * 4;
    rows = sort + (tpb > 1 ? 2 * 128 * 4 + 6 * nodes : 0);
    total = rows + n * rs;
  }
};

// ---- the bound -------------------------------------------------------------
// A tile is NB operands of 32 nodes.  Its W = rts * G waves split the row
// tiles (32 jobs each) and, G ways, the pairs; tpb tiles make a block.  Each
// wave loads its pairs' fragments itself, AHEAD pairs ahead, and there is no
// barrier in the pair loop.
//
// Heads and tails come first, one lane per node and direction, in runs of 64
// nodes.  A wave runs as many steps as its longest prefix, so a block of
// several tiles sorts its nodes by prefix and by suffix length and deals the
// sorted runs to the waves, long runs with short ones.
//
// SUBSET: each tile (of 64 nodes) walks its own pairs.
template <int MM, int KB, int NR, int NB, bool SUBSET, class Src>
__global__ __launch_bounds__(256, (NB == 2 && KB <= 2 ? 3 : 2)) void k_johnson(DevTables T0, Src src,
                                                                              BoundArgs A,
                                                                              JohnsonShape H) {
  extern __shared__ char lds[];
  constexpr int rs = row_bytes(MM);
  constexpr int TN = 32 * NB;      // nodes of a tile
  constexpr int RUNS = NB / 2;     // runs of 64 nodes in a tile, each way
  constexpr bool MULTI = std::is_same<Src, MultiSource>::value;
  const int bt = H.first_block + blockIdx.x;
  // the block's instance and nodes: all of the launch's, or its own
  int first = bt * (TN * H.tpb), N = 0;
  DevTables T = T0;
  if constexpr (MULTI) {
    const int* b = reinterpret_cast<const int*>(src.blocks + bt);
    T = tables_at(src.tabs, ld_const(b, 0));
    first = ld_const(b, 1);
    N = first + ld_const(b, 2);
  } else {
    N = (A.Ndev != nullptr) ? *A.Ndev : A.N;
  }
  const int n = T.n, m = T.m;
  const int rts = H.rts, G = H.groups, W = rts * G;
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int tib = wave / W, wi = wave - tib * W;
  const int g = wi / rts, rt = wi - g * rts;
  const int tpb = H.tpb, nodes = TN * tpb;
  const int col = lane & 31, half = lane >> 5;
  const Layout L(tpb, H.tile_bytes, waves, nodes, n, rs);
  // a tile: st [MM][TN] and ew [MM][TN] (before them, in their place, the
  // permutations [n][TN]), prefix and suffix jobs [2][rts][TN]
  const int sm_at = H.tile_bytes - 2 * rts * TN * 4;
  char* mine = lds + tib * H.tile_bytes;
  int* comb = reinterpret_cast<int*>(lds + L.comb);                // [waves][TN]
  int* hist = reinterpret_cast<int*>(lds + L.sort);                // [2][128]
  uint16_t* lens = reinterpret_cast<uint16_t*>(hist + 256);        // [nodes] d1 | d2 << 8
  uint16_t* order = lens + nodes;                                  // [2][nodes]
  uint8_t* rows = reinterpret_cast<uint8_t*>(lds + L.rows);        // [n][rs]

  const int node0 = first;                   // the block's first node
  const int tile0 = node0 + tib * TN;        // this wave's tile's
  // a child's descriptor is read at any index below the capacity while the
  // live count is on its way; past the count it is read again in range
  int key[RUNS] = {};
  if constexpr (Src::kState)
    if (!H.list)
#pragma unroll
      for (int r = 0; r < RUNS; ++r) key[r] = src.key(min(tile0 + 64 * r + lane, A.N - 1));
  if (node0 >= N) return;
  if constexpr (Src::kState)
#pragma unroll
    for (int r = 0; r < RUNS; ++r)
      if (H.list || tile0 + 64 * r + lane >= N) key[r] = src.key(index_of(H, tile0 + 64 * r + lane, N));

  for (int i = threadIdx.x; i < n * rs / 16; i += blockDim.x)
    reinterpret_cast<int4*>(rows)[i] = T.pr[i];

  // lane l answers for nodes tile0 + 64 r + l
  int l1[RUNS], l2[RUNS];
  bool live[RUNS];
#pragma unroll
  for (int r = 0; r < RUNS; ++r) {
    l1[r] = -1;
    l2[r] = n;
    live[r] = tile0 + 64 * r + lane < N;
  }
  // the wave's runs of prefixes and of suffixes (none: -1); run q covers 64
  // of the block's nodes
  const int R = tpb * RUNS;
  int hp[RUNS], tp[RUNS];
#pragma unroll
  for (int r = 0; r < RUNS; ++r) {
    // R runs each way over the waves: two each way a wave (W < RUNS), one
    // each way, or the first R waves the prefixes and the next R the suffixes
    const int at = r ? 2 * waves - 1 - wave : wave;
    hp[r] = at < R ? at : -1;
    const int back = waves >= 2 * R ? at - R : at;
    tp[r] = back >= 0 && back < R ? R - 1 - back : -1;
  }
  int x[RUNS][MM], y[RUNS][MM], hn[RUNS] = {}, tn[RUNS] = {}, hl[RUNS] = {}, tl[RUNS] = {};
  JobSet<KB> hs[RUNS], ts[RUNS];
  bool h_leaf[RUNS] = {}, t_leaf[RUNS] = {};
  const bool sorted = !Src::kState && tpb > 1;
  Child hc[RUNS], tc[RUNS];
  if constexpr (Src::kState) {
    // every load that hangs on the descriptors before the barrier
#pragma unroll
    for (int r = 0; r < RUNS; ++r) src.limits(key[r], l1[r], l2[r]);
#pragma unroll
    for (int r = 0; r < RUNS; ++r) {
      if (hp[r] >= 0) {
        hn[r] = 64 * hp[r] + lane;
        hc[r] = src.child(src.key(index_of(H, node0 + hn[r], N)));
        src.template load_heads<MM>(hc[r], x[r], hs[r], rts);
      }
      if (tp[r] >= 0) {
        tn[r] = 64 * tp[r] + lane;
        tc[r] = src.child(src.key(index_of(H, node0 + tn[r], N)));
        src.template load_tails<MM>(tc[r], y[r]);
      }
    }
  } else {
    if (sorted)
      for (int i = threadIdx.x; i < 256; i += blockDim.x) hist[i] = 0;
#pragma unroll
    for (int r = 0; r < RUNS; ++r) {
      const int node = tile0 + 64 * r + lane;
      if (node < N) {
        const uint8_t* colp = nullptr;
        int stride = 0, sw0, sw1, a1, a2;
        (void)src.load(node, a1, a2, colp, stride, sw0, sw1);
        l1[r] = a1;
        l2[r] = a2;
        uint8_t* pl = reinterpret_cast<uint8_t*>(mine) + 64 * r + lane;
        // the tile's waves share its columns, sixteen positions at a time
        for (int i0 = 16 * wi; i0 < n; i0 += 16 * W) {
          uint32_t v[16];
#pragma unroll
          for (int u = 0; u < 16; ++u)
            if (i0 + u < n) v[u] = colp[static_cast<size_t>(i0 + u) * stride];
#pragma unroll
          for (int u = 0; u < 16; ++u)
            if (i0 + u < n) pl[(i0 + u) * TN] = static_cast<uint8_t>(v[u]);
        }
        if (!limits_ok(a1, a2, n)) {
          live[r] = false;
          l1[r] = -1;
          l2[r] = n;
        }
      }
    }
  }
  __syncthreads();  // permutations and times are staged
  if (sorted) {
    // counting sorts of the block's nodes by d1 and by d2
    int r1[RUNS] = {}, r2[RUNS] = {};
    if (wi == 0)
#pragma unroll
      for (int r = 0; r < RUNS; ++r) {
        const int d1 = l1[r] + 1, d2 = n - l2[r];
        lens[tib * TN + 64 * r + lane] = static_cast<uint16_t>(d1 | (d2 << 8));
        r1[r] = atomicAdd(&hist[d1], 1);
        r2[r] = atomicAdd(&hist[128 + d2], 1);
      }
    __syncthreads();
    if (wave < 2) wave_exscan128(hist + 128 * wave);
    __syncthreads();
    if (wi == 0)
#pragma unroll
      for (int r = 0; r < RUNS; ++r) {
        const uint16_t me = static_cast<uint16_t>(tib * TN + 64 * r + lane);
        order[hist[l1[r] + 1] + r1[r]] = me;
        order[nodes + hist[128 + n - l2[r]] + r2[r]] = me;
      }
    __syncthreads();
  }
  if constexpr (Src::kState) {
    // children: their parents' heads and tails extended by the jobs they place
    auto row = [&](int j, int(&pk)[MM]) { byte_row<MM>(rows, j, pk); };
#pragma unroll
    for (int r = 0; r < RUNS; ++r) {
      if (hp[r] >= 0) {
        hl[r] = hc[r].a + 1;
        h_leaf[r] = hc[r].b - hc[r].a == 1;
        src.template place_heads<MM>(hc[r], x[r], hs[r], row);
      }
      if (tp[r] >= 0) {
        tl[r] = n - tc[r].b;
        t_leaf[r] = tc[r].b - tc[r].a == 1;
        src.template place_tails<MM>(tc[r], y[r], row);
      }
    }
  } else {
    // the node at a run's place, its prefix and suffix lengths
    auto item = [&](int run, int which, int& place, bool& leaf) {
      int at = 64 * run + lane, d1, d2;
      if (sorted) {
        at = order[which * nodes + at];
        d1 = lens[at] & 255;
        d2 = lens[at] >> 8;
      } else {
        // one tile: the run's nodes are this lane's own
        d1 = l1[0] + 1;
        d2 = n - l2[0];
        if (RUNS > 1 && run > 0) {
          d1 = l1[RUNS - 1] + 1;
          d2 = n - l2[RUNS - 1];
        }
      }
      place = at;
      leaf = d1 + d2 == n;
      return which ? d2 : d1;
    };
    auto column = [&](int at) {
      return reinterpret_cast<const uint8_t*>(lds) + (at / TN) * H.tile_bytes + (at % TN);
    };
#pragma unroll
    for (int r = 0; r < RUNS; ++r) {
      if (hp[r] >= 0) {
        hl[r] = item(hp[r], 0, hn[r], h_leaf[r]);
        const uint8_t* c = column(hn[r]);
#pragma unroll
        for (int k = 0; k < MM; ++k) x[r][k] = 0;
        int jn = hl[r] > 0 ? c[0] : 0;
        for (int i = 0; i < hl[r]; ++i) {
          const int j = jn;
          if (i + 1 < hl[r]) jn = c[(i + 1) * TN];
          hs[r].add(j);
          int pk[MM];
          byte_row<MM>(rows, j, pk);
          head_step<MM>(x[r], pk);
        }
      }
      if (tp[r] >= 0) {
        tl[r] = item(tp[r], 1, tn[r], t_leaf[r]);
        const uint8_t* c = column(tn[r]);
#pragma unroll
        for (int k = 0; k < MM; ++k) y[r][k] = 0;
        int jn = tl[r] > 0 ? c[(n - 1) * TN] : 0;
        for (int i = 0; i < tl[r]; ++i) {
          const int j = jn;
          if (i + 1 < tl[r]) jn = c[(n - 2 - i) * TN];
          ts[r].add(j);
          int pk[MM];
          byte_row<MM>(rows, j, pk);
          tail_step<MM>(y[r], pk);
        }
      }
    }
    __syncthreads();  // every permutation is read: st and ew take their place
  }
  // start clocks (heads, or R0 without prefix) and tails (or Q0 without
  // suffix); a leaf keeps its plain heads and tails
#pragma unroll
  for (int r = 0; r < RUNS; ++r) {
    if (hp[r] >= 0) {
      char* t = lds + (hn[r] / TN) * H.tile_bytes;
      int* o = reinterpret_cast<int*>(t) + hn[r] % TN;
#pragma unroll
      for (int k = 0; k < MM; ++k)
        o[k * TN] = (hl[r] > 0 || h_leaf[r]) ? x[r][k] : ld_const(T.R0, k);
      uint32_t* w = reinterpret_cast<uint32_t*>(t + sm_at) + hn[r] % TN;
      for (int k = 0; k < rts; ++k) w[k * TN] = hs[r].word(k);
    }
    if (tp[r] >= 0) {
      char* t = lds + (tn[r] / TN) * H.tile_bytes;
      int* o = reinterpret_cast<int*>(t) + MM * TN + tn[r] % TN;
#pragma unroll
      for (int k = 0; k < MM; ++k)
        o[k * TN] = tl[r] > 0 ? y[r][k] : (t_leaf[r] ? 0 : ld_const(T.Q0, k));
      uint32_t* w = reinterpret_cast<uint32_t*>(t + sm_at) + rts * TN + tn[r] % TN;
      for (int k = 0; k < rts; ++k) w[k * TN] = ts[r].word(k);
    }
  }
  __syncthreads();

  // the pairs' fragments: the first ones are on their way while the operands
  // are put together
  const uint32_t lane16 = lane * 16;
  const int couples = johnson_couples(m);
  const int d_lo = (g * couples) / G;
  const int next = rts * KB * 1024;  // bytes from a pair's fragments to the next's
  constexpr int AHEAD = 2;
  const char* at = reinterpret_cast<const char*>(T.mf) +
                   (static_cast<size_t>(2 * d_lo) * rts + rt) * KB * 1024;
  v4i a[AHEAD][KB];
  auto fetch = [&](const char* from, v4i(&v)[KB]) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) v[kb] = *reinterpret_cast<const v4i*>(from + kb * 1024 + lane16);
  };
  if constexpr (!SUBSET) {
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) {
      fetch(at, a[q]);
      at += next;
    }
  }

  // operands of the tile's NB x 32 nodes: free jobs as bytes, and the
  // accumulators' start for this wave's 32 rows
  const int* st = reinterpret_cast<const int*>(mine);
  int* ew = reinterpret_cast<int*>(mine) + MM * TN;
  const uint32_t* sm = reinterpret_cast<const uint32_t*>(mine + sm_at);
  const RowMap rm(n, rts);
  uint32_t ones[KB][4];  // the constant columns
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c0 = n - 32 * kb - 16 * half - 4 * q;  // column n relative to this dword
      uint32_t v = 0;
      if (c0 >= 0 && c0 < 4) v |= 1u << (8 * c0);
      if (c0 >= -1 && c0 < 3) v |= static_cast<uint32_t>(kXBase) << (8 * (c0 + 1));
      ones[kb][q] = v;
    }
  v4i B[NB][KB];
  v16i C[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int own = 32 * c + col;
    unsigned long long fr[2] = {0ull, 0ull};  // free jobs
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      uint32_t w = 0;
      if (kb < rts) w = ~(sm[kb * TN + own] | sm[(rts + kb) * TN + own]);
      const int left = n - 32 * kb;  // jobs from this word on
      if (left < 32) w &= left > 0 ? (1u << left) - 1u : 0u;
      fr[kb >> 1] |= static_cast<unsigned long long>(w) << (32 * (kb & 1));
      const uint32_t bits = w >> (16 * half);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        B[c][kb][q] = static_cast<int>(
            (__umul24((bits >> (4 * q)) & 15u, 0x00204081u) & 0x01010101u) | ones[kb][q]);
    }
    // the lane's rows are consecutive jobs from j0; rows past its share of
    // the tile's jobs stay out
    const int j0 = rt * rm.jobs + half * rm.per;
    uint32_t w = 0;
    if (j0 < 64) w = static_cast<uint32_t>(fr[0] >> j0);
    if constexpr (KB > 2) {
      if (j0 >= 64) w = static_cast<uint32_t>(fr[1] >> (j0 - 64));
      else if (j0 > 32) w |= static_cast<uint32_t>(fr[1] << (64 - j0));
    }
    w &= (1u << (half ? rm.jobs - rm.per : rm.per)) - 1u;
#pragma unroll
    for (int r = 0; r < 16; ++r) C[c][r] = ((w >> r) & 1u) ? 0 : kOut;
  }
  // ew: tails + remaining work, one product per 32 nodes (machines as rows)
#pragma unroll
  for (int c = 0; c < NB; ++c)
    if (c % W == wi) {
      v16i z;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int k = 8 * (r >> 2) + 4 * half + (r & 3);
        z[r] = k < MM ? ew[k * TN + 32 * c + col] : 0;
      }
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        z = mfma_i8(reinterpret_cast<const v4i*>(T.pf)[kb * 64 + lane], B[c][kb], z);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int k = 8 * (r >> 2) + 4 * half + (r & 3);
        if (k < MM) ew[k * TN + 32 * c + col] = z[r];
      }
    }
  __syncthreads();

  int lb[NB] = {};
  const int* stc = st + col;
  const int* ewc = ew + col;
  if constexpr (SUBSET) {
    const int tile = min(bt * tpb + tib, (N - 1) / TN);
    const uint32_t* tsel = A.tile_sel + static_cast<size_t>(tile) * A.nsw;
    bool suf[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) suf[c] = __shfl(l2[c >> 1], 32 * (c & 1) + col, 64) < n;
    // the tile's pairs as a list in LDS, one word each: entry, first and
    // second machine (all waves of the tile write the same list)
    uint32_t* list = reinterpret_cast<uint32_t*>(lds + L.total) + tib * 64 * H.list_rows;
    int np = 0;
    for (int s0 = 0; s0 < T.P; s0 += 64) {
      const int s = s0 + lane;
      const bool take = s < T.P && ((tsel[s >> 5] >> (s & 31)) & 1u);
      const unsigned long long bal = __ballot(take);
      if (take) {
        const int2 ab = T.pairs[s];
        const int e = 2 * johnson_first_couple(m, ab.x) + ab.y - ab.x - 1;
        list[np + __popcll(bal & ((1ull << lane) - 1ull))] =
            static_cast<uint32_t>(e) | (ab.x << 16) | (ab.y << 24);
      }
      np += __popcll(bal);
    }
    np = __builtin_amdgcn_readfirstlane(np);
    if (np > 0) {
      // two pairs ahead (a rolled loop: unrolled, four pairs' products were
      // in registers at once and spilled)
      v4i f[3][KB];
      uint32_t w[3];
      auto ask = [&](int i, uint32_t& word, v4i(&v)[KB]) {
        word = __builtin_amdgcn_readfirstlane(list[min(i, np - 1)]);
        fetch(reinterpret_cast<const char*>(T.mf) +
                  (static_cast<size_t>(word & 0xffffu) * rts + rt) * KB * 1024,
              v);
      };
      ask(0, w[0], f[0]);
      ask(1, w[1], f[1]);
#pragma unroll 1
      for (int i = 0; i < np; ++i) {
        ask(i + 2, w[2], f[2]);
        const int xa = (w[0] >> 16) & 0xff, xb = w[0] >> 24;
        int sa[NB], sb[NB], ea[NB], eb[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          sa[c] = stc[xa * TN + 32 * c];
          sb[c] = stc[xb * TN + 32 * c];
          ea[c] = ewc[xa * TN + 32 * c];
          eb[c] = ewc[xb * TN + 32 * c];
        }
        v16i z[NB];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int c = 0; c < NB; ++c) z[c] = mfma_i8(f[0][kb], B[c][kb], kb == 0 ? C[c] : z[c]);
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          const int v = max(max_rows<NR>(z[c]) + sa[c], sb[c]) + eb[c];
          lb[c] = max(lb[c], max(v, suf[c] ? sa[c] + ea[c] : 0));
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          f[0][kb] = f[1][kb];
          f[1][kb] = f[2][kb];
        }
        w[0] = w[1];
        w[1] = w[2];
      }
    }
  } else {
    // row offsets of the couple's machines
    int ao = 0, bo = 1;
    for (int d = 0; d < d_lo; ++d) next_couple(m, ao, bo);
    ao *= TN;
    bo *= TN;
    const int b_end = m * TN;
    int la[NB];  // of machine a's pairs so far, without start(a)
#pragma unroll
    for (int c = 0; c < NB; ++c) la[c] = kOut;
    auto close = [&](int at_a) {
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        lb[c] = max(lb[c], la[c] + stc[at_a + 32 * c]);
        la[c] = kOut;
      }
    };
    // A step multiplies one pair with two of the operands while the rows of
    // the step before are reduced, so that neither unit waits for the other:
    // after each product a few of the maxima.
    constexpr int STEPS = NB;      // per couple: two pairs, NB / 2 steps each
    v16i z[2][2];
    int e[2][2], ends = -1;        // ends: the closed machine's row, or -1
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      e[1][c] = 0;
#pragma unroll
      for (int r = 0; r < 16; ++r) z[1][c][r] = kOut;
    }
    // rows [lo, hi) of the two running maxima
    auto reduce = [&](const v16i(&p)[2], int(&t)[2], int lo, int hi) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if (lo == 0) t[c] = p[c][0];
#pragma unroll
        for (int i = 1; i < NR; i += 2)
          if (i >= lo && i < hi)
            t[c] = i + 1 < NR ? max(max(t[c], p[c][i]), p[c][i + 1]) : max(t[c], p[c][i]);
      }
    };
    // a range may run one couple further, into the next range's pairs or the
    // repeated last one
    const int turns = (couples + G - 1) / G;
    for (int d = 0; d < turns; ++d) {
#pragma unroll
      for (int u = 0; u < STEPS; ++u) {
        constexpr int HALVES = NB / 2;
        const int q = u / HALVES, c0 = 2 * (u % HALVES);       // this step's pair, operands
        const int p0 = 2 * ((u + HALVES - 1) % HALVES);        // the step before's
        v16i(&zn)[2] = z[u & 1];
        const v16i(&zp)[2] = z[(u & 1) ^ 1];
        // tail terms of the couple's first and second pair
        const int* ep = ewc + (q ? min(bo + TN, b_end - TN) : bo);
#pragma unroll
        for (int c = 0; c < 2; ++c) e[u & 1][c] = ep[32 * (c0 + c)];
        int t[2];
        constexpr int PIECE = ((NR / 2 + 2 * KB - 1) / (2 * KB)) * 2;  // rows after each product
#pragma unroll
        for (int i = 0; i < 2 * KB; ++i) {
          const int c = i & 1, kb = i >> 1;
          zn[c] = mfma_i8(a[q][kb], B[c0 + c][kb], kb == 0 ? C[c0 + c] : zn[c]);
          __builtin_amdgcn_sched_barrier(0);
          reduce(zp, t, i * PIECE, i + 1 < 2 * KB ? (i + 1) * PIECE : 16);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) la[p0 + c] = max(la[p0 + c], t[c] + e[(u & 1) ^ 1][c]);
        if (u == 0 && ends >= 0) close(ends);
        if (c0 + 2 == NB) {
          fetch(at, a[q]);
          at += next;
        }
      }
      ends = -1;
      bo += 2 * TN;
      if (bo >= b_end) {  // machine a's last couple
        ends = ao;
        ao = min(ao + TN, b_end - 2 * TN);
        bo = ao + TN;
      }
    }
    // the last step, and the range's end (a machine may be closed here and
    // inside the loop: the last one's repeated pair)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      la[NB - 2 + c] = max(la[NB - 2 + c], max_rows<NR>(z[1][c]) + e[1][c]);
    close(ends >= 0 ? ends : ao);
  }
  // the two lane halves hold different rows of the same nodes
#pragma unroll
  for (int c = 0; c < NB; ++c) lb[c] = max(lb[c], __shfl_xor(lb[c], 32, 64));
#pragma unroll
  for (int r = 0; r < RUNS; ++r) {
    const int mine_l = 64 * r + lane, node = tile0 + mine_l;
    int res = half ? lb[2 * r + 1] : lb[2 * r];
    // start + remaining work + tail of every machine: what a pair (., b) is
    // at least, a leaf's makespan, and with a suffix the one-machine terms
    // (machine 0 is only ever a pair's first)
    const bool leaf = l2[r] - l1[r] == 1;
    int own = 0;
    for (int k = wi; k < m; k += W)
      if (k > 0 || l2[r] < n || leaf) own = max(own, st[k * TN + mine_l] + ew[k * TN + mine_l]);
    // a subset's maximum takes those terms from its own pairs only
    res = SUBSET ? (leaf ? own : res) : max(res, own);
    if (W > 1) {
      comb[wave * TN + mine_l] = res;
      __syncthreads();
      if (wi == 0)
        for (int k = 1; k < W; ++k) res = max(res, comb[(wave + k) * TN + mine_l]);
    }
    if (wi == 0 && live[r]) A.out[H.list ? H.list[node] : node] = res;
  }
}

template <int MM, int KB, int NR, int NB, bool SUBSET, class Src>
hipError_t launch_kernel(const DevTables& T, const Src& src, const BoundArgs& A, JohnsonShape H,
                         int blocks, int grid_cap, hipStream_t stream) {
  constexpr int rs = row_bytes(MM), TN = 32 * NB;
  const int waves = H.rts * H.groups * H.tpb;
  const int body = std::max(Src::kState ? 0 : T.n * TN, 2 * MM * TN * 4);
  H.tile_bytes = ((body + 15) & ~15) + 2 * H.rts * TN * 4;
  H.list_rows = (T.P + 63) / 64;
  const size_t shmem = Layout(H.tpb, H.tile_bytes, waves, TN * H.tpb, T.n, rs).total +
                       (SUBSET ? 256 * H.list_rows * H.tpb : 0);
  // a block bounds its tiles and ends (a loop over tiles kept the whole
  // prologue's constants in registers); more blocks than the cap run as
  // several launches
  for (H.first_block = 0; H.first_block < blocks; H.first_block += grid_cap) {
    const int grid = std::min(blocks - H.first_block, grid_cap);
    hipExtLaunchKernelGGL((k_johnson<MM, KB, NR, NB, SUBSET, Src>), dim3(grid), dim3(64 * waves), shmem,
                          stream, H.first_block == 0 ? A.ev_start : nullptr,
                          H.first_block + grid == blocks ? A.ev_stop : nullptr, 0, T, src, A, H);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// `blocks` > 0: the length of a MultiSource's list
template <int MM, class Src>
hipError_t launch_mm(const DevTables& T, const Src& src, const BoundArgs& A, JohnsonShape H,
                     int blocks, int grid_cap, hipStream_t stream) {
  const bool subset = A.tile_sel != nullptr;
  if (blocks == 0) {
    const int nodes = johnson_block_nodes(H);
    blocks = (A.N + nodes - 1) / nodes;
  }
  using std::integral_constant;
  auto rows = [&](auto kbv, auto nrv) {
    constexpr int KB = decltype(kbv)::value, NR = decltype(nrv)::value;
    if constexpr (std::is_same<Src, ChildSource>::value)
      if (subset)
        return launch_kernel<MM, KB, NR, 2, true, Src>(T, src, A, H, blocks, grid_cap, stream);
    if constexpr (KB >= 2)
      if (H.wide)
        return launch_kernel<MM, KB, NR, 4, false, Src>(T, src, A, H, blocks, grid_cap, stream);
    return launch_kernel<MM, KB, NR, 2, false, Src>(T, src, A, H, blocks, grid_cap, stream);
  };
  const bool few = RowMap(T.n, H.rts).per <= (column_blocks(T.n) == 1 ? 10 : 13);
  auto pick = [&](auto kbv) {
    constexpr int FEW = decltype(kbv)::value == 1 ? 10 : 13;
    return few ? rows(kbv, integral_constant<int, FEW>{}) : rows(kbv, integral_constant<int, 16>{});
  };
  switch (column_blocks(T.n)) {
    case 1: return pick(integral_constant<int, 1>{});
    case 2: return pick(integral_constant<int, 2>{});
    case 3: return pick(integral_constant<int, 3>{});
    case 4: return pick(integral_constant<int, 4>{});
    default: return hipErrorInvalidValue;
  }
}

template <class Src>
hipError_t launch_src(const DevTables& T, const Src& src, const BoundArgs& A, const int* list,
                      int blocks, int grid_cap, hipStream_t stream) {
  JohnsonShape H = johnson_shape(T.n, T.P, A.N, A.waves, A.tile_sel != nullptr, A.num_cus);
  H.list = list;
  switch (padded_machines(T.m)) {
    case 8: return launch_mm<8>(T, src, A, H, blocks, grid_cap, stream);
    case 12: return launch_mm<12>(T, src, A, H, blocks, grid_cap, stream);
    case 16: return launch_mm<16>(T, src, A, H, blocks, grid_cap, stream);
    case 20: return launch_mm<20>(T, src, A, H, blocks, grid_cap, stream);
    default: return launch_mm<24>(T, src, A, H, blocks, grid_cap, stream);
  }
}

}  // namespace

hipError_t build_johnson(const DevTables& T, int4* mf, int4* pf, int4* pr, hipStream_t stream) {
  hipLaunchKernelGGL(k_johnson_tables, dim3(1 + johnson_entries(T.m)), dim3(256), 0, stream, T, mf, pf, pr);
  return hipGetLastError();
}

JohnsonShape johnson_shape(int n, int P, int N, int waves, bool subset, int num_cus) {
  JohnsonShape H{};
  H.rts = (n + 31) >> 5;
  const int simds = 4 * num_cus, tiles = (N + 63) / 64;
  // The pairs are split over waves while that still adds waves to SIMDs that
  // have few, and where a tile's pairs outweigh the heads and tails that the
  // split leaves to one wave (us a launch, back to back, at G = 1 / 2 / 4: 20x20,
  // 50 000 nodes 34 / 27 / 25; 100 003 nodes 42 / 38 / 43; 300 000 nodes 89 / 89
  // / 111; 30x12, 100 000 nodes 24 / 29 / 35).
  H.groups = waves > 0                               ? waves
             : tiles * H.rts < simds                 ? 4
             : tiles * H.rts < 2 * simds && P >= 128 ? 2
                                                     : 1;
  H.groups = subset ? 1 : std::max(1, std::min(H.groups, 4 / H.rts));
  // Tiles of 128 nodes halve the fragments' way through the L1 and the scalar
  // work, for twice the registers: with two row tiles of jobs and more, from
  // two waves per SIMD on (us for 64 / 128 nodes, back to back: 50x20, 65 536
  // nodes 57 / 63; 90 000 nodes 73 / 88; 130 000 nodes 102 / 92; 2^20 nodes 670
  // / 623; 100x10, 50 000 nodes 70 / 52; 65 521 nodes 72 / 54).  With one row
  // tile a block holds four such tiles, whose start clocks and tails leave
  // room in LDS for one wave per SIMD: 300 000 nodes, 32x20 115 / 182, 32x5 30
  // / 40; 2^20 nodes, 32x20 332 / 485, 32x5 79 / 88 (at 262 017 nodes, whose
  // blocks just fill the chip, 32x5 is 28 / 25).  With three row tiles a block
  // is one tile of three waves, two of which run its prefixes and then its
  // suffixes while the third waits: 90 jobs, 131 072 nodes, 5 machines 56 / 72,
  // 20 machines 220 / 244; 2^20 nodes, 5 machines 380 / 520, 10 machines 600 /
  // 787 (95 and 96 jobs, whose fourth column block holds the constants, have
  // two waves per SIMD at 64 nodes too: 96 jobs, 2^20 nodes, 5 machines 629 /
  // 557, 10 machines 953 / 863).
  const bool third_idle = H.rts == 3 && column_blocks(n) == 3;
  H.wide = !subset && H.rts >= 2 && !third_idle && H.groups == 1 &&
           static_cast<long long>((N + 127) / 128) * H.rts >= 2 * simds;
  H.tpb = std::max(1, 4 / (H.rts * H.groups));
  return H;
}

int johnson_class(int n, int m) {
  const int rts = (n + 31) >> 5, kb = column_blocks(n);
  const bool few = RowMap(n, rts).per <= (kb == 1 ? 10 : 13);
  return ((padded_machines(m) * 8 + rts) * 8 + kb) * 2 + few;
}

hipError_t launch_johnson(const DevTables& T, const MultiSource& src, const BoundArgs& A, int blocks,
                          int grid_cap, hipStream_t stream) {
  if (A.tile_sel || blocks < 1) return hipErrorInvalidValue;
  return launch_src(T, src, A, nullptr, blocks, grid_cap, stream);
}

hipError_t launch_johnson(const DevTables& T, const BatchSource& src, const BoundArgs& A,
                          int grid_cap, hipStream_t stream) {
  if (A.tile_sel) return hipErrorInvalidValue;
  return launch_src(T, src, A, nullptr, 0, grid_cap, stream);
}
hipError_t launch_johnson(const DevTables& T, const ChildSource& src, const BoundArgs& A,
                          int grid_cap, hipStream_t stream) {
  return src.has_state() ? launch_src(T, src, A, nullptr, 0, grid_cap, stream) : hipErrorInvalidValue;
}
hipError_t launch_johnson(const DevTables& T, const ListSource& src, const BoundArgs& A,
                          int grid_cap, hipStream_t stream) {
  if (!src.has_state() || A.tile_sel) return hipErrorInvalidValue;
  return launch_src(T, src.base, A, src.list, 0, grid_cap, stream);
}

}  // namespace wsbb
