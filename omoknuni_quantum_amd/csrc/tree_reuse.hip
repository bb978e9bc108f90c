// Subtree reuse: a node of each tree becomes the root, and its subtree is compacted to the
// front of the tree (gfx950).
//
// Reference: CSRTree.shift_root (python/mcts/gpu/csr_tree.py:1020-1229), reached through
// TreeOperations.apply_subtree_reuse (python/mcts/core/tree_operations.py:53-133) from
// MCTS.update_root (python/mcts/core/mcts.py:1205-1245).
//   - The kept nodes are numbered breadth-first from the new root, children in row order.
//   - N, W and P of every kept node are copied, and parents are remapped; the new root has
//     parent -1 and action -1.
//   - Every other node is dropped, and the edge arrays are rebuilt in the new node order.
// With breadth-first numbering, the children of every kept node are again consecutive, and
// the edge of child c is c-1. The implicit-column layout of this library
// (child of edge e = node e+1) therefore holds after the shift as it held before.
//
// One workgroup per tree walks the subtree level by level. A level is a contiguous range of
// new ids. A block-wide scan of the level's row lengths gives each node the new id of its
// first child, and all threads then write the level's children together. Two grid-wide
// kernels follow: one gathers the kept nodes' fields into a workspace, the other writes them
// over the front of the tree. The workspace holds eight int32 arrays of `capacity` entries
// per tree.
#include <algorithm>
#include <mutex>

#include "omq_common.h"

namespace omq {

constexpr int kShiftThreads = 1024;
constexpr int kShiftWaves = kShiftThreads / kWave;

// Workgroup barrier that orders LDS only: global loads in flight stay in flight across it
// (__syncthreads also waits for them).
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Breadth-first numbering of tree t's kept nodes (one workgroup per tree).  Writes, for new
// id i: old_of_new[i], npar[i], nfirst[i], nnch[i]; then num_nodes[t] = kept count.  npar[0]
// is -1 for a tree to move and -2 for a tree left unchanged (no shift, or an inconsistent row:
// a row that leaves [0, num_nodes), or more kept nodes than num_nodes, as from a cycle).
// A level is taken in chunks of kShiftPer nodes per thread, a workgroup's width apart, so that the
// row loads of a chunk are in flight together and consecutive lanes load consecutive nodes (with
// consecutive nodes per thread every load touched four times the lines: 7.4 M nodes of 32 trees
// kept, the whole shift, 1325 -> 822 us, with the chunk's scan by DPP and one barrier less).  The
// chunk's children are written in tiles of 64
// consecutive new ids, one tile per wave at a time: the chunk's nodes with children are
// compacted (their first child's offset strictly increasing), the tile's first node is found
// by a two-level search over that list (64 samples, then 64 entries: two LDS reads per lane),
// and each lane walks forward from it to the node of its own id.
constexpr int kShiftPer = 4;
constexpr int kShiftChunk = kShiftThreads * kShiftPer;
constexpr int kShiftSlots = kShiftWaves * kShiftPer;
static_assert(kShiftSlots == kWave, "one wave scans the slots' totals");

__global__ __launch_bounds__(kShiftThreads) void shift_order_kernel(omq_forest f,
                                                                    const int32_t* new_roots,
                                                                    int32_t* ws) {
  __shared__ int s_ktot[kShiftSlots];  // children, and
  __shared__ int s_ztot[kShiftSlots];  //   rows, of each wave's 64 nodes of the chunk
  __shared__ int s_cex[kShiftChunk];  // compacted nodes with children: first child's offset
  __shared__ int s_cof[kShiftChunk];  //   their old row offset
  __shared__ int s_cid[kShiftChunk];  //   their position in the chunk
  __shared__ int s_bad;               // a row of the chunk is inconsistent
  const int t = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = tid / kWave;
  const int cap = f.capacity;
  const int64_t tb = (int64_t)t * cap;
  int32_t* old_of_new = ws + (int64_t)t * cap * 8;
  int32_t* npar = old_of_new + cap;
  int32_t* nfirst = old_of_new + 2 * (int64_t)cap;
  int32_t* nnch = old_of_new + 3 * (int64_t)cap;
  const int r = new_roots[t];
  const int n_old = f.num_nodes[t];
  if (r <= 0 || r >= n_old) {  // 0: already the root; -1: no shift
    if (tid == 0) npar[0] = -2;
    return;
  }
  if (tid == 0) {
    old_of_new[0] = r;
    s_bad = 0;
  }
  __syncthreads();
  // level [lo, hi) of new ids; its children get [hi, next)
  int lo = 0, hi = 1, next = 1;
  bool bad = false;
  // The rows of a level's next chunk are loaded while the current chunk is processed: a
  // level's new-to-old ids were all written before the level began, and the barriers inside a
  // chunk order LDS only, so the loads stay in flight until the chunk's end.
  int pk[kShiftPer], pof[kShiftPer];
  auto load_rows = [&](int c0) {
    int old[kShiftPer];
#pragma unroll
    for (int e = 0; e < kShiftPer; ++e) {
      const int i = c0 + e * kShiftThreads + tid;
      old[e] = i < hi ? old_of_new[i] : -1;
    }
#pragma unroll
    for (int e = 0; e < kShiftPer; ++e) {
      pk[e] = old[e] >= 0 ? f.num_children[tb + old[e]] : 0;
      pof[e] = old[e] >= 0 ? f.first_child[tb + old[e]] : 0;
    }
  };
  while (lo < hi && !bad) {
    load_rows(lo);
    for (int c0 = lo; c0 < hi; c0 += kShiftChunk) {
      int k[kShiftPer], of[kShiftPer], upto[kShiftPer];
#pragma unroll
      for (int e = 0; e < kShiftPer; ++e) {
        k[e] = pk[e];
        of[e] = pof[e];
      }
      if (c0 + kShiftChunk < hi) load_rows(c0 + kShiftChunk);
      bool row_bad = false;
#pragma unroll
      for (int e = 0; e < kShiftPer; ++e) {
        if (k[e] < 0 || (k[e] > 0 && (of[e] < 0 || (int64_t)of[e] + k[e] >= n_old))) {
          row_bad = true;
          k[e] = 0;
        }
        // (slot e * kShiftWaves + wave: the chunk's nodes in order)
        upto[e] = wave_incl_scan(k[e]);
        const int z = __popcll(__ballot(k[e] > 0));
        if (lane == kWave - 1) {
          s_ktot[e * kShiftWaves + wave] = upto[e];
          s_ztot[e * kShiftWaves + wave] = z;
        }
      }
      if (row_bad) s_bad = 1;  // (read after the barrier)
      lds_barrier();
      const bool any_bad = s_bad != 0;
      // every wave scans the slots' totals, a slot per lane
      int tot, nz;
      const int kslot = wave_excl_scan(s_ktot[lane], &tot);
      const int zslot = wave_excl_scan(s_ztot[lane], &nz);
      if (any_bad || next + tot > n_old) {
        bad = true;
        break;
      }
#pragma unroll
      for (int e = 0; e < kShiftPer; ++e) {
        const int i = c0 + e * kShiftThreads + tid;
        const int slot = e * kShiftWaves + wave;
        const int ex = readlane_i(kslot, slot) + upto[e] - k[e];
        const uint64_t rows = __ballot(k[e] > 0);
        if (i < hi) {
          nnch[i] = k[e];
          nfirst[i] = k[e] > 0 ? next + ex - 1 : -1;
        }
        if (k[e] > 0) {
          const int zx = readlane_i(zslot, slot) +
                         (int)__builtin_amdgcn_mbcnt_hi(
                             (uint32_t)(rows >> 32),
                             __builtin_amdgcn_mbcnt_lo((uint32_t)rows, 0u));
          s_cex[zx] = ex;
          s_cof[zx] = of[e];
          s_cid[zx] = e * kShiftThreads + tid;
        }
      }
      lds_barrier();
      // the chunk's children, tile by tile: output q belongs to the last listed node j with
      // s_cex[j] <= q, as its child q - s_cex[j]
      for (int q0 = wave * kWave; q0 < tot; q0 += kShiftThreads) {
        // the tile's first node: a sample every 64 entries, then the entries after the sample
        const int si = lane * kWave;
        const uint64_t b1 = __ballot(si < nz && s_cex[si] <= q0);  // lane 0 always qualifies
        const int L = kWave - 1 - __clzll(b1);
        const int sj = L * kWave + lane;
        const uint64_t b2 = __ballot(sj < nz && s_cex[sj] <= q0);
        int j = L * kWave + (kWave - 1 - __clzll(b2));
        const int q = q0 + lane;
        if (q < tot) {
          // forward to the last node starting at or before q (at most nz - 1 - j steps)
          while (j + 1 < nz && s_cex[j + 1] <= q) ++j;
          old_of_new[next + q] = s_cof[j] + 1 + (q - s_cex[j]);  // child of edge of+x is node of+x+1
          npar[next + q] = c0 + s_cid[j];
        }
      }
      next += tot;
      __syncthreads();
    }
    lo = hi;
    hi = next;
  }
  if (tid == 0) {
    npar[0] = bad ? -2 : -1;
    if (!bad) f.num_nodes[t] = next;
  }
}

// Gathers the kept nodes' N, W, P and action into the workspace (grid-stride over new ids).
__global__ void shift_gather_kernel(omq_forest f, int32_t* ws) {
  const int t = blockIdx.y;
  const int cap = f.capacity;
  const int64_t tb = (int64_t)t * cap;
  const int32_t* old_of_new = ws + (int64_t)t * cap * 8;
  const int32_t* npar = old_of_new + cap;
  if (npar[0] != -1) return;
  int32_t* nN = const_cast<int32_t*>(old_of_new) + 4 * (int64_t)cap;
  float* nW = reinterpret_cast<float*>(nN + cap);
  float* nP = reinterpret_cast<float*>(nN + 2 * (int64_t)cap);
  int32_t* nA = nN + 3 * (int64_t)cap;
  const int n_new = f.num_nodes[t];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n_new; i += gridDim.x * blockDim.x) {
    const int64_t o = tb + old_of_new[i];
    nN[i] = f.visit_counts[o];
    nW[i] = f.value_sums[o];
    nP[i] = f.priors[o];
    nA[i] = i == 0 ? -1 : f.actions[o];
  }
}

// Writes the compacted tree over the front of the tree's arrays.
__global__ void shift_write_kernel(omq_forest f, const int32_t* ws) {
  const int t = blockIdx.y;
  const int cap = f.capacity;
  const int64_t tb = (int64_t)t * cap;
  const int32_t* base = ws + (int64_t)t * cap * 8;
  const int32_t* npar = base + cap;
  if (npar[0] != -1) return;
  const int32_t* nfirst = base + 2 * (int64_t)cap;
  const int32_t* nnch = base + 3 * (int64_t)cap;
  const int32_t* nN = base + 4 * (int64_t)cap;
  const float* nW = reinterpret_cast<const float*>(nN + cap);
  const float* nP = reinterpret_cast<const float*>(nN + 2 * (int64_t)cap);
  const int32_t* nA = nN + 3 * (int64_t)cap;
  const int n_new = f.num_nodes[t];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n_new; i += gridDim.x * blockDim.x) {
    const int64_t d = tb + i;
    f.visit_counts[d] = nN[i];
    f.value_sums[d] = nW[i];
    f.priors[d] = nP[i];
    f.parents[d] = npar[i];
    f.first_child[d] = nfirst[i];
    f.num_children[d] = nnch[i];
    f.actions[d] = nA[i];
  }
}

// ---- the workspace of omq_shift_root_noalloc ----------------------------------------------
// A file-scope device array, one copy per GPU the library runs on, held until the process
// ends.  Its address on a device is looked up once per device, with that device current
// (hipGetSymbolAddress); host code never passes the array's name to a kernel.  Every entry the
// shift kernels read is written earlier in the same call, so nothing has to start at zero.
// Calls that overlap on one GPU share the array and race.
static __device__ __align__(256) int32_t scratch[OMQ_NOALLOC_SHIFT_INTS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
int32_t* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

// The address of this device's scratch (looked up on the first call on the device).
hipError_t shift_scratch(int32_t** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (p == nullptr) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = static_cast<int32_t*>(p);
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}

hipError_t launch_shift_root(const omq_forest& f, const int32_t* new_roots, int32_t* ws,
                             hipStream_t st) {
  hipLaunchKernelGGL(shift_order_kernel, dim3(f.num_trees), dim3(kShiftThreads), 0, st, f,
                     new_roots, ws);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int blocks = (int)std::min<int64_t>(64, ((int64_t)f.capacity + 255) / 256);
  hipLaunchKernelGGL(shift_gather_kernel, dim3(blocks, f.num_trees), dim3(256), 0, st, f, ws);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(shift_write_kernel, dim3(blocks, f.num_trees), dim3(256), 0, st, f, ws);
  return hipGetLastError();
}

}  // namespace omq

// ===========================================================================================
// The reference's two-step subtree API: parallel_bfs_subtree and extract_subtree_edges
// (python/mcts/gpu/mcts_kernels.cu:2095-2337, bound at :2396-2408), over a CSR graph
// (row_ptr [max_nodes + 1], col_indices [num_edges]).  Their callers are
// python/mcts/gpu/gpu_bfs.py:49,149 and python/mcts/gpu/compact_subtree.py:220.
//   - BFS: breadth-first from root_idx, each level's nodes in order and each row's children in
//     row order; a child not yet in the subtree gets the next new index at its first
//     occurrence (the order of the reference's fallback, gpu_bfs.py:70-127, and of a FIFO
//     queue).  Children outside [0, max_nodes) are skipped.  The reference kernel numbers
//     children in the order its atomics land and marks a bool array through 32-bit CAS at the
//     child's index (touching the three bytes after it and reading past the array): its order
//     is one of the orders that can arise, and no other.
//   - Edges: for every node of the subtree in ascending old index, the edges of its row (in
//     row order) whose child lies in the subtree, as (new parent, new child, action); the
//     reference appends them in atomic order, of which this is one.
// ===========================================================================================
namespace omq {

constexpr int kBfsThreads = 1024;
constexpr int kBfsWaves = kBfsThreads / kWave;

// exclusive scan of one int64 per thread over the workgroup; total through *tot
__device__ inline int64_t bfs_block_scan(int64_t v, int64_t* s_wtot, int64_t* tot) {
  const int wave = (int)threadIdx.x / kWave, lane = lane_id();
  int64_t x = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int64_t y = __shfl_up(x, off, kWave);
    if (lane >= off) x += y;
  }
  if (lane == kWave - 1) s_wtot[wave] = x;
  __syncthreads();
  int64_t before = 0, all = 0;
  for (int i = 0; i < kBfsWaves; ++i) {
    const int64_t t = s_wtot[i];
    before += i < wave ? t : 0;
    all += t;
  }
  __syncthreads();  // s_wtot is reused by the next scan
  *tot = all;
  return before + x - v;
}

// row [a, b) of node, clamped to the edge array
__device__ inline void bfs_row(const int32_t* row_ptr, int num_edges, int node, int* a, int* b) {
  int lo = row_ptr[node], hi = row_ptr[node + 1];
  lo = lo < 0 ? 0 : (lo > num_edges ? num_edges : lo);
  hi = hi < lo ? lo : (hi > num_edges ? num_edges : hi);
  *a = lo;
  *b = hi;
}

// ---- breadth-first subtree ------------------------------------------------------------------
// Marks, ids and claims of every node before the search: by the whole chip (one workgroup took
// about a fifth of the search for it), or, up to kBfsClearHere nodes, by the search's workgroup
// itself, which saves a launch (a graph of 10 nodes 14.5 -> 5.4 us with the narrow levels below; one
// of 8000 43 us so, of 9000 48 us with the launch).
__device__ inline void bfs_clear(int root, int max_nodes, uint8_t* in_subtree, int32_t* remap,
                                 int32_t* claim, int32_t* queue, int64_t first, int64_t step) {
  for (int64_t i = first; i < max_nodes; i += step) {
    in_subtree[i] = i == root ? 1 : 0;
    remap[i] = i == root ? 0 : -1;
    claim[i] = 0x7FFFFFFF;
  }
  if (first == 0) queue[0] = root;
}
__global__ void bfs_clear_kernel(int root, int max_nodes, uint8_t* in_subtree, int32_t* remap,
                                 int32_t* claim, int32_t* queue) {
  bfs_clear(root, max_nodes, in_subtree, remap, claim, queue,
            (int64_t)blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// Exclusive scan of one int per thread over the workgroup in the vector registers (the total
// within 31 bits); the waves' totals through LDS, scanned by every wave.
__device__ inline int bfs_block_scan32(int v, int* s_wtot, int* tot) {
  const int wave = (int)threadIdx.x / kWave, lane = lane_id();
  const int upto = wave_incl_scan(v);
  if (lane == kWave - 1) s_wtot[wave] = upto;
  __syncthreads();
  const int waves = wave_excl_scan(lane < kBfsWaves ? s_wtot[lane] : 0, tot);
  __syncthreads();  // s_wtot is reused by the next scan
  return readlane_i(waves, wave) + upto - v;
}

// Exclusive scans of an int64 and an int per thread over the workgroup, together.
__device__ inline int64_t bfs_block_scan2(int64_t v, int n, int64_t* s_wtot, int64_t* tot,
                                          int* n_ex, int* n_tot) {
  // (n's total stays below 2^16: it rides in the low bits of the scanned value)
  const int64_t ex = bfs_block_scan((v << 16) | n, s_wtot, tot);
  *n_ex = (int)(ex & 0xFFFF);
  *n_tot = (int)(*tot & 0xFFFF);
  *tot >>= 16;
  return ex >> 16;
}

// The same for values whose totals stay below 2^31 each, in 32 bits.
__device__ inline int bfs_block_scan2_32(int v, int n, int64_t* s_wtot, int64_t* tot, int* n_ex,
                                         int* n_tot) {
  const int wave = (int)threadIdx.x / kWave, lane = lane_id();
  const int upto = wave_incl_scan(v), n_upto = wave_incl_scan(n);
  if (lane == kWave - 1) s_wtot[wave] = (int64_t)upto << 32 | n_upto;
  __syncthreads();
  const int64_t w = lane < kBfsWaves ? s_wtot[lane] : 0;
  int t32;
  const int waves = wave_excl_scan((int)(w >> 32), &t32);
  const int n_waves = wave_excl_scan((int)w, n_tot);
  __syncthreads();  // s_wtot is reused by the next scan
  *tot = t32;
  *n_ex = readlane_i(n_waves, wave) + n_upto - n;
  return readlane_i(waves, wave) + upto - v;
}

// The search, by one workgroup; its time is its chains of dependent loads, so every round has
// many of them in flight.  A level's rows are taken kBfsPer nodes per thread at a time: a scan of
// their lengths gives each row its place in the level's list of candidate edges, the rows with
// edges are compacted in LDS, and the candidates are dealt in tiles of 64 (their row found by a
// two-level search of that list, kBfsTiles tiles of a wave in flight).  Every candidate outside
// the subtree claims its child with its place (the earliest wins), and is kept in the queue past
// the level, where the winners are then numbered in order and compacted in place, kBfsNumber
// candidates per thread and scan.  100k of 300k nodes: 208 us with one candidate per thread,
// its row found by a binary search in memory, twice, and the clearing in this workgroup; 79 us
// so.  A level of more candidates than the queue has room for (rows that overlap, repeated
// children) finds its candidates again for the numbering.
// A level costs the workgroup its barriers and scans whatever its size, so the levels that one wave
// can take (at most 64 nodes, kNarrowTiles * 64 candidates) are taken by one wave, with the nodes in
// registers and no barrier, one after the other until a wider level comes.  Device time of the
// search, one candidate per thread / without the narrow levels / so: a chain of 2000 nodes 6391 /
// 9010 / 2715 us, a binary tree of 4095 65.0 / 84.9 / 37.9, 40k nodes in levels of about 225 with
// rows of one or two 1012 / 1543 / 822 (the row of a candidate by halving, and the scans in 32
// bits); the 100k of 300k nodes above, with the edges, 136 -> 129.  (Four nodes per lane and 512
// candidates in the narrow levels: the chain 3963 us, the 300k nodes 141.)
// Workspace: queue [max_nodes], claim [max_nodes].
constexpr int kBfsPer = 4;
constexpr int kBfsChunk = kBfsThreads * kBfsPer;
constexpr int kBfsTiles = 8;
constexpr int kBfsNumber = 8;
constexpr int kBfsShort = 8;  // rows shorter than this on average: a candidate's row by halving
constexpr int kBfsEdges32 = 0x7FFFFFFF / kBfsChunk;  // a chunk's rows add up to 31 bits at most
constexpr int kNarrowTiles = 4;
constexpr int kBfsClearHere = 8192;

__global__ __launch_bounds__(kBfsThreads) void bfs_subtree_kernel(
    const int32_t* row_ptr, const int32_t* col, int num_edges, int root, int max_nodes,
    uint8_t* in_subtree, int32_t* remap, int32_t* count_out, int32_t* queue, int32_t* claim) {
  __shared__ int64_t s_wtot[kBfsWaves];
  __shared__ int s_wtot32[kBfsWaves];
  __shared__ int s_level[2];
  __shared__ int s_cex[kBfsChunk];  // rows with edges: place of the first edge in the chunk
  __shared__ int s_cof[kBfsChunk];  //   and its index in col
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = tid / kWave;
  int start = 0, end = 1;  // the current level: queue[start, end)
  // The rows of level nodes [c0, c0 + kBfsChunk) into s_cex / s_cof; returns their number of
  // edges, *nz the rows with any.  Ends with a barrier.
  auto load_chunk = [&](int64_t c0, int* nz) -> int64_t {
    int of[kBfsPer], len[kBfsPer];
    int64_t mine = 0;
    int nzm = 0;
    const int64_t i0 = start + c0 + tid * kBfsPer;  // (64 bits: up to a chunk past max_nodes)
    int node[kBfsPer];
#pragma unroll
    for (int e = 0; e < kBfsPer; ++e) node[e] = i0 + e < end ? queue[i0 + e] : -1;
#pragma unroll
    for (int e = 0; e < kBfsPer; ++e) {
      of[e] = len[e] = 0;
      if (node[e] >= 0) {
        int a, b;
        bfs_row(row_ptr, num_edges, node[e], &a, &b);
        of[e] = a;
        len[e] = b - a;
      }
    }
#pragma unroll
    for (int e = 0; e < kBfsPer; ++e) {
      mine += len[e];
      nzm += len[e] > 0 ? 1 : 0;
    }
    int64_t tot;
    int zx;
    int64_t ex = num_edges <= kBfsEdges32
                     ? bfs_block_scan2_32((int)mine, nzm, s_wtot, &tot, &zx, nz)
                     : bfs_block_scan2(mine, nzm, s_wtot, &tot, &zx, nz);
#pragma unroll
    for (int e = 0; e < kBfsPer; ++e) {
      if (len[e] > 0) {
        s_cex[zx] = (int)min(ex, (int64_t)0x7FFFFFFF);
        s_cof[zx] = of[e];
        ++zx;
      }
      ex += len[e];
    }
    __syncthreads();
    return tot;
  };
  // the child of candidate q0 + lane of the chunk (nz rows, tot candidates); called by whole waves
  auto child_of = [&](int q0, int nz, int tot) -> int {
    const int si = lane * kWave;
    const uint64_t b1 = __ballot(si < nz && s_cex[si] <= q0);  // lane 0 always qualifies
    const int S = kWave - 1 - __clzll(b1);
    const int sj = S * kWave + lane;
    const uint64_t b2 = __ballot(sj < nz && s_cex[sj] <= q0);
    int j = S * kWave + (kWave - 1 - __clzll(b2));
    const int q = q0 + lane;
    if (q >= tot) return -1;
    // on to the last row that starts at or before q, at most 63 further (the rows have edges)
    if (nz * kBfsShort > tot) {
#pragma unroll
      for (int h = kWave / 2; h >= 1; h >>= 1)
        if (j + h < nz && s_cex[j + h] <= q) j += h;
    } else {
      while (j + 1 < nz && s_cex[j + 1] <= q) ++j;
    }
    return col[s_cof[j] + (q - s_cex[j])];
  };
  auto outside = [&](int c) { return c >= 0 && c < max_nodes && !in_subtree[c]; };
  auto claimed_by = [&](int c) {  // (past this CU's L1: claims are made by atomics in L2)
    return __hip_atomic_load(&claim[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  // The narrow levels from [start, end) on, by one wave; returns at the first that is not.
  auto narrow_levels = [&]() {
    int node = lane < end - start ? queue[start + lane] : -1;
    while (start < end && end - start <= kWave) {
      int a = 0, len = 0;
      if (node >= 0) {
        int b;
        bfs_row(row_ptr, num_edges, node, &a, &b);
        len = b - a;
      }
      if (__any(len > kNarrowTiles * kWave)) return;
      const int upto = wave_incl_scan(len);
      const int tot = readlane_i(upto, kWave - 1);
      if (tot > kNarrowTiles * kWave) return;
      int c[kNarrowTiles];
      bool win[kNarrowTiles];
#pragma unroll
      for (int u = 0; u < kNarrowTiles; ++u) {
        c[u] = -1;
        win[u] = false;
        if (u * kWave >= tot) continue;
        const int q = u * kWave + lane;
        int lo = 0;  // the first lane whose rows end past q
#pragma unroll
        for (int h = kWave / 2; h >= 1; h >>= 1)
          if (__shfl(upto, lo + h - 1, kWave) <= q) lo += h;
        lo = min(lo, kWave - 1);
        const int at = __shfl(a, lo, kWave) + (q - __shfl(upto - len, lo, kWave));
        if (q < tot) c[u] = col[at];
      }
#pragma unroll
      for (int u = 0; u < kNarrowTiles; ++u)
        if (!outside(c[u])) c[u] = -1;
      if (tot <= kWave) {
        // a child's first candidate, from the lanes of the same child (a ballot per bit)
        uint64_t same = __ballot(c[0] >= 0);
        for (int b = 0; b < 32 - __clz(max_nodes); ++b) {
          const bool one = (c[0] >> b) & 1;
          const uint64_t bal = __ballot(one);
          same &= one ? bal : ~bal;
        }
        win[0] = c[0] >= 0 && lowest_lane(same) == lane;
      } else {
        bool some = false;
#pragma unroll
        for (int u = 0; u < kNarrowTiles; ++u) {
          if (c[u] >= 0) win[u] = atomicMin(&claim[c[u]], u * kWave + lane) > u * kWave + lane;
          some = some || win[u];
        }
        if (__any(some)) {  // (on every claim's result: all are made before any is read)
#pragma unroll
          for (int u = 0; u < kNarrowTiles; ++u)
            win[u] = win[u] && claimed_by(c[u]) == u * kWave + lane;
        }
      }
      int added = 0;
#pragma unroll
      for (int u = 0; u < kNarrowTiles; ++u) {
        const uint64_t m = __ballot(win[u]);
        const int r = added + (int)__builtin_amdgcn_mbcnt_hi(
                                  (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (win[u]) {
          remap[c[u]] = end + r;
          in_subtree[c[u]] = 1;
          queue[end + r] = c[u];
          s_cex[r] = c[u];
        }
        added += __popcll(m);
      }
      wave_sync();
      node = lane < added ? s_cex[lane] : -1;
      wave_sync();
      start = end;
      end += added;
    }
  };
  if (max_nodes <= kBfsClearHere) {
    bfs_clear(root, max_nodes, in_subtree, remap, claim, queue, tid, kBfsThreads);
    __syncthreads();
  }
  bool overflow = false;
  while (start < end) {
    if (end - start <= kWave) {
      if (wave == 0) {
        narrow_levels();
        if (lane == 0) {
          s_level[0] = start;
          s_level[1] = end;
        }
      }
      __syncthreads();
      start = s_level[0];
      end = s_level[1];
      if (start == end) break;
    }
    const int L = end - start;
    int64_t run = 0;
    bool stash = true;  // the level's candidates so far are in queue[end, end + run)
    for (int64_t c0 = 0; c0 < L; c0 += kBfsChunk) {
      int nz;
      const int64_t tot = load_chunk(c0, &nz);
      if (run + tot > 0x7FFFFFFF) {  // more candidates than int32 keys (rows that overlap)
        overflow = true;
        break;
      }
      stash = stash && end + run + tot <= max_nodes;
      for (int64_t q0 = wave * kWave; q0 < tot; q0 += kBfsTiles * kBfsThreads) {
        int c[kBfsTiles];
        bool ok[kBfsTiles];
#pragma unroll
        for (int u = 0; u < kBfsTiles; ++u)
          c[u] = q0 + u * kBfsThreads < tot
                     ? child_of((int)q0 + u * kBfsThreads, nz, (int)tot) : -1;
#pragma unroll
        for (int u = 0; u < kBfsTiles; ++u) ok[u] = outside(c[u]);
#pragma unroll
        for (int u = 0; u < kBfsTiles; ++u) {
          const int64_t q = q0 + u * kBfsThreads + lane;
          if (ok[u]) atomicMin(&claim[c[u]], (int)(run + q));
          if (stash && q < tot) queue[end + run + q] = ok[u] ? c[u] : -1;
        }
      }
      run += tot;
      __syncthreads();  // the next chunk's rows overwrite the list
    }
    if (overflow) break;
    // the winners, numbered in the order of the candidates
    int added = 0;
    if (stash) {
      for (int64_t k0 = 0; k0 < run; k0 += kBfsNumber * kBfsThreads) {
        const int64_t k = k0 + tid * kBfsNumber;
        int c[kBfsNumber], by[kBfsNumber];
        int won = 0;
#pragma unroll
        for (int e = 0; e < kBfsNumber; ++e) c[e] = k + e < run ? queue[end + k + e] : -1;
#pragma unroll
        for (int e = 0; e < kBfsNumber; ++e) by[e] = c[e] >= 0 ? claimed_by(c[e]) : -1;
#pragma unroll
        for (int e = 0; e < kBfsNumber; ++e) won += c[e] >= 0 && by[e] == (int)(k + e) ? 1 : 0;
        int tot;
        int at = end + added + bfs_block_scan32(won, s_wtot32, &tot);
#pragma unroll
        for (int e = 0; e < kBfsNumber; ++e) {
          if (c[e] >= 0 && by[e] == (int)(k + e)) {
            remap[c[e]] = at;
            in_subtree[c[e]] = 1;
            queue[at] = c[e];  // (at or before the candidate's own place, read by now)
            ++at;
          }
        }
        added += tot;
      }
    } else {
      run = 0;
      for (int64_t c0 = 0; c0 < L; c0 += kBfsChunk) {
        int nz;
        const int tot = (int)load_chunk(c0, &nz);
        for (int64_t k0 = 0; k0 < tot; k0 += kBfsThreads) {
          const int c = k0 + wave * kWave < tot ? child_of((int)k0 + wave * kWave, nz, tot) : -1;
          const bool win = outside(c) && claimed_by(c) == (int)(run + k0 + tid);
          int wins;
          const int at = end + added + bfs_block_scan32(win ? 1 : 0, s_wtot32, &wins);
          if (win) {
            remap[c] = at;
            queue[at] = c;
          }
          added += wins;
        }
        run += tot;
        __syncthreads();
      }
      for (int i = tid; i < added; i += kBfsThreads) in_subtree[queue[end + i]] = 1;
    }
    __syncthreads();
    start = end;
    end += added;
  }
  if (tid == 0) count_out[0] = overflow ? -1 : end;
}

// Edge extraction: kept edges per group of nodes and scan in the chunk (pass 1), scan of the chunk
// totals (pass 2), writes (pass 3).  A chunk is 256 nodes, 16 groups of 16.  A workgroup takes
// kEdgeParts chunks, a grid's width apart, and each of its waves one group of each: 64 rows, whose
// edges are one list, 64 edges at a time, kEdgeTiles such tiles in flight, so that consecutive lanes
// read consecutive edges and write consecutive outputs.  The time is dependent loads, so it goes with
// the number of waves where few nodes are kept (64 rows a wave), and where the nodes that have edges
// lie together, as in a search tree, with the waves that these are spread over (16 of their rows a
// wave).  Device time of the three launches, one node per thread with its row in a loop / 16 nodes a
// wave with 64-bit scans / so:
//   random tree of 300k nodes, none kept 8.7 / 19.7 / 8.3 us, 30 % 18.6 / 40.1 / 13.8, all 30.4 / 43.0 /
//   17.8; of 2M 18.5 / 83.7 / 18.1, 47.9 / 198 / 47.4 and 99.4 / 215 / 75.1; of 20k, 30 % 14.5 / 15.5 / 11.3;
//   64 children to a node, 300k nodes, 30 % 68.6 / 26.1 / 25.4, all 338 / 36.3 / 36.0; ten nodes 7.9 /
//   9.9 / 9.0 (three short launches), a chain of 20k 9.0 / 15.5 / 11.5.
// Workspace: the groups' first edges in the chunk, then the chunk totals.
constexpr int kEdgeThreads = 1024;
constexpr int kEdgeWaves = kEdgeThreads / kWave;
constexpr int kEdgeTiles = 4;
constexpr int kEdgeNodes = 16;  // of a group
constexpr int kEdgeParts = kWave / kEdgeNodes;
constexpr int kEdgeChunk = kEdgeWaves * kEdgeNodes;

// The node of a lane (past the nodes where there is none); part p's group is that of lane 16 p.
__device__ inline int64_t edge_node(int lane) {
  const int64_t chunk = blockIdx.x + (int64_t)(lane / kEdgeNodes) * gridDim.x;
  return chunk * kEdgeChunk + (int)threadIdx.x / kWave * kEdgeNodes + lane % kEdgeNodes;
}

// Inclusive prefix sums of the lanes' row lengths.
__device__ inline int rows_upto(int len, int) { return wave_incl_scan(len); }
__device__ inline int64_t rows_upto(int len, int64_t) {
  int64_t upto = len;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int64_t y = __shfl_up(upto, off, kWave);
    if (lane_id() >= off) upto += y;
  }
  return upto;
}

// Calls emit(kept by this lane, edge, child, owner lane) for every tile of the edges of the lanes'
// rows [a, a + len), in order.  Called by whole waves; Int holds the rows' total and a round more.
template <class Int, class Emit>
__device__ inline void walk_rows(const int32_t* col, const uint8_t* in_subtree, int num_nodes,
                                 int a, int len, Emit emit) {
  const int lane = lane_id();
  const Int upto = rows_upto(len, Int());
  const Int total = __shfl(upto, kWave - 1, kWave);
  for (Int q0 = 0; q0 < total; q0 += kEdgeTiles * kWave) {
    int edge[kEdgeTiles], own[kEdgeTiles], c[kEdgeTiles];
    bool keep[kEdgeTiles];
    const int tiles = (int)min((total - q0 + kWave - 1) / kWave, (Int)kEdgeTiles);
#pragma unroll
    for (int u = 0; u < kEdgeTiles; ++u) {
      edge[u] = -1;
      own[u] = 0;
      if (u >= tiles) continue;
      const Int q = q0 + u * kWave + lane;
      int lo = 0;  // the first lane whose rows end past q
#pragma unroll
      for (int h = kWave / 2; h >= 1; h >>= 1)
        if (__shfl(upto, lo + h - 1, kWave) <= q) lo += h;
      const Int from = __shfl(upto - len, lo, kWave);
      const int base = __shfl(a, lo, kWave);
      own[u] = lo;
      if (q < total) edge[u] = (int)(base + (q - from));
    }
#pragma unroll
    for (int u = 0; u < kEdgeTiles; ++u) c[u] = edge[u] >= 0 ? col[edge[u]] : -1;
#pragma unroll
    for (int u = 0; u < kEdgeTiles; ++u)
      keep[u] = c[u] >= 0 && c[u] < num_nodes && in_subtree[c[u]];
#pragma unroll
    for (int u = 0; u < kEdgeTiles; ++u)
      if (u < tiles) emit(keep[u], edge[u], c[u], own[u]);
  }
}
template <class Emit>
__device__ inline void walk_edges(const int32_t* col, int num_edges, const uint8_t* in_subtree,
                                  int num_nodes, int a, int len, Emit emit) {
  // (rows may overlap: a wave's add up to kWave * num_edges at most)
  if (num_edges <= (0x7FFFFFFF - kEdgeTiles * kWave) / kWave)
    walk_rows<int>(col, in_subtree, num_nodes, a, len, emit);
  else
    walk_rows<int64_t>(col, in_subtree, num_nodes, a, len, emit);
}

// The lane's row: its first edge and its length (0 outside the subtree).
__device__ inline int edge_row(const int32_t* row_ptr, int num_edges, const uint8_t* in_subtree,
                               int num_nodes, int64_t node, int* a) {
  *a = 0;
  if (node >= num_nodes || !in_subtree[node]) return 0;
  int b;
  bfs_row(row_ptr, num_edges, (int)node, a, &b);
  return b - *a;
}

__global__ __launch_bounds__(kEdgeThreads) void edges_count_kernel(
    const int32_t* row_ptr, const int32_t* col, int num_edges, const uint8_t* in_subtree,
    int num_nodes, int32_t* local, int32_t* chunk_tot) {
  __shared__ int64_t s_kept[kEdgeWaves][kEdgeParts];
  const int wave = (int)threadIdx.x / kWave;
  const int lane = lane_id();
  int64_t n[kEdgeParts] = {};
  int a;
  const int len = edge_row(row_ptr, num_edges, in_subtree, num_nodes, edge_node(lane), &a);
  if (__any(len > 0))
    walk_edges(col, num_edges, in_subtree, num_nodes, a, len,
               [&](bool mine, int, int, int owner) {
#pragma unroll
                 for (int p = 0; p < kEdgeParts; ++p)
                   n[p] += __popcll(__ballot(mine && owner / kEdgeNodes == p));
               });
  if (lane == 0)
#pragma unroll
    for (int p = 0; p < kEdgeParts; ++p) s_kept[wave][p] = n[p];
  __syncthreads();
  if (lane >= kEdgeParts) return;
  int64_t before = 0;
  for (int i = 0; i < wave; ++i) before += s_kept[i][lane];
  const int64_t first = edge_node(lane * kEdgeNodes);
  if (first < num_nodes) local[first / kEdgeNodes] = (int32_t)before;
  const int64_t chunk = first / kEdgeChunk;
  if (wave == kEdgeWaves - 1 && chunk * kEdgeChunk < num_nodes)
    chunk_tot[chunk] = (int32_t)(before + s_kept[wave][lane]);
}

// kScanPer chunks per thread and scan
constexpr int kScanPer = 4;
__global__ __launch_bounds__(kEdgeThreads) void edges_scan_kernel(int32_t* chunk_tot, int chunks,
                                                                  int32_t* edge_count) {
  __shared__ int64_t s_wtot[kEdgeWaves];
  int64_t run = 0;
  for (int b0 = 0; b0 < chunks; b0 += kEdgeThreads * kScanPer) {
    const int b = b0 + (int)threadIdx.x * kScanPer;
    int v[kScanPer];
    int64_t mine = 0;
#pragma unroll
    for (int e = 0; e < kScanPer; ++e) v[e] = b + e < chunks ? chunk_tot[b + e] : 0;
#pragma unroll
    for (int e = 0; e < kScanPer; ++e) mine += v[e];
    int64_t tot;
    int64_t at = run + bfs_block_scan(mine, s_wtot, &tot);
#pragma unroll
    for (int e = 0; e < kScanPer; ++e) {
      if (b + e < chunks) chunk_tot[b + e] = (int32_t)at;
      at += v[e];
    }
    run += tot;
  }
  if (threadIdx.x == 0) edge_count[0] = (int32_t)min(run, (int64_t)0x7FFFFFFF);
}

__global__ __launch_bounds__(kEdgeThreads) void edges_write_kernel(
    const int32_t* row_ptr, const int32_t* col, const int16_t* actions, int num_edges,
    const uint8_t* in_subtree, const int32_t* remap, int num_nodes, int max_edges,
    const int32_t* local, const int32_t* chunk_off, int32_t* out_parent, int32_t* out_child,
    int16_t* out_action) {
  const int lane = lane_id();
  const int64_t node = edge_node(lane);
  int a;
  const int len = edge_row(row_ptr, num_edges, in_subtree, num_nodes, node, &a);
  if (!__any(len > 0)) return;
  const int id = node < num_nodes ? remap[node] : -1;
  const int64_t first = edge_node(lane % kEdgeParts * kEdgeNodes);
  const int64_t off = first < num_nodes
                          ? (int64_t)chunk_off[first / kEdgeChunk] + local[first / kEdgeNodes] : 0;
  int64_t pos[kEdgeParts];  // the next output of each part's group
#pragma unroll
  for (int p = 0; p < kEdgeParts; ++p) pos[p] = __shfl(off, p, kWave);
  walk_edges(col, num_edges, in_subtree, num_nodes, a, len,
             [&](bool mine, int edge, int child, int owner) {
               const int parent = __shfl(id, owner, kWave);
               int64_t at = 0;
#pragma unroll
               for (int p = 0; p < kEdgeParts; ++p) {
                 const bool here = mine && owner / kEdgeNodes == p;
                 const uint64_t kept = __ballot(here);
                 const int before = (int)__builtin_amdgcn_mbcnt_hi(
                     (uint32_t)(kept >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)kept, 0u));
                 if (here) at = pos[p] + before;
                 pos[p] += __popcll(kept);
               }
               if (mine && at < max_edges) {
                 out_parent[at] = parent;
                 out_child[at] = remap[child];
                 out_action[at] = actions != nullptr ? actions[edge] : (int16_t)0;
               }
             });
}

hipError_t launch_bfs_subtree(const int32_t* row_ptr, const int32_t* col, int num_edges,
                              int root, int max_nodes, uint8_t* in_subtree, int32_t* remap,
                              int32_t* count, int32_t* ws, hipStream_t st) {
  int32_t* queue = ws;
  int32_t* claim = ws + max_nodes;
  if (max_nodes > kBfsClearHere) {
    const int blocks = (int)std::min<int64_t>(1024, ((int64_t)max_nodes + 255) / 256);
    hipLaunchKernelGGL(bfs_clear_kernel, dim3(blocks), dim3(256), 0, st, root, max_nodes,
                       in_subtree, remap, claim, queue);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(bfs_subtree_kernel, dim3(1), dim3(kBfsThreads), 0, st, row_ptr, col,
                     num_edges, root, max_nodes, in_subtree, remap, count, queue, claim);
  return hipGetLastError();
}

hipError_t launch_extract_edges(const int32_t* row_ptr, const int32_t* col, const int16_t* actions,
                                int num_edges, const uint8_t* in_subtree, const int32_t* remap,
                                int num_nodes, int max_edges, int32_t* out_parent,
                                int32_t* out_child, int16_t* out_action, int32_t* edge_count,
                                int32_t* ws, hipStream_t st) {
  // (OMQ_EDGES_WORKSPACE_INTS: local and chunk_tot, and one so that it is never empty)
  static_assert(kEdgeNodes == 16 && kEdgeChunk == 256, "OMQ_EDGES_WORKSPACE_INTS");
  const int chunks = (int)(((int64_t)num_nodes + kEdgeChunk - 1) / kEdgeChunk);
  const int blocks = (chunks + kEdgeParts - 1) / kEdgeParts;
  int32_t* local = ws;
  int32_t* chunk_tot = ws + ((int64_t)num_nodes + kEdgeNodes - 1) / kEdgeNodes;
  hipError_t e = hipSuccess;
  if (blocks > 0) {
    hipLaunchKernelGGL(edges_count_kernel, dim3(blocks), dim3(kEdgeThreads), 0, st, row_ptr, col,
                       num_edges, in_subtree, num_nodes, local, chunk_tot);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(edges_scan_kernel, dim3(1), dim3(kEdgeThreads), 0, st, chunk_tot, chunks,
                     edge_count);
  e = hipGetLastError();
  if (e != hipSuccess || blocks == 0) return e;
  hipLaunchKernelGGL(edges_write_kernel, dim3(blocks), dim3(kEdgeThreads), 0, st, row_ptr, col,
                     actions, num_edges, in_subtree, remap, num_nodes, max_edges, local, chunk_tot,
                     out_parent, out_child, out_action);
  return hipGetLastError();
}

}  // namespace omq
