// Backup with virtual-loss revert (gfx950).
//
// Sequential definition: for every simulation s in order and every node x on its path,
//   N[x] = N[x] - VL + 1                      (cython_tree_optimized.pyx:222)
//   W[x] = W[x] + sign(x) * v(leaf of s)      (optimized_wave_search.py:472-483: leaf +v,
//                                              parent -v, ...; or root-positive, pyx:216-224)
// Ordered mode uses the group log of the selection: a node appears in exactly one group per
// wave, and the group's members are in simulation order, so folding the members' signed
// values into W[x] in that order gives the sequential result bit for bit, with no atomics.
// Small groups are folded by one lane each; groups with more than kBigGroup members by the
// whole wave (lanes load, one running sum through v_readlane).
#include "backup_groups.h"

namespace omq {

// signed value per simulation (sim_value_at)
__global__ void sim_value_kernel(omq_forest f, omq_wave w, int W, int sign_mode) {
  int bx = blockIdx.x, by = blockIdx.y;
  xcd_block(&bx, &by);  // one contiguous run of blocks (leaves of few trees) per XCD
  const int s = bx * blockDim.x + threadIdx.x;
  if (s >= W) return;
  sim_value_at(f, w, by, s, sign_mode);
}

template <bool FUSED>
__global__ __launch_bounds__(kBackupThreads) void backup_groups_kernel(omq_forest f, omq_wave w,
                                                                       int vli, int sign_mode) {
  int bx = blockIdx.x, by = blockIdx.y;
  xcd_block(&bx, &by);  // one contiguous run of blocks (leaves of few trees) per XCD
  backup_groups_block<FUSED>(f, w, vli, sign_mode, bx, by, (int)gridDim.x);
}

// atomic mode: one lane per simulation walks its path with float atomics (order not fixed)
__global__ void backup_atomic_kernel(omq_forest f, omq_wave w, int W, int vli) {
  const int t = blockIdx.y;
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= W) return;
  const int64_t tb = (int64_t)t * f.capacity;
  const int64_t wb = (int64_t)t * w.max_wave;
  const int L = w.path_len[wb + s];
  const float v = w.sim_value[wb + s];
  const int32_t* path = w.paths + (wb + s) * w.max_depth;
  for (int d = 0; d < L; ++d) {
    const int x = path[d];
    atomicAdd(&f.visit_counts[tb + x], 1 - vli);
    unsafeAtomicAdd(&f.value_sums[tb + x], (d & 1) ? -v : v);
  }
}

// Counts (and value sums) per node gathered in a workgroup's LDS before they go to memory.  An
// atomic on one address of device memory costs about 24 ns after the one before it (each is carried
// out past the XCD's own L2), and every path adds to its root, so the nodes of the first levels set
// the time; a workgroup adds to each of them once.
// The workgroup's entries (kEntries nodes) meet in a table of slots without probing or compare-and-
// swap: every entry writes its number to its node's slot, and after a barrier the entries whose
// node is that of the number left there add up in the slot.  The entry left (the slot's owner) adds
// the result to memory; an entry that finds another node's number adds to memory directly.  A node
// that no other entry shares so costs a few LDS accesses more than a direct add and keeps its place
// in the list's order (a table probed by compare-and-swap and written out in its own order took
// up to 4.7 us more than direct adds on such lists, and 159 against 11.2 us on 4M nodes in order).
template <bool SUMS, int kEntries>
struct NodeTable {
  static constexpr int kBits = 11;
  static constexpr int kSlots = 1 << kBits;
  static_assert(kEntries <= 65536, "entries are numbered in 16 bits");
  int64_t node[kEntries];  // an entry's node, as an index into the forest's arrays
  uint16_t left[kSlots];   // the number of one of the slot's entries
  int count[kSlots];
  float sum[SUMS ? kSlots : 1];

  __device__ static int slot(int64_t nd) {
    return (int)(((uint32_t)nd * 0x9E3779B1u) >> (32 - kBits));
  }
  // before the first barrier
  __device__ void enter(int e, int64_t nd) {
    const int h = slot(nd);
    node[e] = nd;
    left[h] = (uint16_t)e;
    count[h] = 0;
    if (SUMS) sum[h] = 0.0f;
  }
  // between the barriers (an entry's owner stays what it is; the callers read all their owners
  // before any of the owners' nodes, and those before any add, so that the reads overlap)
  __device__ int owner(int64_t nd) const { return left[slot(nd)]; }
  __device__ void add(int64_t nd, int c, float v) {
    const int h = slot(nd);
    atomicAdd(&count[h], c);
    if (SUMS) __hip_atomic_fetch_add(&sum[h], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  // after the second barrier, by the slot's owner
  __device__ void flush(int64_t nd, int32_t* counts, float* sums) const {
    const int h = slot(nd);
    atomicAdd(&counts[nd], count[h]);
    if (SUMS) unsafeAtomicAdd(&sums[nd], sum[h]);
  }
};

// reference-style backup over an explicit path matrix (vectorized_backup_kernel), one thread per
// path.  The nodes of the first kSharedDepth levels go through the workgroup's table, the deeper
// ones, which few paths share, straight to memory, in one add where all of a wave's paths are on the
// same node (a line that every path follows: 64 paths of 64 such nodes 134 -> 22 us, 8192 of them
// 4173 -> 74).  A thread enters its deepest node first: where two nodes of a workgroup meet in a slot,
// the shallower one, which more paths share, mostly keeps it (49152 paths of one tree: 175 us the
// other way round, 26 us so).
// Up to kFewPaths paths, one wave, there is no table (8 nodes each: 3.5 us, 4.1 with it and one wave);
// up to kSomePaths a workgroup is one wave, whose table's LDS accesses, which take most of a small
// call, are a quarter of four waves'.  Device time a call, an atomic per entry / workgroups of 64 /
// of 256, 8 nodes a path, in a tree whose nodes have two children and with no node shared: 512
// paths 19.8 / 4.6 / 7.5 us and 5.3 / 4.4 / 7.4; 4096 132 / 7.6 / 10 and 5.5 / 5.2 / 8; 8192 260 / 11.7 /
// 9.9 and 5.9 / 6.6 / 8.7; 16384 514 / 19.6 / 12.7 and 7.6 / 9.2 / 11.2; 32768 1040 / 36.6 / 18.5 and
// 13.0 / 15.6 / 16.5.  With six children 8192 paths of 16 nodes 162 / 14.6 / 19.0.
constexpr int kPathThreads = 256;
constexpr int kSharedDepth = 8;
constexpr int kFewPaths = kWave;
constexpr int kSomePaths = 8192;

template <bool SHARED, int NT>
__global__ __launch_bounds__(NT) void paths_backup_kernel(
    omq_forest f, const int32_t* paths, const int32_t* plen, const int32_t* tree_of,
    const float* values, int batch, int max_depth, int sign_mode) {
  constexpr int kTabled = SHARED ? kSharedDepth : 0;
  __shared__ NodeTable<true, SHARED ? NT * kSharedDepth : 1> table;
  const int tid = threadIdx.x;
  const int b = blockIdx.x * NT + tid;
  const int t = b < batch && tree_of ? tree_of[b] : 0;
  const bool on = b < batch && t >= 0 && t < f.num_trees;  // entries naming no tree are skipped
  const int64_t tb = (int64_t)t * f.capacity;
  // entries d < min(length, max_depth); the leaf-positive sign counts the distance from the
  // leaf by the length as given (vectorized_backup_kernel, mcts_kernels.cu:142-146), also for a
  // length past the row
  const int Lp = on ? plen[b] : 0;
  const int L = min(Lp, max_depth);
  const float v = on ? values[b] : 0.0f;
  const int32_t* row = paths + (int64_t)b * max_depth;
  auto signed_value = [&](int d) {
    const int e = sign_mode == OMQ_SIGN_LEAF_POSITIVE ? (Lp - 1 - d) : d;
    return (e & 1) ? -v : v;
  };
  auto to_memory = [&](int64_t node, float sv) {
    atomicAdd(&f.visit_counts[node], 1);
    unsafeAtomicAdd(&f.value_sums[node], sv);
  };
  int xs[kSharedDepth];  // (-1 padding and out-of-range entries are skipped)
  int own[kSharedDepth];  // their slots' owners
  if constexpr (SHARED) {
#pragma unroll
    for (int d = 0; d < kSharedDepth; ++d) xs[d] = d < L ? row[d] : -1;
#pragma unroll
    for (int d = kSharedDepth - 1; d >= 0; --d) {
      if (xs[d] >= f.capacity) xs[d] = -1;
      if (xs[d] >= 0) table.enter(d * NT + tid, tb + xs[d]);
    }
    __syncthreads();
    bool taken[kSharedDepth];
#pragma unroll
    for (int d = 0; d < kSharedDepth; ++d) own[d] = xs[d] >= 0 ? table.owner(tb + xs[d]) : 0;
#pragma unroll
    for (int d = 0; d < kSharedDepth; ++d) taken[d] = table.node[own[d]] == tb + xs[d];
#pragma unroll
    for (int d = 0; d < kSharedDepth; ++d) {
      if (xs[d] < 0) continue;
      if (taken[d])
        table.add(tb + xs[d], 1, signed_value(d));
      else
        to_memory(tb + xs[d], signed_value(d));
    }
  }
  constexpr int kB = 4;  // deeper entries whose loads are in flight together
  for (int d0 = kTabled; __any(d0 < L); d0 += kB) {
    int ys[kB];
#pragma unroll
    for (int j = 0; j < kB; ++j) ys[j] = d0 + j < L ? row[d0 + j] : -1;
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      const bool in = ys[j] >= 0 && ys[j] < f.capacity;
      const uint64_t lanes = __ballot(in);
      if (lanes == 0) continue;
      const int64_t node = tb + ys[j];
      const int64_t one = __shfl(node, lowest_lane(lanes), kWave);
      const float sv = in ? signed_value(d0 + j) : 0.0f;
      if (__all(!in || node == one) && __popcll(lanes) > 1) {
        const float sum = wave_sum_canonical(sv);
        if (lane_id() == 0) {
          atomicAdd(&f.visit_counts[one], __popcll(lanes));
          unsafeAtomicAdd(&f.value_sums[one], sum);
        }
      } else if (in) {
        to_memory(node, sv);
      }
    }
  }
  if constexpr (SHARED) {
    __syncthreads();
#pragma unroll
    for (int d = 0; d < kSharedDepth; ++d)
      if (xs[d] >= 0 && own[d] == d * NT + tid)
        table.flush(tb + xs[d], f.visit_counts, f.value_sums);
  }
}

// delta per listed node; a workgroup takes kVlPer nodes per thread through its table, but for 64
// consecutive nodes in order, whose add is coalesced already (4M nodes in order: 15.6 us through the
// table, 11.7 so, 11.2 without a table at all).
// Device time a call, against an atomic per entry: the path nodes of the 32768 paths above 27.6 ->
// 6.6 us, of the 49152 588 -> 38; 1000 entries of one node 13.0 -> 2.2, of 1000 nodes 2.2 -> 2.4.
// One node per thread up to kVlShort entries: at most 64 workgroups, so a node that all of them
// share costs 1.5 us, and a workgroup of a quarter of the entries is done sooner (1000 to 16000
// entries 2.2-2.7 us, 3.6-4.2 with four nodes per thread; 225k entries of one tree 59 us with one,
// 38 with four).
constexpr int kVlShort = 64 * kPathThreads;

template <int kVlPer>
__global__ __launch_bounds__(kPathThreads) void virtual_loss_kernel(omq_forest f,
                                                                    const int32_t* nodes,
                                                                    const int32_t* tree_of,
                                                                    int count, int delta) {
  __shared__ NodeTable<false, kPathThreads * kVlPer> table;
  const int tid = threadIdx.x;
  const int64_t i0 = (int64_t)blockIdx.x * (kPathThreads * kVlPer) + tid;
  int64_t nd[kVlPer];  // -1: none
#pragma unroll
  for (int j = 0; j < kVlPer; ++j) {
    const int64_t i = i0 + j * kPathThreads;
    const int x = i < count ? nodes[i] : -1;
    const int t = i < count && tree_of ? tree_of[i] : 0;
    const bool on = x >= 0 && x < f.capacity && t >= 0 && t < f.num_trees;
    nd[j] = on ? (int64_t)t * f.capacity + x : -1;
    const int64_t from = (int64_t)__shfl(nd[j], 0, kWave);
    if (__all(on && nd[j] == from + lane_id())) {
      atomicAdd(&f.visit_counts[nd[j]], delta);
      nd[j] = -1;
    }
  }
#pragma unroll
  for (int j = 0; j < kVlPer; ++j)
    if (nd[j] >= 0) table.enter(j * kPathThreads + tid, nd[j]);
  __syncthreads();
  int own[kVlPer];
  bool taken[kVlPer];
#pragma unroll
  for (int j = 0; j < kVlPer; ++j) own[j] = nd[j] >= 0 ? table.owner(nd[j]) : 0;
#pragma unroll
  for (int j = 0; j < kVlPer; ++j) taken[j] = table.node[own[j]] == nd[j];
#pragma unroll
  for (int j = 0; j < kVlPer; ++j) {
    if (nd[j] < 0) continue;
    if (taken[j])
      table.add(nd[j], delta, 0.0f);
    else
      atomicAdd(&f.visit_counts[nd[j]], delta);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kVlPer; ++j)
    if (nd[j] >= 0 && own[j] == j * kPathThreads + tid)
      table.flush(nd[j], f.visit_counts, nullptr);
}

__global__ void reset_kernel(omq_forest f) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= f.num_trees) return;
  const int64_t r = (int64_t)t * f.capacity;
  f.visit_counts[r] = 1;
  f.value_sums[r] = 0.0f;
  f.priors[r] = 1.0f;
  f.parents[r] = -1;
  f.first_child[r] = -1;
  f.num_children[r] = 0;
  f.actions[r] = -1;
  f.num_nodes[t] = 1;
}

// ---------------------------------------------------------------------------------------
hipError_t launch_backup(const omq_forest& f, const omq_wave& w, int W, float virtual_loss,
                         int sign_mode, int w_mode, hipStream_t st) {
  const int vli = (int)virtual_loss;
  dim3 g1((W + 255) / 256, f.num_trees);
  const bool fused = w_mode != OMQ_WACC_ATOMIC && W <= kFuseMaxWave;
  if (!fused) {
    hipLaunchKernelGGL(sim_value_kernel, g1, dim3(256), 0, st, f, w, W, sign_mode);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (w_mode == OMQ_WACC_ATOMIC) {
    hipLaunchKernelGGL(backup_atomic_kernel, g1, dim3(256), 0, st, f, w, W, vli);
    return hipGetLastError();
  }
  // (the group count is on the device)
  const int blocks = backup_group_blocks(W);
  if (fused)
    hipLaunchKernelGGL(backup_groups_kernel<true>, dim3(blocks, f.num_trees),
                       dim3(kBackupThreads), 0, st, f, w, vli, sign_mode);
  else
    hipLaunchKernelGGL(backup_groups_kernel<false>, dim3(blocks, f.num_trees),
                       dim3(kBackupThreads), 0, st, f, w, vli, sign_mode);
  return hipGetLastError();
}

hipError_t launch_paths_backup(const omq_forest& f, const int32_t* paths, const int32_t* plen,
                               const int32_t* tree_of, const float* values, int batch,
                               int max_depth, int sign_mode, hipStream_t st) {
  const int threads = batch <= kSomePaths ? kWave : kPathThreads;
  const auto kernel = batch <= kFewPaths    ? paths_backup_kernel<false, kWave>
                      : batch <= kSomePaths ? paths_backup_kernel<true, kWave>
                                            : paths_backup_kernel<true, kPathThreads>;
  hipLaunchKernelGGL(kernel, dim3(batch / threads + (batch % threads != 0)), dim3(threads), 0, st,
                     f, paths, plen, tree_of, values, batch, max_depth, sign_mode);
  return hipGetLastError();
}

hipError_t launch_virtual_loss(const omq_forest& f, const int32_t* nodes, const int32_t* tree_of,
                               int count, int delta, hipStream_t st) {
  auto blocks = [&](int per) { return dim3(count / per + (count % per != 0)); };
  if (count <= kVlShort)
    hipLaunchKernelGGL(virtual_loss_kernel<1>, blocks(kPathThreads), dim3(kPathThreads), 0, st, f,
                       nodes, tree_of, count, delta);
  else
    hipLaunchKernelGGL(virtual_loss_kernel<4>, blocks(4 * kPathThreads), dim3(kPathThreads), 0, st,
                       f, nodes, tree_of, count, delta);
  return hipGetLastError();
}

hipError_t launch_reset(const omq_forest& f, hipStream_t st) {
  hipLaunchKernelGGL(reset_kernel, dim3((f.num_trees + 255) / 256), dim3(256), 0, st, f);
  return hipGetLastError();
}

}  // namespace omq
