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

// Counts (and value sums) per node gathered in a workgroup's LDS before they go to memory: a
// hash table of the nodes its paths share.  An atomic on one address of device memory costs
// about 24 ns after the one before it (each is carried out past the XCD's own L2), and every path
// adds to its root, so the nodes of the first levels set the time; a workgroup adds to each of
// them once.  A node that finds no slot within kProbes is added to memory directly.
template <bool SUMS>
struct NodeTable {
  static constexpr int kSlots = 1024;
  static constexpr int kProbes = 8;
  static constexpr unsigned long long kFree = ~0ull;
  unsigned long long key[kSlots];  // the node's index in the forest's arrays
  int count[kSlots];
  float sum[SUMS ? kSlots : 1];

  __device__ void clear(int tid, int threads) {
    for (int i = tid; i < kSlots; i += threads) {
      key[i] = kFree;
      count[i] = 0;
      if (SUMS) sum[i] = 0.0f;
    }
  }
  __device__ bool add(int64_t node, int c, float v) {
    const unsigned long long k = (unsigned long long)node;
    uint32_t h = ((uint32_t)k * 0x9E3779B1u) >> 22;  // (10 bits: kSlots)
    for (int i = 0; i < kProbes; ++i, h = (h + 1) & (kSlots - 1)) {
      unsigned long long at = key[h];
      if (at == kFree) at = atomicCAS(&key[h], kFree, k);
      if (at == kFree || at == k) {
        atomicAdd(&count[h], c);
        if (SUMS) __hip_atomic_fetch_add(&sum[h], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return true;
      }
    }
    return false;
  }
  __device__ void flush(int tid, int threads, int32_t* counts, float* sums) {
    for (int i = tid; i < kSlots; i += threads) {
      const unsigned long long k = key[i];
      if (k == kFree) continue;
      atomicAdd(&counts[k], count[i]);
      if (SUMS) unsafeAtomicAdd(&sums[k], sum[i]);
    }
  }
};

// reference-style backup over an explicit path matrix (vectorized_backup_kernel), one thread per
// path.  The nodes of the first kSharedDepth levels go through the workgroup's table, the deeper
// ones, which few paths share, straight to memory.  32768 paths of 32 trees (depth 6 on average):
// 58.6 -> 14.1 us; 49152 paths of one tree, with the virtual loss on and off: 1945 -> 142 us.
// Workgroups of 512 or 1024 threads add to a root less often (the one tree 92 and 66 us) but wait
// longer at its LDS address: 4096 paths of 8 trees 16.8 us with 256, 22.8 and 35.1 us.  Adding a
// wave's equal nodes up first changed neither.
constexpr int kPathThreads = 256;
constexpr int kSharedDepth = 8;

__global__ __launch_bounds__(kPathThreads) void paths_backup_kernel(
    omq_forest f, const int32_t* paths, const int32_t* plen, const int32_t* tree_of,
    const float* values, int batch, int max_depth, int sign_mode) {
  __shared__ NodeTable<true> table;
  const int tid = threadIdx.x;
  table.clear(tid, kPathThreads);
  __syncthreads();
  const int b = blockIdx.x * kPathThreads + tid;
  const int t = b < batch && tree_of ? tree_of[b] : 0;
  if (b < batch && t >= 0 && t < f.num_trees) {  // entries naming no tree are skipped
    const int64_t tb = (int64_t)t * f.capacity;
    // entries d < min(length, max_depth); the leaf-positive sign counts the distance from the
    // leaf by the length as given (vectorized_backup_kernel, mcts_kernels.cu:142-146), also for a
    // length past the row
    const int Lp = plen[b];
    const int L = min(Lp, max_depth);
    const float v = values[b];
    const int32_t* row = paths + (int64_t)b * max_depth;
    constexpr int kB = 4;  // entries whose loads are in flight together
    for (int d0 = 0; d0 < L; d0 += kB) {
      int xs[kB];
#pragma unroll
      for (int j = 0; j < kB; ++j) xs[j] = d0 + j < L ? row[d0 + j] : -1;
#pragma unroll
      for (int j = 0; j < kB; ++j) {
        const int x = xs[j];
        if (x < 0 || x >= f.capacity) continue;  // -1 padding and out-of-range entries
        const int d = d0 + j;
        const int e = sign_mode == OMQ_SIGN_LEAF_POSITIVE ? (Lp - 1 - d) : d;
        const float sv = (e & 1) ? -v : v;
        if (d >= kSharedDepth || !table.add(tb + x, 1, sv)) {
          atomicAdd(&f.visit_counts[tb + x], 1);
          unsafeAtomicAdd(&f.value_sums[tb + x], sv);
        }
      }
    }
  }
  __syncthreads();
  table.flush(tid, kPathThreads, f.visit_counts, f.value_sums);
}

// delta per listed node; a workgroup takes kVlPer nodes per thread through its table (the path
// nodes of the 32768 paths above: 25.0 -> 7.2 us)
constexpr int kVlPer = 4;
__global__ __launch_bounds__(kPathThreads) void virtual_loss_kernel(omq_forest f,
                                                                    const int32_t* nodes,
                                                                    const int32_t* tree_of,
                                                                    int count, int delta) {
  __shared__ NodeTable<false> table;
  const int tid = threadIdx.x;
  const int64_t i0 = (int64_t)blockIdx.x * (kPathThreads * kVlPer) + tid;
  int xs[kVlPer], ts[kVlPer];
#pragma unroll
  for (int j = 0; j < kVlPer; ++j) {
    const int64_t i = i0 + j * kPathThreads;
    xs[j] = i < count ? nodes[i] : -1;
    ts[j] = i < count && tree_of ? tree_of[i] : 0;
  }
  table.clear(tid, kPathThreads);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kVlPer; ++j) {
    const int x = xs[j], t = ts[j];
    if (x < 0 || x >= f.capacity || t < 0 || t >= f.num_trees) continue;
    const int64_t node = (int64_t)t * f.capacity + x;
    if (!table.add(node, delta, 0.0f)) atomicAdd(&f.visit_counts[node], delta);
  }
  __syncthreads();
  table.flush(tid, kPathThreads, f.visit_counts, nullptr);
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
  hipLaunchKernelGGL(paths_backup_kernel, dim3((batch + kPathThreads - 1) / kPathThreads),
                     dim3(kPathThreads), 0, st, f, paths, plen, tree_of, values, batch, max_depth,
                     sign_mode);
  return hipGetLastError();
}

hipError_t launch_virtual_loss(const omq_forest& f, const int32_t* nodes, const int32_t* tree_of,
                               int count, int delta, hipStream_t st) {
  constexpr int kPer = kPathThreads * kVlPer;
  hipLaunchKernelGGL(virtual_loss_kernel, dim3(count / kPer + (count % kPer != 0)),
                     dim3(kPathThreads), 0, st, f, nodes, tree_of, count, delta);
  return hipGetLastError();
}

hipError_t launch_reset(const omq_forest& f, hipStream_t st) {
  hipLaunchKernelGGL(reset_kernel, dim3((f.num_trees + 255) / 256), dim3(256), 0, st, f);
  return hipGetLastError();
}

}  // namespace omq
