// Gomoku positions of the unique leaves of a wave: terminal check and feature planes (gfx950).
//
// The reference decides after every move whether a child state is terminal.
// CPUGameStates.apply_actions (python/mcts/cpu/cpu_game_states.py:352-412) calls
// FastTerminalChecker._check_gomoku_terminal_cpu with last_move=None, which is a full-board
// scan (python/mcts/utils/fast_terminal_check.py:132-232):
//   - cells are visited in row-major order; at an occupied cell, the directions horizontal,
//     vertical, down-right and down-left are tried in that order;
//   - a direction counts when there is room for five cells (col <= bs-5 / row <= bs-5 / both /
//     row <= bs-5 and col >= 4) and all five belong to the cell's player;
//   - the first cell with a counting direction names the winner;
//   - with use_renju, a five of player 1 that continues on either side (an overline) does not
//     count, and it ends the scan of that cell: the reference's `continue` skips the
//     remaining directions of the cell;
//   - a full board without a five is a draw.
// The driver does not expand a terminal leaf (python/mcts/cpu/optimized_wave_search.py:374-376),
// but it still backs up the evaluator's value for it.
//
// Here a leaf's position is never stored.  It is rebuilt from the root board and the moves on
// the leaf's path, colours alternating from the root's player to move, by one wavefront per unique
// leaf: as row masks in registers, one row of either player per lane, whose fives are shifts of
// whole rows, or (small boards, other stones than 1 and 2) as a board in LDS that is scanned
// cell-parallel, lane l taking cells l, l+64, ...  Either way the row-major first winning cell names
// the winner.  A terminal leaf gets ulegal = 0, which keeps omq_expand from expanding it.
#include "omq_common.h"

namespace omq {

// Rebuilds the position of unique leaf u of tree t into the wave's LDS board b: the root board
// with the path's moves played in alternating colours from the root's player to move.  Returns
// the path length L (the leaf has L-1 moves on it).  *rp_out receives the root's player to
// move: root_player[t], or 1 when the root board holds an even number of stones, else 2
// (python/mcts/core/mcts.py:1503-1508); *stones_out the root board's stone count.
// AHEAD: the path's first entries (most paths; one line of the row) are loaded with its length
// instead of after it, and the board under the path's loads.  That is one of three dependent
// rounds less for a kernel that waits for them (the feature planes: 512 slots 9.0 -> 6.0 us in the
// kernel trace, 16384 slots 52.3 -> 48.9 us); the rule kernels gain nothing.
template <bool AHEAD>
__device__ inline int rebuild_leaf_board(const omq_forest& f, const omq_wave& w,
                                         const int8_t* root_boards, const int32_t* root_player,
                                         int t, int u, int cells, int8_t* b, int* rp_out,
                                         int* stones_out) {
  const int lane = lane_id();
  const int8_t* rb = root_boards + (int64_t)t * cells;
  int L = 0, a_lo = -1, a_hi = -1;
  if constexpr (AHEAD) {
    constexpr int kAhead = 16;
    const int64_t s0 = (int64_t)t * w.max_wave + w.ufirst[(int64_t)t * w.max_wave + u];
    const int64_t tb = (int64_t)t * f.capacity;
    const int32_t* path = w.paths + s0 * w.max_depth;
    const bool ahead = lane + 1 < min(kAhead, w.max_depth);
    L = w.path_len[s0];
    int node = ahead ? path[lane + 1] : 0;  // (past the path: unused)
    if (!ahead && lane + 1 < L) node = path[lane + 1];
    if (lane + 1 < L) a_lo = f.actions[tb + node];
    if (lane + 65 < L) a_hi = f.actions[tb + path[lane + 65]];
  }
  int stones = 0;
  for (int i = lane; i < cells; i += kWave) {
    const int8_t v = rb[i];
    b[i] = v;
    stones += v != 0;
  }
  stones = wave_sum_i(stones);
  if constexpr (!AHEAD) {
    const int s0 = w.ufirst[(int64_t)t * w.max_wave + u];
    L = load_path_actions(f, w, t, s0, &a_lo, &a_hi);
  }
  const int rp = root_player != nullptr ? root_player[t] : ((stones & 1) == 0 ? 1 : 2);
  wave_sync();
  // move j (0-based, depth j+1) is played by rp when j is even; lane l holds moves l and l+64
  const int8_t mine = (int8_t)((lane & 1) == 0 ? rp : 3 - rp);
  if (lane + 1 < L && a_lo >= 0 && a_lo < cells) b[a_lo] = mine;
  if (lane + 65 < L && a_hi >= 0 && a_hi < cells) b[a_hi] = mine;
  wave_sync();
  *rp_out = rp;
  *stones_out = stones;
  return L;
}

// LDS of a wave of the rule kernels: a board in bytes, or row words for two players.
__host__ __device__ inline int rule_lds_per_wave(int cells) {
  const int words = 2 * (2 * ((OMQ_MAX_ROW + kWave - 1) / kWave) + 2) * 4;
  const int board = (cells + 15) & ~15;
  return board > words ? board : (words + 15) & ~15;
}

// ---- boards as row masks ----------------------------------------------------------------------
// Lane r holds row r of a board as bits (bit c: column c), at most 22 rows and columns.  The rules
// are then shifts of whole rows: a few dozen instructions a leaf, where the scan of the cells
// from LDS bytes takes up to 20 dependent reads per cell and direction.
constexpr int kRowWords = 2 * ((OMQ_MAX_ROW + kWave - 1) / kWave) + 2;  // and a pad

// The set of cells as rows, from one ballot per 64 cells in the wave's LDS words.
struct RowBits {
  uint32_t* words;  // [kRowWords] of the wave's LDS
  __device__ void clear() const {
    if (lane_id() < kRowWords) words[lane_id()] = 0u;
  }
  __device__ void put(int c0, uint64_t cells64) const {  // cells c0 .. c0 + 63
    if (lane_id() < 2)
      words[(c0 >> 5) + lane_id()] = lane_id() == 0 ? (uint32_t)cells64
                                                    : (uint32_t)(cells64 >> 32);
  }
  __device__ uint32_t row(int bs) const {  // (after wave_sync)
    const int r = lane_id();
    if (r >= bs) return 0u;
    const int o = r * bs;
    const uint64_t x = (uint64_t)words[(o >> 5) + 1] << 32 | words[o >> 5];
    return (uint32_t)(x >> (o & 31)) & ((1u << bs) - 1u);
  }
};

// Calls stone(move, bit) for the path's moves on the board in order: bit is the move's column in
// the lane of its row, 0 in the others.
template <class Stone>
__device__ inline void each_move(int L, int a_lo, int a_hi, int cells, int bs, Stone stone) {
  const int lane = lane_id();
  const int r_lo = a_lo / bs, r_hi = a_hi / bs;
  const int c_lo = a_lo - r_lo * bs, c_hi = a_hi - r_hi * bs;
  for (int j = 0; j + 1 < L; ++j) {
    const bool lo = j < kWave;
    const int jj = j & (kWave - 1);
    const int a = lo ? readlane_i(a_lo, jj) : readlane_i(a_hi, jj);
    if (a < 0 || a >= cells) continue;
    const int r = lo ? readlane_i(r_lo, jj) : readlane_i(r_hi, jj);
    const int c = lo ? readlane_i(c_lo, jj) : readlane_i(c_hi, jj);
    stone(j, lane == r ? 1u << c : 0u);
  }
}

// Row l + k of the rows in m (0 past the board: lanes past it hold 0).
__device__ inline uint32_t row_at(uint32_t m, int k) {
  const int l = lane_id() + k;
  const uint32_t x = (uint32_t)__shfl((int)m, l & (kWave - 1), kWave);
  return l >= 0 ? x : 0u;
}

// The cells of the player's rows m where a counting five starts (the file comment's rule; over:
// renju's player 1, whose overlines end the scan of their cell).
__device__ inline uint32_t five_starts(uint32_t m, bool over) {
  const uint32_t d1 = row_at(m, 1), d2 = row_at(m, 2), d3 = row_at(m, 3), d4 = row_at(m, 4);
  const uint32_t h = m & m >> 1 & m >> 2 & m >> 3 & m >> 4;
  const uint32_t v = m & d1 & d2 & d3 & d4;
  const uint32_t dr = m & d1 >> 1 & d2 >> 2 & d3 >> 3 & d4 >> 4;
  const uint32_t dl = m & d1 << 1 & d2 << 2 & d3 << 3 & d4 << 4;
  if (!over) return h | v | dr | dl;
  const uint32_t d5 = row_at(m, 5), u1 = row_at(m, -1);
  uint32_t win = 0u, ended = 0u;  // (the directions in the scan's order)
  auto dir = [&](uint32_t five, uint32_t longer) {
    const uint32_t f = five & ~win & ~ended;
    ended |= f & longer;
    win |= f & ~longer;
  };
  dir(h, m >> 5 | m << 1);
  dir(v, d5 | u1);
  dir(dr, d5 >> 5 | u1 << 1);
  dir(dl, d5 << 5 | u1 >> 1);
  return win;
}

// The terminal code of the position in the wave's LDS board b by a scan of its cells.
__device__ inline int scan_terminal(const int8_t* b, int cells, int bs, int rule) {
  const int lane = lane_id();
  constexpr int dr[4] = {0, 1, 1, 1};
  constexpr int dc[4] = {1, 0, 1, -1};
  int win = 0x7FFFFFFF;
  int empty = 0;
  for (int cell = lane; cell < cells; cell += kWave) {
    const int p = b[cell];
    if (p == 0) {
      ++empty;
      continue;
    }
    const int r = cell / bs, c = cell - (cell / bs) * bs;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int re = r + 4 * dr[d], ce = c + 4 * dc[d];
      if (re >= bs || ce < 0 || ce >= bs) continue;  // no room for five in this direction
      bool five = true;
#pragma unroll
      for (int k = 1; k < 5; ++k) five = five && b[(r + k * dr[d]) * bs + c + k * dc[d]] == p;
      if (!five) continue;
      if (rule == OMQ_RULE_RENJU && p == 1) {
        const int rn = r + 5 * dr[d], cn = c + 5 * dc[d];
        const int rq = r - dr[d], cq = c - dc[d];
        const bool after = rn < bs && cn >= 0 && cn < bs && b[rn * bs + cn] == p;
        const bool before = rq >= 0 && cq >= 0 && cq < bs && b[rq * bs + cq] == p;
        if (after || before) break;  // overline: the reference skips the rest of this cell
      }
      win = min(win, cell);
      break;
    }
  }
  win = (int)~wave_max_u32(~(uint32_t)win);  // wave min
  empty = wave_sum_i(empty);
  int code = OMQ_TERM_NONE;
  if (win != 0x7FFFFFFF) code = b[win];
  else if (empty == 0) code = OMQ_TERM_DRAW;
  return code;
}

// One wavefront per unique leaf, on the row masks of the two players; a board with other stones
// than 1 and 2, or another root player, is scanned cell by cell as the reference scans it.  64
// trees of 256 leaves, 15x15: 13.0 us with the scan for every board, 10.3 us so; 16 trees of 32
// leaves 5.8 and 4.2 us.
// A board of one cell per lane is scanned too, and so is one of two cells per lane in large waves,
// where the work counts and not its latency.  Device time, row masks / scan: 32 trees of 1024 leaves
// 5x5 16.5 / 12.3 us, 8x8 16.4 / 13.0, 9x9 17.1 / 15.5, 11x11 16.4 / 16.6, 12x12 17.0 / 18.6; 32 of 256
// 9x9 6.3 / 5.9; 16 of 64 9x9 4.1 / 4.4.
constexpr int kRuleManySlots = 8192;

__global__ void gomoku_terminal_kernel(omq_forest f, omq_wave w, const int8_t* root_boards,
                                       const int32_t* root_player, int rule, int bs, bool scan,
                                       int32_t* uterm) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int cells = bs * bs;
  const int stride = rule_lds_per_wave(cells);
  const int t = blockIdx.y;
  const int wave = threadIdx.x / kWave;
  const int u = blockIdx.x * (blockDim.x / kWave) + wave;
  const int lane = lane_id();
  const int64_t wb = (int64_t)t * w.max_wave;
  if (u >= w.ucount[t]) return;
  auto scanned = [&]() {
    int8_t* b = reinterpret_cast<int8_t*>(smem + (size_t)wave * stride);
    int rp, stones;
    rebuild_leaf_board<false>(f, w, root_boards, root_player, t, u, cells, b, &rp, &stones);
    return scan_terminal(b, cells, bs, rule);
  };
  const int s0 = w.ufirst[wb + u];
  int a_lo, a_hi;
  const int L = load_path_actions(f, w, t, s0, &a_lo, &a_hi);
  if (L <= 1) {  // the root position itself is not checked (the reference never flags it)
    if (uterm != nullptr && lane == 0) uterm[wb + u] = OMQ_TERM_NONE;
    return;
  }
  if (scan) {
    const int code = scanned();
    if (lane == 0) {
      if (code != OMQ_TERM_NONE) w.ulegal[wb + u] = 0;
      if (uterm != nullptr) uterm[wb + u] = code;
    }
    return;
  }
  const RowBits one{reinterpret_cast<uint32_t*>(smem + (size_t)wave * stride)};
  const RowBits two{one.words + kRowWords};
  one.clear();
  two.clear();
  wave_sync();
  const int8_t* rb = root_boards + (int64_t)t * cells;
  int stones = 0;
  uint64_t other = 0;
  for (int c0 = 0; c0 < cells; c0 += kWave) {
    const int v = c0 + lane < cells ? rb[c0 + lane] : 0;
    const uint64_t b1 = __ballot(v == 1), b2 = __ballot(v == 2), bx = __ballot(v != 0);
    one.put(c0, b1);
    two.put(c0, b2);
    stones += __popcll(bx);
    other |= bx & ~(b1 | b2);
  }
  const int rp = root_player != nullptr ? root_player[t] : ((stones & 1) == 0 ? 1 : 2);
  wave_sync();
  int code = OMQ_TERM_NONE;
  if (other == 0 && (rp == 1 || rp == 2)) {
    uint32_t m1 = one.row(bs), m2 = two.row(bs);
    each_move(L, a_lo, a_hi, cells, bs, [&](int j, uint32_t bit) {
      const bool first = ((j & 1) == 0) == (rp == 1);  // played by player 1
      m1 = first ? m1 | bit : m1 & ~bit;
      m2 = first ? m2 & ~bit : m2 | bit;
    });
    const uint32_t f1 = five_starts(m1, rule == OMQ_RULE_RENJU), f2 = five_starts(m2, false);
    const uint64_t rows = __ballot((f1 | f2) != 0u);
    if (rows != 0) {  // the first cell in row-major order names the winner
      const int c = __ffs(f1 | f2) - 1;
      code = readlane_i((f1 >> (c & 31)) & 1u ? 1 : 2, lowest_lane(rows));
    } else if (wave_sum_i(__popc(m1 | m2)) == cells) {
      code = OMQ_TERM_DRAW;
    }
  } else {
    wave_sync();
    code = scanned();
  }
  if (lane == 0) {
    if (code != OMQ_TERM_NONE) w.ulegal[wb + u] = 0;
    if (uterm != nullptr) uterm[wb + u] = code;
  }
}

// Go rules of unique leaf u of tree t (one wavefront per leaf), on the row masks of the empty
// points (a pass, action cells, places no stone).  A point is legal when it is empty, is not the
// root's ko point (OMQ_GO_KO: the reference's clones inherit a state's ko point, so it holds at
// every depth), and, with OMQ_GO_SUICIDE, has an empty orthogonal neighbour; the pass is always
// legal.  The rows are put together to the leaf's mask words in LDS.  Trailing passes are counted
// from the path's end (the root's own when every path move is a pass).  16 trees of 512 leaves,
// 19x19: 11.5 us with the points read one by one from an LDS board, 7.0 us so.
__global__ void go_rules_kernel(omq_forest f, omq_wave w, const int8_t* root_boards,
                                const int32_t* root_player, const int32_t* root_passes,
                                const int32_t* root_ko, int flags, int bs, int32_t* uterm) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int cells = bs * bs;
  const int stride = rule_lds_per_wave(cells);
  const int t = blockIdx.y;
  const int wave = threadIdx.x / kWave;
  const int u = blockIdx.x * (blockDim.x / kWave) + wave;
  const int lane = lane_id();
  const int64_t wb = (int64_t)t * w.max_wave;
  if (u >= w.ucount[t]) return;
  const int s0 = w.ufirst[wb + u];
  int a_lo, a_hi;
  const int L = load_path_actions(f, w, t, s0, &a_lo, &a_hi);
  const RowBits bits{reinterpret_cast<uint32_t*>(smem + (size_t)wave * stride)};
  bits.clear();
  wave_sync();
  const int8_t* rb = root_boards + (int64_t)t * cells;
  for (int c0 = 0; c0 < cells; c0 += kWave)
    bits.put(c0, __ballot(c0 + lane < cells && rb[c0 + lane] == 0));
  // trailing passes of the path (moves 0..L-2; lane j holds moves j and j+64)
  int trail = 0;
  for (int j = L - 2; j >= 0; --j) {
    const int a = j < kWave ? readlane_i(a_lo, j) : readlane_i(a_hi, j - kWave);
    if (a != cells) break;
    ++trail;
  }
  if (trail == L - 1 && root_passes != nullptr) trail += root_passes[t];
  const int ko = ((flags & OMQ_GO_KO) && root_ko != nullptr) ? root_ko[t] : -1;
  wave_sync();
  uint32_t empty = bits.row(bs);
  const int rp = root_player != nullptr ? root_player[t] : 1;  // (whose stone does not matter)
  each_move(L, a_lo, a_hi, cells, bs, [&](int j, uint32_t bit) {
    const bool stone = (int8_t)((j & 1) == 0 ? rp : 3 - rp) != 0;
    empty = stone ? empty & ~bit : empty | bit;
  });
  uint32_t ok = empty;
  if (flags & OMQ_GO_SUICIDE)
    ok &= empty << 1 | empty >> 1 | row_at(empty, 1) | row_at(empty, -1);
  if (ko >= 0 && ko < cells && lane == ko / bs) ok &= ~(1u << (ko - ko / bs * bs));
  // rows to words: row r starts at bit r * bs; then the pass
  wave_sync();
  bits.clear();
  wave_sync();
  if (lane < bs) {
    const int o = lane * bs;
    const uint64_t x = (uint64_t)ok << (o & 31);
    atomicOr(&bits.words[o >> 5], (uint32_t)x);
    if ((uint32_t)(x >> 32) != 0u) atomicOr(&bits.words[(o >> 5) + 1], (uint32_t)(x >> 32));
  }
  if (lane == bs) atomicOr(&bits.words[cells >> 5], 1u << (cells & 31));
  wave_sync();
  uint32_t* mask = w.umask + (wb + u) * (int64_t)f.legal_words;
  if (lane < f.legal_words) mask[lane] = bits.words[lane];
  const int legal = wave_sum_i(__popc(ok)) + 1;
  const int free_points = wave_sum_i(__popc(empty));
  if (lane == 0) {
    const bool term = L > 1 && (trail >= 2 || free_points == 0);
    w.ulegal[wb + u] = term ? 0 : legal;
    if (uterm != nullptr) uterm[wb + u] = term ? OMQ_TERM_END : OMQ_TERM_NONE;
  }
}

hipError_t launch_go_rules(const omq_forest& f, const omq_wave& w, const int8_t* boards,
                           const int32_t* root_player, const int32_t* root_passes,
                           const int32_t* root_ko, int flags, int bs, int32_t* uterm,
                           hipStream_t st) {
  constexpr int wpb = 4;
  const size_t lds = (size_t)rule_lds_per_wave(bs * bs) * wpb;
  dim3 grid((w.max_wave + wpb - 1) / wpb, f.num_trees);
  hipLaunchKernelGGL(go_rules_kernel, grid, dim3(wpb * kWave), lds, st, f, w, boards, root_player,
                     root_passes, root_ko, flags, bs, uterm);
  return hipGetLastError();
}

hipError_t launch_gomoku_terminal(const omq_forest& f, const omq_wave& w, const int8_t* boards,
                                  const int32_t* root_player, int rule, int bs, int32_t* uterm,
                                  hipStream_t st) {
  constexpr int wpb = 4;
  const size_t lds = (size_t)rule_lds_per_wave(bs * bs) * wpb;
  dim3 grid((w.max_wave + wpb - 1) / wpb, f.num_trees);
  const bool scan = bs * bs <= kWave ||
                    (bs * bs <= 2 * kWave && (int64_t)w.max_wave * f.num_trees >= kRuleManySlots);
  hipLaunchKernelGGL(gomoku_terminal_kernel, grid, dim3(wpb * kWave), lds, st, f, w, boards,
                     root_player, rule, bs, scan, uterm);
  return hipGetLastError();
}

// Feature planes of every wave slot (slot u of tree t; NW wavefronts each, below).  Slot
// u < ucount[t] holds the position of unique leaf u; the other slots are written with zeros.
// Planes follow CPUGameStates.get_nn_features, representation 'basic'
// (python/mcts/cpu/cpu_game_states.py:430-494), with the leaf's player to move and move count
// as CPUGameStates.apply_actions (cpu_game_states.py:352-412) leaves them after the path:
//   0 stones of the player to move, 1 stones of the opponent, 2-15 zero (history, unused by
//   the reference), 16 ones when player 1 is to move, 17 move count / 100 (the reference's
//   int16 count divided in double, stored as float), 18 ones (only with 19 planes).
// NW wavefronts per slot: the first rebuilds the leaf's board in LDS, all write the slot's block
// of PLANES*cells values, 16 bytes per lane and store where the address allows (an unaligned
// head and tail of single values; the caller's buffer need not be aligned to more than two values,
// and a slot of odd length starts anywhere).  The stores are bound by HBM, but a slot's chain of
// dependent loads (leaf count and first simulation, length, path, actions) takes longer than its
// share of the stores, so with many slots what counts is how many chains are in flight: one wave
// per slot keeps 32 of them on a CU, a workgroup of four 8.  With few slots, which one wave each
// would leave most of the chip idle, four waves share a slot's stores.
// Measured, 15x15, a call among others, against one 256-thread workgroup per slot with 8-byte
// stores and the planes found per value: 16384 slots float32 NCHW 99.7 -> 65.5 us (4.3 TB/s; a
// fill of the same buffers takes 42 us), bfloat16 NHWC 71.0 -> 36.2 us; 8192 slots 53.5 -> 35.2 and
// 34.6 -> 16.6 us; 2048 slots (four waves) 16.0 -> 10.6 and 12.7 -> 10.4 us, where the launch bounds
// both.  With one wave per slot each XCD writes one run of slots (the first of these 65.0 -> 63.3
// us; all slots zero, without the chains, 51).  One wave per slot from 4096 slots (16 per CU) on, and
// from 2048 for channels-last planes, whose four waves each set up the words of their stores, and for
// boards of at most 81 cells, whose slots are too short for four.  Device time, one wave / four:
// 15x15 NCHW float32 512 slots 6.9 / 5.2 us, 2048 11.1 / 9.5, 4096 15.4 / 15.4, 8192 23.4 / 24.9; NHWC
// bfloat16 512 slots 5.5 / 5.3, 2048 7.9 / 8.8, 4096 10.8 / 14.7; 7x7 NHWC bfloat16 2048 slots 5.1 /
// 6.4, 3900 6.5 / 10.0 (NCHW 7.0 / 8.6).
constexpr int kFeatOneWaveSlots = 4096;
constexpr int kFeatOneWaveSlotsShort = 2048;
constexpr int kFeatShortCells = 81;

template <typename OutT>
struct PlaneStore;
template <>
struct PlaneStore<float> {
  static constexpr int kVec = 4;
  __device__ static float one(float v) { return v; }
  __device__ static uint32_t word(const float* v) { return __float_as_uint(v[0]); }
};
template <>
struct PlaneStore<uint16_t> {  // bfloat16, rounded to nearest even
  static constexpr int kVec = 8;
  __device__ static uint16_t one(float v) {
    const uint32_t x = __float_as_uint(v);
    return (uint16_t)((x + 0x7FFFu + ((x >> 16) & 1u)) >> 16);
  }
  __device__ static uint32_t word(const float* v) {
    return (uint32_t)one(v[0]) | ((uint32_t)one(v[1]) << 16);
  }
};

template <typename OutT, int PLANES, bool NHWC, int NW>
__global__ __launch_bounds__(NW * kWave) void leaf_features_kernel(
    omq_forest f, omq_wave w, const int8_t* root_boards, const int32_t* root_player,
    const int32_t* root_moves, int bs, OutT* out) {
  using S = PlaneStore<OutT>;
  constexpr int NT = NW * kWave;
  constexpr int V = S::kVec;       // values per 16-byte store
  constexpr int VW = V / 4;        // values per 32-bit word
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_pos[2];  // player to move at the leaf, move count
  const int cells = bs * bs;
  int t = blockIdx.y, u = blockIdx.x;
  if (NW == 1) xcd_block(&u, &t);
  const int tid = threadIdx.x;
  const int per = PLANES * cells;
  OutT* o = out + ((int64_t)t * w.max_wave + u) * per;
  // the slot's whole 16-byte stores: values [hd, hd + V * nv)
  const int hd = min(per, (int)((16 - (reinterpret_cast<uintptr_t>(o) & 15)) & 15) /
                              (int)sizeof(OutT));
  const int nv = (per - hd) / V;
  const int ends = per - V * nv;   // single values: the head and the tail
  uint4* ov = reinterpret_cast<uint4*>(o + hd);
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  if (u >= w.ucount[t]) {
    for (int i = tid; i < nv; i += NT) ov[i] = zero;
    for (int i = tid; i < ends; i += NT) o[i < hd ? i : V * nv + i] = (OutT)0;
    return;
  }
  int8_t* b = reinterpret_cast<int8_t*>(smem);
  int tm, mc;
  if (NW == 1 || tid < kWave) {
    int rp, stones;
    const int moves =
        rebuild_leaf_board<true>(f, w, root_boards, root_player, t, u, cells, b, &rp, &stones) - 1;
    tm = (moves & 1) == 0 ? rp : 3 - rp;
    mc = (root_moves != nullptr ? root_moves[t] : stones) + moves;
    if (NW > 1 && tid == 0) {
      s_pos[0] = tm;
      s_pos[1] = mc;
    }
  }
  if (NW > 1) {
    __syncthreads();
    tm = s_pos[0];
    mc = s_pos[1];
  }
  const float colour = tm == 1 ? 1.0f : 0.0f;
  const float mcv = (float)((double)mc / 100.0);
  // the value of plane c at a cell
  auto value = [&](int c, int cell) -> float {
    const bool stone = c < 2;
    const int v = b[stone ? cell : 0];
    const float rest = c == 16 ? colour : c == 17 ? mcv : c == 18 ? 1.0f : 0.0f;
    return stone ? (v == (c == 0 ? tm : 3 - tm) ? 1.0f : 0.0f) : rest;
  };
  auto value_at = [&](int i) -> float {  // the slot's value i
    const int outer = i / (NHWC ? PLANES : cells);
    const int inner = i - outer * (NHWC ? PLANES : cells);
    return NHWC ? value(inner, outer) : value(outer, inner);
  };
  if constexpr (NHWC) {
    // The planes that a store's values fall on repeat every PLANES / gcd(PLANES, V) stores, so
    // with a stride of a multiple of that a thread's stores all start on the same plane c0: its
    // words are set up once (base: the planes that no stone decides; mo and mp: where the two
    // stone planes of its one cell go), and a store is one board read and a few selects (the
    // planes found anew for each value: 55 us against 36 us for 16384 slots of 15x15 in bfloat16).
    constexpr int kPeriod = PLANES % 2 != 0 ? PLANES : PLANES / 2;  // (18: gcd 2 with 4 and 8)
    static_assert(PLANES == 18 || PLANES == 19, "gcd of the planes and 4 or 8");
    constexpr int kUse = NT / kPeriod * kPeriod;  // threads that store
    if (tid < kUse) {
      int cell = (hd + V * tid) / PLANES;
      const int c0 = hd + V * tid - cell * PLANES;
      uint32_t base[4], mo[4], mp[4];
      const int next = c0 >= 2 ? 1 : 0;  // the stones of the next cell, or of this one
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float x[VW];
        mo[k] = mp[k] = 0u;
#pragma unroll
        for (int e = 0; e < VW; ++e) {
          const int ce = c0 + k * VW + e;
          const int c = ce >= PLANES ? ce - PLANES : ce;
          x[e] = c == 16 ? colour : c == 17 ? mcv : c == 18 ? 1.0f : 0.0f;
          const uint32_t m = VW == 1 ? 0xFFFFFFFFu : 0xFFFFu << (16 * e);
          mo[k] |= c == 0 ? m : 0u;
          mp[k] |= c == 1 ? m : 0u;
        }
        base[k] = S::word(x);
      }
      constexpr uint32_t kOne = VW == 1 ? 0x3F800000u : 0x3F803F80u;  // 1.0 in each value
      constexpr int kCells = kUse * V / PLANES;  // cells per round
      static_assert(kUse * V % PLANES == 0, "a round is a whole number of cells");
      cell += next;
      for (int i = tid; i < nv; i += kUse, cell += kCells) {
        const int v = b[min(cell, cells - 1)];  // (past the board where no mask takes it)
        const uint32_t own = v == tm ? kOne : 0u, opp = v == 3 - tm ? kOne : 0u;
        ov[i] = make_uint4(base[0] | (own & mo[0]) | (opp & mp[0]),
                           base[1] | (own & mo[1]) | (opp & mp[1]),
                           base[2] | (own & mo[2]) | (opp & mp[2]),
                           base[3] | (own & mo[3]) | (opp & mp[3]));
      }
    }
  } else {
    // the stores [z0, z1) lie in planes 2..15 (zeros)
    const int z0 = min(nv, max(0, 2 * cells - hd + V - 1) / V);
    const int z1 = max(z0, min(nv, (16 * cells - hd) / V));
    for (int i = z0 + tid; i < z1; i += NT) ov[i] = zero;
    const int rest = nv - (z1 - z0);
    for (int q = tid; q < rest; q += NT) {
      const int i = q < z0 ? q : q + (z1 - z0);
      int c = (hd + V * i) / cells;
      int cell = hd + V * i - c * cells;
      float x[V];
#pragma unroll
      for (int e = 0; e < V; ++e) {
        x[e] = value(c, cell);
        const bool wrap = cell + 1 == cells;
        cell = wrap ? 0 : cell + 1;
        c += wrap ? 1 : 0;
      }
      ov[i] = make_uint4(S::word(x), S::word(x + VW), S::word(x + 2 * VW), S::word(x + 3 * VW));
    }
  }
  for (int i = tid; i < ends; i += NT) {
    const int e = i < hd ? i : V * nv + i;
    o[e] = S::one(value_at(e));
  }
}

template <typename OutT>
hipError_t launch_leaf_features_t(const omq_forest& f, const omq_wave& w, const int8_t* boards,
                                  const int32_t* root_player, const int32_t* root_moves, int bs,
                                  int planes, bool nhwc, OutT* out, hipStream_t st) {
  const size_t lds = (size_t)(((bs * bs) + 15) & ~15);
  dim3 grid(w.max_wave, f.num_trees);
  const int from = nhwc || bs * bs <= kFeatShortCells ? kFeatOneWaveSlotsShort : kFeatOneWaveSlots;
  const bool one_wave = (int64_t)w.max_wave * f.num_trees >= from;
#define OMQ_FEAT_LAUNCH(P, NH)                                                               \
  if (one_wave)                                                                              \
    hipLaunchKernelGGL((leaf_features_kernel<OutT, P, NH, 1>), grid, dim3(kWave), lds, st, f, \
                       w, boards, root_player, root_moves, bs, out);                         \
  else                                                                                       \
    hipLaunchKernelGGL((leaf_features_kernel<OutT, P, NH, 4>), grid, dim3(4 * kWave), lds,    \
                       st, f, w, boards, root_player, root_moves, bs, out)
  if (planes == 18) {
    if (nhwc) { OMQ_FEAT_LAUNCH(18, true); }
    else { OMQ_FEAT_LAUNCH(18, false); }
  } else {
    if (nhwc) { OMQ_FEAT_LAUNCH(19, true); }
    else { OMQ_FEAT_LAUNCH(19, false); }
  }
#undef OMQ_FEAT_LAUNCH
  return hipGetLastError();
}

hipError_t launch_leaf_features(const omq_forest& f, const omq_wave& w, const int8_t* boards,
                                const int32_t* root_player, const int32_t* root_moves, int bs,
                                int planes, int dtype, int nhwc, void* out, hipStream_t st) {
  if (dtype == OMQ_DTYPE_BF16)
    return launch_leaf_features_t(f, w, boards, root_player, root_moves, bs, planes, nhwc != 0,
                                  static_cast<uint16_t*>(out), st);
  return launch_leaf_features_t(f, w, boards, root_player, root_moves, bs, planes, nhwc != 0,
                                static_cast<float*>(out), st);
}

}  // namespace omq
