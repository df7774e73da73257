// What the cross-attention kernels share: the tile of a workgroup, the window lengths, the pieces of a window and the
// launch that deals them out.
//
// A kernel's parameters P carry B, H, Q, D, q_tiles, the window lengths (kv_len / cu_seqlens / kv_cap, kv_mask), with
// a key mask the windows' lists of blocks that hold an attended key (kv_blocks, rows sb_b apart: the count, then the
// block indices in order, the window's last block the last; the split form with a key mask always has them), the
// output (o, so_*), v_scale, `lone` and `piece_blocks` (pieces_of), and for the split form `part` (one slot of
// split_slot_floats(D) floats for every team and query tile, then a SplitUnit for every window and head), `teams`
// (teams of q_tiles workgroups in the grid, a multiple of kXcds) and `resident` (the teams that the chip holds at
// once).
#pragma once

#include "common.hpp"

namespace svhip {

constexpr int kQTile = 128;   // queries per workgroup
constexpr int kKB = 64;       // keys per block
constexpr int kThreads = 256;
constexpr int kCusPerXcd = 32;  // MI355X: 8 XCDs x 32 CUs
constexpr int kXcds = 8;
// Pieces: the key blocks from which a window is cut, and the most pieces.
constexpr int kPieceWindow = 24;
constexpr int kMaxPieces = 16;
// Split launch: windows a plan covers (one lane each), and the rounds of resident workgroups above which, and the share
// of them filled from which, the unsplit launch is kept.
constexpr int kSplitMaxWindows = 64;
constexpr int kSplitMaxRounds = 4;
constexpr int kSplitFullPercent = 85;
// Running max that every piece but a window's first starts from, without a key mask: finite, so that keys whose scores
// are all -inf weigh nothing until a finite score raises it, as they do further inside a piece (from -inf their weights
// would be exp2(-inf + inf), NaN). The first piece keeps -inf: a query without any finite score is NaN.
constexpr float kPieceMax = -3.0e38f;

// Keys of window b.
template <typename P>
__device__ __forceinline__ int window_length(const P& p, int64_t b) {
  int64_t L;
  if (p.cu_seqlens) {
    L = static_cast<int64_t>(p.cu_seqlens[b + 1]) - p.cu_seqlens[b];
    if (p.kv_len && L > p.kv_len[b]) L = p.kv_len[b];  // cut at the last attended key
  } else if (p.kv_len) {
    L = p.kv_len[b];
    if (L > p.kv_cap) L = p.kv_cap;
  } else {
    L = p.kv_cap;  // key-mask form without lengths: every key up to the capacity, the mask decides
  }
  if (p.kv_mask && L > p.kv_cap) L = p.kv_cap;  // the mask rows hold kv_cap keys
  return L < 0 ? 0 : static_cast<int>(L);
}

// The highest index j < n with row[j] != 0 among the ones this thread reads (thread t of kThreads: 16-byte chunks
// t, t + kThreads, ... of a 16-byte aligned row, four loads in flight; the rest, or an unaligned row, byte by byte
// with eight loads in flight), or -1. The caller takes the maximum over the workgroup.
__device__ __forceinline__ int last_attended(const uint8_t* row, int n) {
  int last = -1;
  const int nvec = (reinterpret_cast<uintptr_t>(row) & 15) == 0 ? n / 16 : 0;
  for (int c0 = threadIdx.x; c0 < nvec; c0 += 4 * kThreads) {
    uint4 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = c0 + u * kThreads;
      x[u] = c < nvec ? reinterpret_cast<const uint4*>(row)[c] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t w[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {  // the highest nonzero byte of word q: byte 4 q + (31 - clz) / 8
        if (w[q] != 0u) last = max(last, 16 * (c0 + u * kThreads) + 4 * q + ((31 - __clz(w[q])) >> 3));
      }
    }
  }
  for (int j0 = 16 * nvec + threadIdx.x; j0 < n; j0 += 8 * kThreads) {
    uint8_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = row[min(j0 + u * kThreads, n - 1)];  // no branch around the loads
#pragma unroll
    for (int u = 0; u < 8; ++u) last = (v[u] && j0 + u * kThreads < n) ? max(last, j0 + u * kThreads) : last;
  }
  return last;
}

// Pieces. A window of kPieceWindow key blocks or more is attended in pieces, each from a running max and sums of its
// own, joined in order in fp32 (join_value). Where a window is cut depends on its own blocks and on the launch's H and
// Q alone, never on the other windows, and the joins are the same whoever makes them: a workgroup that walks several
// pieces, or split_join_kernel. So a window gives the same bits alone and in any batch, split or not.
struct Pieces {
  int blocks, each, count;  // key blocks of the window, of a piece (even), and the pieces
};

// The pieces of a window: of as many blocks each as give `lone` teams (lone_teams) an equal share when the window is
// alone, at least `least`, and at most kMaxPieces pieces. The last one holds what is left, half of `least` or more.
__host__ __device__ __forceinline__ Pieces pieces_of(int blocks, int64_t H, int lone, int least) {
  Pieces s{blocks, blocks, 1};
  if (blocks < kPieceWindow) return s;
  const int64_t share = (static_cast<int64_t>(blocks) * H + lone - 1) / lone;
  const int shortest = (blocks + kMaxPieces - 1) / kMaxPieces;
  int64_t each = share > least ? share : least;
  if (each < shortest) each = shortest;
  if (each >= blocks) return s;
  s.each = static_cast<int>(each + (each & 1));
  s.count = blocks / s.each;
  if (2 * (blocks - s.count * s.each) >= least) ++s.count;
  if (s.count < 1) s.count = 1;
  return s;
}

// First block of piece i (i == count: the end). Even, so that a walk two blocks at a time ends a piece with a pair.
__host__ __device__ __forceinline__ int piece_start(const Pieces& s, int i) {
  return i == s.count ? s.blocks : i * s.each;
}

// The next piece (mi, li, oi) joined to the ones before it (m, l, o): `x` and `y` are the factors of the two, m the new
// running max. A running max of -inf (only with a key mask) is one that has seen no attended key.
__device__ __forceinline__ void join_factors(float& m, float mi, float& x, float& y) {
  const float mn = fmaxf(m, mi);
  x = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
  y = mi == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mi - mn);
  m = mn;
}
__device__ __forceinline__ float join_value(float o, float oi, float x, float y) {
  return __builtin_fmaf(o, x, oi * y);
}

// Split launch. One workgroup per (window, head, query tile) leaves CUs idle when there are few of them (one window:
// 96 of 256 CUs, each a serial chain of 153 key blocks) or when the windows' lengths differ (the longest one's chain
// runs on alone). The split form deals out teams, q_tiles workgroups that walk the same keys for their own query tiles
// on one XCD, so its L2 still serves a block to all of them: first for every (window, head) its leading pieces, as
// many as an equal share of all blocks allows (joined as they are walked; the whole unit where the share holds it),
// then every other piece by itself, which fill the chip as the first ones end. (All walks sorted by length: 3 windows
// x 8 heads x 96 122 us for 124, but 20 short windows 44 for 40.) A team with a whole unit writes its output, any
// other leaves O, its running max and its row sum in fp32 in its slot, and split_join_kernel joins the slots of a
// unit. The lengths are on the device, so every workgroup forms the plan for itself: lane b holds window b's numbers.
struct SplitPlan {
  Pieces pieces;             // of window b
  int lead;                  // the leading ones walked together
  int rank;                  // place of window b among the leading runs, longest first
  int before, others;        // other pieces of all heads of the windows before b, and of all windows
};

template <typename P>
__device__ __forceinline__ SplitPlan split_plan(const P& p) {
  SplitPlan s;
  const int lane = threadIdx.x & 63, H = static_cast<int>(p.H);
  int blocks = 0, work = 0;  // key blocks of one head, and the ones to do (with a key mask the listed ones)
  if (lane < p.B) {
    blocks = (window_length(p, lane) + kKB - 1) / kKB;
    work = p.kv_blocks ? p.kv_blocks[lane * p.sb_b] : blocks;
  }
  s.pieces = pieces_of(blocks, p.H, p.lone, p.piece_blocks);
  // The share by the blocks to do. Should its leading runs leave more pieces than the grid has teams: by all blocks,
  // for which split_teams has allowed; against every expectation, each unit whole.
  for (int pass = 0; pass < 3; ++pass) {
    const int mine = pass == 0 ? work : blocks;
    int64_t sum = mine;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
    const int64_t share = sum * H / p.resident;
    int64_t end = share;  // the block at which the share ends
    if (pass == 0 && p.kv_blocks && share < work) end = p.kv_blocks[lane * p.sb_b + 1 + share];
    s.lead = s.pieces.count;
    if (pass < 2 && share < mine) s.lead = min(s.lead, max(1, static_cast<int>(end) / s.pieces.each));
    const int count = lane < p.B ? H * (s.pieces.count - s.lead) : 0;
    int incl = count;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off, 64);
      if (lane >= off) incl += up;
    }
    s.before = incl - count;
    s.others = __builtin_amdgcn_readlane(incl, 63);
    if (static_cast<int>(p.B) * H + s.others <= p.teams) break;
  }
  const int run = piece_start(s.pieces, s.lead);
  s.rank = 0;
  for (int o = 0; o < static_cast<int>(p.B); ++o) {
    const int other = __builtin_amdgcn_readlane(run, o);
    s.rank += other > run || (other == run && o < lane) ? 1 : 0;
  }
  return s;
}

// Pieces [first, end) of (window b, head h); window b's numbers of the plan.
struct SplitItem {
  int b, h, first, end, before;
  int pieces;
};

// What team t walks; false: nothing.
template <typename P>
__device__ __forceinline__ bool split_item(const P& p, const SplitPlan& s, int t, SplitItem& item) {
  const int lane = threadIdx.x & 63, H = static_cast<int>(p.H), units = H * static_cast<int>(p.B);
  if (t >= units + s.others) return false;
  if (t < units) {
    const int r = t / H;
    item.h = t - r * H;
    item.b = __builtin_ctzll(__builtin_amdgcn_ballot_w64(lane < p.B && s.rank == r));
    item.first = 0;
    item.end = __builtin_amdgcn_readlane(s.lead, item.b);
  } else {
    t -= units;
    item.b = __popcll(__builtin_amdgcn_ballot_w64(lane < p.B && s.before <= t)) - 1;
    t -= __builtin_amdgcn_readlane(s.before, item.b);
    const int i = t / H;  // all heads' first other piece, then their second one, ...: the short last ones at the end
    item.h = t - i * H;
    item.first = __builtin_amdgcn_readlane(s.lead, item.b) + i;
    item.end = item.first + 1;
  }
  item.pieces = __builtin_amdgcn_readlane(s.pieces.count, item.b);
  item.before = __builtin_amdgcn_readlane(s.before, item.b);
  return true;
}

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void split_store(float* slot, int d0, int ql, float a, float b, float c, float d) {
  *reinterpret_cast<float4*>(slot + (static_cast<int64_t>(d0 >> 2) * kQTile + ql) * 4) = make_float4(a, b, c, d);
}

// Entry i of window b's list of blocks, through the scalar cache: a vector load would have to wait for the staged
// loads in flight before it.
template <typename P>
__device__ __forceinline__ int listed_block(const P& p, int64_t b, int i) {
  typedef const __attribute__((address_space(4))) int32_t* list_t;
  return __builtin_amdgcn_readfirstlane(((list_t)(p.kv_blocks + b * p.sb_b + 1))[i]);
}

__host__ __device__ __forceinline__ int64_t split_slot_floats(int64_t D) { return kQTile * (D + 2); }

template <typename P>
__device__ __forceinline__ float* split_slot(const P& p, int team, int qt) {
  return p.part + (static_cast<int64_t>(team) * p.q_tiles + qt) * split_slot_floats(p.D);
}

// The unit's row of the table behind the slots, written by the team of its leading pieces: that team, and the first
// team and the number of its other pieces, which have every H-th team from there.
struct SplitUnit {
  int lead, others, count, pad;
};

template <typename P>
__device__ __forceinline__ SplitUnit* split_unit(const P& p, int64_t b, int64_t h) {
  return reinterpret_cast<SplitUnit*>(p.part + static_cast<int64_t>(p.teams) * p.q_tiles * split_slot_floats(p.D)) +
         b * p.H + h;
}

template <typename P>
__device__ __forceinline__ void split_publish(const P& p, const SplitItem& item, int team, int qt) {
  if (item.first != 0 || qt != 0 || threadIdx.x != 0) return;
  const int units = static_cast<int>(p.B * p.H), count = item.pieces - item.end;
  *split_unit(p, item.b, item.h) = {team, units + item.before + item.h, count, 0};
}

// Entries of window b's list of blocks (count of them in `count`) below `block`.
template <typename P>
__device__ __forceinline__ int listed_before(const P& p, int64_t b, int count, int block) {
  const int32_t* list = p.kv_blocks + b * p.sb_b + 1;
  const int lane = threadIdx.x & 63;
  int n = 0;
  for (int i = 0; i < count; i += 64) {
    n += __popcll(__builtin_amdgcn_ballot_w64(i + lane < count && list[min(i + lane, count - 1)] < block));
  }
  return n;
}

// Joins the slots of the units that several teams walked, then v_scale O / l in the output's type. l is 0 without an
// attended key (only under a key mask, where it gives zeros), and also where the query is NaN (the weights' clamp
// turns NaN to 0): 0 / 0 is NaN again. Workgroup = (unit, query tile, kJoinQueries queries, kJoinDims head_dim
// elements), a thread 4 elements of one query. The parts are read once, from the last-level cache where they were just
// written: a short chain of loads, so the workgroups are many and a thread has kJoinAhead parts in flight (one window
// of 12 heads, nine parts a unit: 10.7 us with four queries a thread and three parts in flight, 7.3 us here; the five
// parts of a unit now 5.1 us).
constexpr int kJoinDims = 32;
constexpr int kJoinQueries = kThreads / (kJoinDims / 4);
constexpr int kJoinAhead = 6;

inline dim3 split_join_grid(unsigned tiles, int64_t D) {
  return dim3(tiles, static_cast<unsigned>(cdiv(D, kJoinDims)), kQTile / kJoinQueries);
}

template <typename T, typename P>
__global__ __launch_bounds__(kThreads) void split_join_kernel(P p) {
  const int u = static_cast<int>(blockIdx.x / p.q_tiles), qt = static_cast<int>(blockIdx.x % p.q_tiles);
  const int H = static_cast<int>(p.H), b = u / H, h = u - b * H;
  const SplitUnit unit = *split_unit(p, b, h);
  const int others = unit.count;
  if (others == 0) return;  // one team walked the unit: its output is written
  const int d0 = static_cast<int>(blockIdx.y) * kJoinDims + 4 * static_cast<int>(threadIdx.x % (kJoinDims / 4));
  const int ql = static_cast<int>(blockIdx.z) * kJoinQueries + static_cast<int>(threadIdx.x / (kJoinDims / 4));
  const int64_t q = static_cast<int64_t>(qt) * kQTile + ql;
  if (d0 >= p.D || q >= p.Q) return;
  float m = 0.f, l = 0.f;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
  for (int t = 0; t <= others; t += kJoinAhead) {
    float mi[kJoinAhead], li[kJoinAhead];
    f32x4_t oi[kJoinAhead];
#pragma unroll
    for (int a = 0; a < kJoinAhead; ++a) {
      if (t + a > others) break;  // uniform
      const float* slot = split_slot(p, t + a == 0 ? unit.lead : unit.others + (t + a - 1) * H, qt);
      mi[a] = slot[kQTile * p.D + ql];
      li[a] = slot[kQTile * (p.D + 1) + ql];
      oi[a] = *reinterpret_cast<const f32x4_t*>(slot + (static_cast<int64_t>(d0 >> 2) * kQTile + ql) * 4);
    }
#pragma unroll
    for (int a = 0; a < kJoinAhead; ++a) {
      if (t + a > others) break;
      if (t + a == 0) {
        m = mi[a];
        l = li[a];
        o = oi[a];
        continue;
      }
      float x, y;
      join_factors(m, mi[a], x, y);
      l = join_value(l, li[a], x, y);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = join_value(o[e], oi[a][e], x, y);
    }
  }
  T* out = static_cast<T*>(p.o) + b * p.so_b + h * p.so_h + q * p.so_q + d0;
  const float inv = p.kv_mask && !(l > 0.f) ? 0.f : (p.v_scale ? p.v_scale[b * p.H + h] : 1.f) / l;
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = o[e] * inv;  // rows of any alignment
  } else {
    *reinterpret_cast<uint2*>(out) = make_uint2(bf16_pack2(o[0] * inv, o[1] * inv), bf16_pack2(o[2] * inv, o[3] * inv));
  }
}

// Teams that the chip holds at once; 0: more query tiles than a quarter of an XCD's workgroups.
inline int resident_teams(int64_t Q, int resident) {
  const int64_t q_tiles = cdiv(Q, kQTile), per_xcd = kCusPerXcd * resident;
  return q_tiles < 1 || q_tiles > per_xcd / 4 ? 0 : static_cast<int>(kXcds * (per_xcd / q_tiles));
}

// Teams of a window that is alone, by which windows are cut: two workgroups for every CU.
inline int lone_teams(int64_t Q) {
  const int64_t n = 2 * kXcds * kCusPerXcd / (Q < 1 ? 1 : cdiv(Q, kQTile));
  return n < 1 ? 1 : static_cast<int>(n);
}

// Teams of the split form for these sizes, or 0 where the launch keeps one workgroup per (window, head, query tile):
// windows beyond one wave's lanes, no window long enough to be cut, query tiles that fill the rounds of resident
// workgroups by themselves, or more than `per_block` tiles for every key block of the longest window. The unsplit
// launch takes the longest window's chain of blocks and the split one the parts' traffic and the join, which grow with
// the tiles; bf16 (per_block 8), windows of one length, unsplit -> split:
//   12 x 64 heads, 25 / 64 / 153 blocks:  96 tiles 24 -> 23, 49 -> 31, 106 -> 48 us;  192 tiles 26 -> 30, 50 -> 46,
//   108 -> 82;  384 tiles 34 -> 37, 70 -> 76, 155 -> 145;  576 tiles 44 -> 52, 100 -> 98, 225 -> 209
//   8 x 96 heads: 128 tiles 28 -> 28, 63 -> 50, 139 -> 83;  256 tiles 31 -> 36, 66 -> 73, 144 -> 152
// and windows of different lengths better by up to a third more; a full round of 768 tiles in 8 such windows 170 ->
// 175. fp32 (no such bound, its blocks take six times as long): 96 tiles of 25 blocks 154 -> 81 us, 384 tiles 262 ->
// 229.
// resident: workgroups of the split kernel that a CU holds. A unit of n pieces and `blocks` blocks beside a share of s
// blocks leaves at most n (1 - s / blocks) + 2 pieces to themselves (one for the last piece, one for the pieces of the
// share, a part of one for the share's own rounding), and k units of equal length hold R / k shares each, R = resident
// teams: n k (1 - k / R) in all, the most at k = R / 2.
inline int split_teams(int64_t B, int64_t H, int64_t Q, int64_t kv_cap, int resident, int least,
                       int per_block) {
  const int64_t R = resident_teams(Q, resident), q_tiles = cdiv(Q, kQTile), slots = kXcds * kCusPerXcd * resident;
  const int64_t blocks = cdiv(kv_cap, kKB);
  if (B < 1 || B > kSplitMaxWindows || R == 0 || blocks < kPieceWindow) return 0;
  const int lone = lone_teams(Q);
  if (pieces_of(static_cast<int>(blocks), H, lone, least).count < 2) return 0;
  // The most pieces of any window (a shorter one may have more than the longest).
  int64_t n = lone / H + 1 < blocks / least + 1 ? lone / H + 1 : blocks / least + 1;
  if (n > kMaxPieces) n = kMaxPieces;
  const int64_t units = B * H, tiles = units * q_tiles, rounds = cdiv(tiles, slots);
  if (rounds > kSplitMaxRounds || tiles * 100 >= rounds * slots * kSplitFullPercent) return 0;
  if (per_block && tiles > per_block * blocks) return 0;
  const int64_t k = units < R / 2 ? units : R / 2, long_units = units < R ? units : R;
  const int64_t spread = units + cdiv(n * k * (R - k), R) + cdiv(9 * long_units, 4);
  return static_cast<int>(kXcds * cdiv(n * units < spread ? n * units : spread, kXcds));
}

inline size_t split_workspace_bytes(int64_t B, int64_t H, int64_t Q, int64_t D, int64_t kv_cap, int resident,
                                    int least, int per_block) {
  const int64_t teams = split_teams(B, H, Q, kv_cap, resident, least, per_block);
  return teams ? static_cast<size_t>(teams * cdiv(Q, kQTile) * split_slot_floats(D)) * sizeof(float) +
                     static_cast<size_t>(B * H) * sizeof(SplitUnit)
               : 0;
}

}  // namespace svhip
