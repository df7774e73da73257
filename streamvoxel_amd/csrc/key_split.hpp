// What the cross-attention kernels share: the tile of a workgroup, the window lengths and the key split.
//
// A kernel's parameters P carry B, H, Q, D, q_tiles, the window lengths (kv_len / cu_seqlens / kv_cap, kv_mask), with a
// key mask the windows' lists of blocks that hold an attended key (kv_blocks, rows sb_b apart: the count, then the
// block indices in order, the window's last block the last; the split form with a key mask always has them), the
// output (o, so_*), v_scale, and for the split form `part` (the slots of the parts, [team][2][query tile] of
// split_slot_floats(D) floats) and `teams` (teams of q_tiles workgroups in the grid, a multiple of kXcds).
#pragma once

#include "common.hpp"

namespace svhip {

constexpr int kQTile = 128;   // queries per workgroup
constexpr int kKB = 64;       // keys per block
constexpr int kThreads = 256;
constexpr int kCusPerXcd = 32;  // MI355X: 8 XCDs x 32 CUs
constexpr int kXcds = 8;
// Key split: windows a plan covers (one lane each), the key blocks below which no window's keys are split, the
// smallest range worth a team, and the rounds of resident workgroups above which, and the share of them filled from
// which, the unsplit launch is kept.
constexpr int kSplitMaxWindows = 64;
constexpr int kSplitMinBlocks = 24;
constexpr int kSplitMinRange = 6;
constexpr int kSplitMaxRounds = 4;
constexpr int kSplitFullPercent = 85;
// Running max that a part without the unit's first keys starts from, without a key mask: finite, so that keys whose
// scores are all -inf weigh nothing until a finite score raises it, as they do further inside a walk (from -inf their
// weights would be exp2(-inf + inf), NaN). The unit's first keys keep -inf: a query without any finite score is NaN.
constexpr float kPartMax = -3.0e38f;

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

// Key split. One workgroup per (window, head, query tile) leaves CUs idle when there are few of them (one window: 96
// of 256 CUs, each a serial chain of 153 key blocks) or when the windows' lengths differ (the longest one's chain
// runs on alone). The split form lays the key blocks of all (window, head) units end to end and cuts that line into
// equal ranges, one per team; a team is q_tiles workgroups that walk the same keys for their own query tiles, on one
// XCD, so its L2 still serves a block to all of them. The grid is what the chip holds at once, so every CU has the
// same count of key blocks to do. A range that holds a unit whole writes its output; a part of a unit leaves O, its
// running max and its row sum in fp32, in the team's slot 0 (the range starts inside the unit) or 1 (it only ends
// inside it), and split_join_kernel joins the parts. Where a unit is cut depends on all windows' lengths, and the last
// bits of its result with it (one rounding of P against another running max).
// The lengths are on the device, so every workgroup forms the plan for itself: lane b holds window b's block count.
struct SplitPlan {
  int before, blocks;  // of lane b: blocks of one head in the windows before b, and in b
  int total;           // blocks of the line
  int teams;           // ranges the line is cut into
  bool whole;          // every window is short: ranges are cut at unit boundaries
};

template <typename P>
__device__ __forceinline__ SplitPlan split_plan(const P& p) {
  SplitPlan s;
  const int lane = threadIdx.x & 63;
  s.blocks = 0;
  if (lane < p.B) {
    s.blocks = p.kv_blocks ? p.kv_blocks[lane * p.sb_b] : (window_length(p, lane) + kKB - 1) / kKB;
  }
  int incl = s.blocks, longest = s.blocks;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int up = __shfl_up(incl, off, 64);
    if (lane >= off) incl += up;
    longest = max(longest, __shfl_xor(longest, off, 64));
  }
  s.before = incl - s.blocks;
  s.total = __builtin_amdgcn_readlane(incl, 63) * static_cast<int>(p.H);
  s.whole = __builtin_amdgcn_readfirstlane(longest) < kSplitMinBlocks;
  s.teams = s.whole ? p.teams : min(p.teams, (s.total + kSplitMinRange - 1) / kSplitMinRange);
  return s;
}

// First block (on the line) of team t's range (t <= teams).
template <typename P>
__device__ __forceinline__ int split_cut(const P& p, const SplitPlan& s, int t) {
  if (!s.whole) return static_cast<int>(static_cast<int64_t>(s.total) * t / s.teams);
  const int H = static_cast<int>(p.H), units = H * static_cast<int>(p.B);
  const int u = static_cast<int>(static_cast<int64_t>(units) * t / s.teams);  // the range starts with unit u = b H + h
  if (u >= units) return s.total;
  const int b = u / H, h = u - b * H;
  return H * __builtin_amdgcn_readlane(s.before, b) + h * __builtin_amdgcn_readlane(s.blocks, b);
}

// The window whose blocks hold position pos < total of the line.
template <typename P>
__device__ __forceinline__ int split_window(const P& p, const SplitPlan& s, int pos) {
  const int lane = threadIdx.x & 63;
  const uint64_t at = __builtin_amdgcn_ballot_w64(lane < p.B && static_cast<int>(p.H) * s.before <= pos);
  return __popcll(at) - 1;
}

// The workspace: the slots of the parts, then for every unit the first and last team that hold a part of it (last <
// first where one range holds it whole), written by the workgroups that start the units.
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
__device__ __forceinline__ int2* split_units(const P& p) {
  return reinterpret_cast<int2*>(p.part + 2ll * p.teams * p.q_tiles * split_slot_floats(p.D));
}

// `first`: the unit's first block on the line. No range of a line that is cut inside units is empty (teams is at most
// total / kSplitMinRange, rounded up), so the last team is the last t with floor(total t / teams) <= the last block.
__device__ __forceinline__ int2 split_unit_teams(int team, int first, int unit_blocks, bool whole, int total, int teams) {
  if (whole) return make_int2(0, -1);
  return make_int2(team, static_cast<int>((static_cast<int64_t>(first + unit_blocks) * teams - 1) / total));
}

// Joins the parts of the units that the split kernel cut: O = sum_i w_i O_i, l = sum_i w_i l_i with w_i =
// exp2(m_i - max m) over the parts in key order, then v_scale O / l in the output's type. A part's l is 0 without an
// attended key (only a key mask makes such parts), and also where the query is NaN (the weights' clamp turns NaN to 0):
// only under a key mask is it taken for nothing, so that a NaN query ends in 0 / 0 as in the unsplit form. Workgroup = (unit, query
// tile, kJoinQueries queries, kJoinDims head_dim elements), a thread 4 elements of one query. The parts are read once,
// from the last-level cache where they were just written: a short chain of loads, so the workgroups are many and a
// thread has kJoinAhead parts in flight (one window of 12 heads, nine parts a unit: 10.7 us with four queries a thread
// and three parts in flight, 7.3 us here). Windows without keys get
// their zeros here.
constexpr int kJoinDims = 32;
constexpr int kJoinQueries = kThreads / (kJoinDims / 4);
constexpr int kJoinAhead = 6;

inline dim3 split_join_grid(unsigned tiles, int64_t D) {
  return dim3(tiles, static_cast<unsigned>(cdiv(D, kJoinDims)), kQTile / kJoinQueries);
}

template <typename T, typename P>
__global__ __launch_bounds__(kThreads) void split_join_kernel(P p) {
  const int u = static_cast<int>(blockIdx.x / p.q_tiles), qt = static_cast<int>(blockIdx.x % p.q_tiles);
  const int H = static_cast<int>(p.H);
  const int64_t b = u / H, h = u % H;
  // (The plan's own count: a window without blocks has no part on the line and left no teams.)
  const bool empty = (p.kv_blocks ? p.kv_blocks[b * p.sb_b] : window_length(p, b)) == 0, masked = p.kv_mask != nullptr;
  const int2 teams = split_units(p)[u];  // (left as it was for an empty window)
  const int t0 = empty ? 0 : teams.x, t1 = empty ? -1 : teams.y;
  if (!empty && t1 < t0) return;  // one range holds the unit: its output is written
  const int64_t slot_floats = split_slot_floats(p.D);
  const int d0 = static_cast<int>(blockIdx.y) * kJoinDims + 4 * static_cast<int>(threadIdx.x % (kJoinDims / 4));
  const int ql = static_cast<int>(blockIdx.z) * kJoinQueries + static_cast<int>(threadIdx.x / (kJoinDims / 4));
  const int64_t q = static_cast<int64_t>(qt) * kQTile + ql;
  if (d0 >= p.D || q >= p.Q) return;
  float m = -INFINITY, l = 0.f;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
  for (int t = t0; t <= t1; t += kJoinAhead) {
    float mi[kJoinAhead], li[kJoinAhead];
    f32x4_t oi[kJoinAhead];
#pragma unroll
    for (int a = 0; a < kJoinAhead; ++a) {
      if (t + a > t1) break;  // uniform
      // The first part is the one its team's range ends in (slot 1), the others begin their teams' ranges (slot 0).
      const float* slot =
          p.part + (static_cast<int64_t>(2 * (t + a) + (t + a == t0 ? 1 : 0)) * p.q_tiles + qt) * slot_floats;
      mi[a] = slot[kQTile * p.D + ql];
      li[a] = slot[kQTile * (p.D + 1) + ql];
      oi[a] = *reinterpret_cast<const f32x4_t*>(slot + (static_cast<int64_t>(d0 >> 2) * kQTile + ql) * 4);
    }
#pragma unroll
    for (int a = 0; a < kJoinAhead; ++a) {
      if (t + a > t1) break;
      if (masked && li[a] == 0.f) continue;  // a part without an attended key
      const float mn = fmaxf(m, mi[a]);
      const float x = __builtin_amdgcn_exp2f(m - mn), y = __builtin_amdgcn_exp2f(mi[a] - mn);
      m = mn;
      l = l * x + li[a] * y;
      o = o * x + oi[a] * y;
    }
  }
  T* out = static_cast<T*>(p.o) + b * p.so_b + h * p.so_h + q * p.so_q + d0;
  const float inv = empty || (masked && l == 0.f) ? 0.f : (p.v_scale ? p.v_scale[b * p.H + h] : 1.f) / l;
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = o[e] * inv;  // rows of any alignment
  } else {
    *reinterpret_cast<uint2*>(out) = make_uint2(bf16_pack2(o[0] * inv, o[1] * inv), bf16_pack2(o[2] * inv, o[3] * inv));
  }
}

// Teams of the split form for these sizes, or 0 where the launch keeps one workgroup per (window, head, query tile):
// windows beyond one wave's lanes, no window long enough to be split, or query tiles that fill the rounds of resident
// workgroups by themselves. There the longest-first order balances uneven windows as well, without the parts' 50 MB
// (8 windows x 12 heads x 1024 queries, 768 tiles = one full round of 3 per CU: 223-230 us unsplit, 232-240 split; of
// it the kernel 224-230 against 241 and the join 17). One window of 12 heads (96 tiles) goes from 105 to 48 us, the 512
// tiles of 8 windows x 8 heads x 48 from 180 to 153.
// resident: workgroups of the split kernel that a CU holds; turns: ranges per resident team.
inline int split_teams(int64_t B, int64_t H, int64_t Q, int64_t kv_cap, int resident, int turns = 1) {
  const int64_t q_tiles = cdiv(Q, kQTile);
  const int64_t per_xcd = kCusPerXcd * resident, slots = kXcds * per_xcd;
  if (B < 1 || B > kSplitMaxWindows || q_tiles < 1 || q_tiles > per_xcd / 4) return 0;
  if (cdiv(kv_cap, kKB) < kSplitMinBlocks) return 0;
  const int64_t tiles = B * H * q_tiles, rounds = cdiv(tiles, slots);
  if (rounds > kSplitMaxRounds || tiles * 100 >= rounds * slots * kSplitFullPercent) return 0;
  if (B * H * cdiv(kv_cap, kKB) >= (1ll << 31)) return 0;
  return static_cast<int>(kXcds * (per_xcd / q_tiles) * turns);
}

inline size_t split_workspace_bytes(int64_t B, int64_t H, int64_t Q, int64_t D, int64_t kv_cap, int resident,
                                    int turns = 1) {
  const int64_t teams = split_teams(B, H, Q, kv_cap, resident, turns);
  return teams ? static_cast<size_t>(2 * teams * cdiv(Q, kQTile) * split_slot_floats(D)) * sizeof(float) +
                     static_cast<size_t>(B * H) * sizeof(int2)
               : 0;
}

}  // namespace svhip
