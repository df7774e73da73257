// Cross attention in fp32 arithmetic: fp32 Q/K/V/O, every product, sum and exponential in fp32.
//
// The single-column configuration runs the reference's cross attention in fp32 (the masked SDPA of
// SlotCrossAttention.forward, streamvoxel/stream/engine.py:28-47, on fp32 tensors). The bf16 kernel rounds its
// operands to bf16 for the matrix cores; this one keeps the reference's arithmetic width: both products are
// v_mfma_f32_32x32x2_f32 (fp32 operands and accumulation, no rounding of either operand).
//
// Bound: the fp32 matrix cores (64 FLOP a cycle and SIMD, a sixteenth of bf16; a large fp32 matrix product reaches
// 154 TFLOP/s on the card). A 32-key x 32-query half costs 64 of these products at head_dim 64 (4096 cycles) against
// 16 exponentials, so the softmax and the LDS reads hide behind them; K and V are staged once for the workgroup's
// 128 queries.
//
// Work item: one workgroup = (window b, head h, 128-query tile), 4 waves x 32 queries, 64-key blocks in LDS (the next
// block's loads in flight in registers while the current one is computed). Per wave and 32-key half:
//   S^T[key, q] = K . Q^T     A = K rows from LDS, B = the wave's Q (registers). The k order is free as long as both
//                             operands share it: lane half hh takes head_dim 8 s + 4 hh + j at step 4 s + j, so a
//                             lane reads K in 16-byte chunks.
//   P^T = exp2(S^T - m)       online softmax, lane (col, hh) owns query col and the keys 8 (i / 4) + 4 hh + i % 4
//   O^T[d, q] += V^T . P^T    step i pairs the keys of accumulator entry i of both lane halves, so P^T is the B
//                             operand as it stands; A = V[that key][32 j + col] from LDS.
// The split form (SPLIT) is the bf16 kernel's: see key_split.hpp.
//
// One window of 12 x 64 heads, 1024 queries, 9744 keys: 816 us on the VALU (one query a lane, K and V rows broadcast
// from LDS: 37 TFLOP/s), 316 us here (97 TFLOP/s), 6 us of it the join (286 us where each workgroup walked an equal
// share of the blocks, whose cuts moved with the other windows' lengths). The instruction alone reaches 141 TFLOP/s
// with two waves a SIMD and dependent accumulators, 147 with three.
//
// KMASK: a key mask on top of the window length (the reference's `prefix_valid ++ local_valid`): key j of window b
// is attended only where kv_mask[b * sm_b + j] != 0. A block that the mask wholly masks is skipped; a query may have
// seen no attended key yet, its running max then stays -inf and the exponentials are taken against 0.
#include <type_traits>

#include "key_split.hpp"

namespace svhip {

constexpr int kF32Row = 64;      // floats of an LDS row (one key)
constexpr int kF32Resident = 2;  // workgroups per CU (two waves per SIMD)
// Least key blocks of a piece (key_split.hpp); a block takes six times the bf16 kernel's. One window of 8 x 48 heads
// and 29 blocks at 6 / 12: 63 / 90 us; 2 windows of 8 x 64 and 33 blocks at 12 / 16: 115 / 156.
constexpr int kF32PieceBlocks = 6;
// Key blocks summed into one accumulator before it is added to the total: short chains of fp32 sums, as the two chains
// of a score are. From float64, 128 / 400 / 2300 / 9000 keys: 2.6 / 3.0 / 4.0 / 7.0e-7 on the VALU before, 2.2 / 2.3 /
// 2.6 / 2.8e-7 so; with one chain a score and two blocks 3.1 / 3.4 / 3.5 / 3.8e-7 (8 us faster on the single column),
// with one chain over all blocks of a range 8.1e-7 there.
constexpr int kF32Fold = 1;
// Scores may pass the running max by this much (log2 units) before it is raised. Small: the exponent is rounded at its
// own size, so weights far above 1 would carry 2^-24 times that size.
constexpr float kF32Rise = 1.f;

typedef float f32x16_t __attribute__((ext_vector_type(16)));

struct XattnF32Params {
  const float* q;
  const float* k;
  const float* v;
  float* o;
  const int32_t* kv_len;
  const int32_t* cu_seqlens;
  const uint8_t* kv_mask;  // KMASK: [B, kv_cap] bytes, rows sm_b apart
  const float* v_scale;    // none (the join's output scale)
  int64_t sm_b;
  const int32_t* kv_blocks;  // SPLIT with KMASK: the windows' attended blocks (key_split.hpp)
  int64_t sb_b;
  int64_t B, H, Q, D, kv_cap;
  int64_t sq_b, sq_h, sq_q;
  int64_t sk_b, sk_h, sk_k;
  int64_t sv_b, sv_h, sv_k, sv_d;
  int64_t so_b, so_h, so_q;
  float scale_log2;  // softmax scale * log2(e)
  int q_tiles;
  int lone, piece_blocks;  // by which windows are cut into pieces (pieces_of)
  float* part;   // split form: the slots of the parts, the teams in the grid and the teams that the chip holds at once
  int teams;
  int resident;
};

// LDS rows are 256 bytes, every bank once. K: 16 rows are read at one 16-byte chunk, so chunk c of row r lies at
// c ^ (r % 16). V: a read takes 32 consecutive floats of row r in lane half 0 and of row r + 4 in half 1, so the
// halves of the rows with bit 2 set are swapped.
__device__ __forceinline__ int f32_swz_k(int r, int c) { return c ^ (r & 15); }
__device__ __forceinline__ int f32_swz_v(int r, int c) { return c ^ (((r >> 2) & 1) << 3); }

// VT: V given as V^T rows (keys contiguous, element (key, d) at d * sv_d + key), else V rows (head_dim
// contiguous). Rows start 16-byte aligned (checked by the entry point).
template <int D, bool VT, bool KMASK, bool SPLIT>
__global__ __launch_bounds__(kThreads, kF32Resident) void xattn_f32_kernel(XattnF32Params p) {
  constexpr int kChunks = D / 4;                      // 16-byte chunks of a key's row
  constexpr int kPer = kKB * kChunks / kThreads;      // chunks per thread and block
  constexpr int kTiles = (D + 31) / 32;               // output tiles of 32 head_dim elements
  static_assert(kKB * kChunks % kThreads == 0, "head_dim a multiple of 16");
  __shared__ __attribute__((aligned(16))) float sK[kKB * kF32Row], sV[kKB * kF32Row];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wg = static_cast<int>(blockIdx.x);
  int qt;
  [[maybe_unused]] int team = 0;
  [[maybe_unused]] SplitItem item = {};
  int64_t b = 0, h = 0;
  if constexpr (SPLIT) {
    const int seq = wg >> 3;
    qt = seq % p.q_tiles;
    team = (seq / p.q_tiles) * kXcds + (wg & 7);
    if (!split_item(p, split_plan(p), team, item)) return;
    b = item.b;
    h = item.h;
  } else {
    qt = wg % p.q_tiles;
    const int64_t unit = wg / p.q_tiles;
    b = unit / p.H;
    h = unit % p.H;
  }
  const float sl2 = p.scale_log2;

  const int tid = threadIdx.x;
  const int lane = tid & 63, col = lane & 31, hh = lane >> 5;
  const int64_t q = static_cast<int64_t>(qt) * kQTile + w * 32 + col;
  const bool q_ok = q < p.Q;
  const int L = [&]() __attribute__((always_inline)) {
    const int n = window_length(p, b);
    if constexpr (!KMASK || SPLIT) {
      return n;  // (the split form's lengths are cut at the windows' last attended keys)
    } else {
      __shared__ int s_last;
      if (tid == 0) s_last = -1;
      __syncthreads();
      const int last = last_attended(p.kv_mask + b * p.sm_b, n);
      if (last >= 0) atomicMax(&s_last, last);
      __syncthreads();
      return __builtin_amdgcn_readfirstlane(s_last) + 1;
    }
  }();
  // The walk: pieces [piece, piece_end) of the unit, blocks [blk0, blk1) (with a list, of its entries).
  constexpr bool LIST = SPLIT && KMASK;
  const int unit_blocks = (L + kKB - 1) / kKB;
  const Pieces pieces = pieces_of(unit_blocks, p.H, p.lone, kF32PieceBlocks);
  const int piece_end = SPLIT ? item.end : pieces.count;
  int piece = SPLIT ? item.first : 0;
  auto next_piece = [&]() __attribute__((always_inline)) -> int {
    return piece + 1 < piece_end ? piece_start(pieces, piece + 1) : 0x7fffffff;
  };
  int bound = next_piece();  // first block of the walk's next piece
  int blk0 = 0, blk1 = unit_blocks;
  [[maybe_unused]] int listed = 0;
  if constexpr (SPLIT) {
    blk0 = piece_start(pieces, item.first);
    blk1 = piece_start(pieces, item.end);
  }
  if constexpr (LIST) {
    listed = __builtin_amdgcn_readfirstlane(p.kv_blocks[b * p.sb_b]);
    blk0 = listed_before(p, b, listed, blk0);
    blk1 = listed_before(p, b, listed, blk1);
  }
  const int64_t off = p.cu_seqlens ? p.cu_seqlens[b] : 0;
  const uint8_t* mrow = KMASK ? p.kv_mask + b * p.sm_b : nullptr;
  const float* K = p.k + (p.cu_seqlens ? 0 : b * p.sk_b) + h * p.sk_h + off * p.sk_k;
  const float* V = p.v + (p.cu_seqlens ? 0 : b * p.sv_b) + h * p.sv_h + off * p.sv_k;

  // Q as B operands: entry 4 s + j is head_dim 8 s + 4 hh + j.
  float qf[D / 2];
#pragma unroll
  for (int s = 0; s < D / 8; ++s) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (q_ok) x = *reinterpret_cast<const float4*>(p.q + b * p.sq_b + h * p.sq_h + q * p.sq_q + 8 * s + 4 * hh);
    qf[4 * s] = x.x;
    qf[4 * s + 1] = x.y;
    qf[4 * s + 2] = x.z;
    qf[4 * s + 3] = x.w;
  }
  f32x16_t o[kTiles], total[kTiles];  // O^T of the last blocks, and of those before
#pragma unroll
  for (int j = 0; j < kTiles; ++j) o[j] = total[j] = f32x16_t{0};
  float m = SPLIT && !KMASK && piece > 0 ? kPieceMax : -INFINITY, l = 0.f;  // l: the lane's own keys

  // Block loads: chunk c = thread + 256 r is key c / kChunks, head_dim 4 (c % kChunks) .. + 3 (of V^T key c % 64,
  // head_dim 4 (c / 64) .. + 3: consecutive lanes read consecutive keys of a row). Every load is issued
  // (keys >= L read row L - 1, in bounds); their scores are masked, and V rows past L are zeros so that 0 . V
  // stays 0.
  f32x4_t nk[kPer], nv[kPer];
  auto load_block = [&](int kv0) __attribute__((always_inline)) {
    // Opaque again: the chunks' addresses are formed per block (hidden behind the products); hoisted, they took 16
    // registers and were spilled.
    int tb = tid;
    asm volatile("" : "+v"(tb));
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const int c = tb + kThreads * r;
      const int key = kv0 + c / kChunks, d = 4 * (c % kChunks);
      const int64_t kc = key < L ? key : L - 1;
      nk[r] = *reinterpret_cast<const f32x4_t*>(K + kc * p.sk_k + d);
      if constexpr (VT) {
        const int kt = kv0 + c % kKB;
        const float* src = V + 4 * (c / kKB) * p.sv_d + (kt < L ? kt : L - 1);
        nv[r] = f32x4_t{src[0], src[p.sv_d], src[2 * p.sv_d], src[3 * p.sv_d]};
        if (kt >= L) nv[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      } else {
        nv[r] = *reinterpret_cast<const f32x4_t*>(V + kc * p.sv_k + d);
        if (key >= L) nv[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
  };
  auto store_block = [&]() __attribute__((always_inline)) {
    int tb = tid;
    asm volatile("" : "+v"(tb));
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const int c = tb + kThreads * r;
      const int key = c / kChunks, dc = c % kChunks;
      *reinterpret_cast<f32x4_t*>(sK + key * kF32Row + 4 * f32_swz_k(key, dc)) = nk[r];
      const int vkey = VT ? c % kKB : key, vc = VT ? c / kKB : dc;
      *reinterpret_cast<f32x4_t*>(sV + vkey * kF32Row + 4 * f32_swz_v(vkey, vc)) = nv[r];
    }
  };
  // Bit i: key kv0 + i is below L and attended (wave-uniform; lane i's byte).
  auto load_mask = [&](int kv0) __attribute__((always_inline)) -> int {
    const int j = kv0 + lane;
    if constexpr (KMASK) {
      const int jc = j < L ? j : L - 1;
      return (mrow[jc] != 0 && j < L) ? 1 : 0;
    } else {
      return j < L ? 1 : 0;
    }
  };
  // First key of block i of the unit (of the list).
  auto key_of = [&](int i) __attribute__((always_inline)) -> int {
    if constexpr (LIST) {
      return kKB * listed_block(p, b, min(i, listed - 1));
    } else {
      return kKB * i;
    }
  };
  // The pieces walked before the current one, joined (in LDS, of which two workgroups leave enough: a slot per lane).
  __shared__ __attribute__((aligned(16))) f32x4_t s_joined[4 * kTiles + 1][kThreads];
  bool folded = false;
  // The current piece's sums, joined to the pieces before it: m, l (of both lane halves) and `total` are the walk's.
  auto join = [&]() __attribute__((always_inline)) {
    l += __shfl_xor(l, 32, 64);
    if (!folded) return;
    const f32x4_t ml = s_joined[4 * kTiles][tid];
    float x, y, mn = ml[0];
    join_factors(mn, m, x, y);
    m = mn;
    l = join_value(ml[1], l, x, y);
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4_t at = s_joined[4 * j + g][tid];
#pragma unroll
        for (int e = 0; e < 4; ++e) total[j][4 * g + e] = join_value(at[e], total[j][4 * g + e], x, y);
      }
    }
  };
  // A piece has ended inside the walk: start the one that holds the next block, block `next`.
  auto fold = [&](int next) __attribute__((always_inline)) {
    join();
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        s_joined[4 * j + i / 4][tid] = f32x4_t{total[j][i], total[j][i + 1], total[j][i + 2], total[j][i + 3]};
      }
      total[j] = f32x16_t{0};
    }
    s_joined[4 * kTiles][tid] = f32x4_t{m, l, 0.f, 0.f};
    m = KMASK ? -INFINITY : kPieceMax;
    l = 0.f;
    folded = true;
    do {
      ++piece;
      bound = next_piece();
    } while (next >= bound);
  };
  int on = 0;
  if (blk0 < blk1) {
    const int kv0 = key_of(blk0);
    while (kv0 / kKB >= bound) {  // pieces without a listed block add nothing
      ++piece;
      bound = next_piece();
    }
    load_block(kv0);
    on = load_mask(kv0);
    store_block();
  }
  int kv_next = blk0 < blk1 ? key_of(blk0 + 1) : 0;
  __syncthreads();
  for (int blk = blk0; blk < blk1; ++blk) {
    const uint64_t bits = __builtin_amdgcn_ballot_w64(on != 0);
    const bool more = blk + 1 < blk1;
    const int next = kv_next / kKB;
    if (more) {
      load_block(kv_next);
      on = load_mask(kv_next);
      kv_next = key_of(blk + 2);
    }
    if (!KMASK || bits != 0ull) {
      // The running max taken off the scores. Without a key mask -inf stays: a query whose every score is -inf gets
      // NaN, as a softmax over them does.
      auto bias = [&]() __attribute__((always_inline)) { return KMASK && m == -INFINITY ? 0.f : -m; };
      // One weight, formed where it stands in the code: the volatile asm keeps it from sinking to its use.
      auto weight = [&](float& x, float nm, float& sum) __attribute__((always_inline)) {
        x = __builtin_amdgcn_exp2f(__builtin_fmaf(x, sl2, nm));
        sum += x;
        asm volatile("" : "+v"(x), "+v"(sum));
      };
      // S^T of half t (keys 32 t .. 32 t + 31 of the block), the weights of `w` (UNDER) between its products.
      auto score = [&](int t, auto under, f32x16_t& w) __attribute__((always_inline)) {
        constexpr bool UNDER = decltype(under)::value;
        constexpr int kSteps = D / 8, kEach = (16 + kSteps - 1) / kSteps;
        const float nm = UNDER ? bias() : 0.f;
        f32x16_t s, odd;  // the even and the odd steps' products: two chains half as long
        float sum = 0.f;
        const float* kr = sK + (32 * t + col) * kF32Row;
        f32x4_t x = *reinterpret_cast<const f32x4_t*>(kr + 4 * f32_swz_k(col, hh));
#pragma unroll
        for (int c = 0; c < kSteps; ++c) {
          f32x4_t next = x;
          if (c + 1 < kSteps) next = *reinterpret_cast<const f32x4_t*>(kr + 4 * f32_swz_k(col, 2 * (c + 1) + hh));
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f32x16_t& acc = e % 2 == 0 ? s : odd;
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], qf[4 * c + e], c + e / 2 == 0 ? f32x16_t{0} : acc, 0, 0,
                                                       0);
          }
          x = next;
          if constexpr (UNDER) {
#pragma unroll
            for (int i = kEach * c; i < kEach * (c + 1) && i < 16; ++i) {
              float y = w[i];
              weight(y, nm, sum);
              w[i] = y;
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (UNDER) l += sum;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] += odd[i];
        return s;
      };
      // The half's largest score, keys not attended put to -inf.
      auto mask_max = [&](f32x16_t& s, int t) __attribute__((always_inline)) {
        if (bits != ~0ull) {
          const uint32_t mine = static_cast<uint32_t>(bits >> (32 * t)) >> (4 * hh);
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            if (!((mine >> (8 * (i / 4) + i % 4)) & 1u)) s[i] = -INFINITY;
          }
        }
        float mb = s[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) mb = fmaxf(mb, s[i]);
        return fmaxf(mb, __shfl_xor(mb, 32, 64)) * sl2;
      };
      // The running max is raised only where a score passes it by kF32Rise (the weights stay below 2^kF32Rise, which
      // costs fp32 sums nothing); O, l and the weights `held` already formed come down with it.
      auto raise = [&](float mb, f32x16_t* held) __attribute__((always_inline)) {
        if (__builtin_amdgcn_ballot_w64(mb > m + kF32Rise) != 0ull) {
          // alpha is 0 on a query's first attended keys (m = -inf), with O and l still 0.
          const float mn = fmaxf(m, mb);
          const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
          m = mn;
          l *= alpha;
#pragma unroll
          for (int j = 0; j < kTiles; ++j) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              o[j][i] *= alpha;
              total[j][i] *= alpha;
            }
          }
          if (held) {
#pragma unroll
            for (int i = 0; i < 16; ++i) (*held)[i] *= alpha;
          }
        }
      };
      // O^T += V^T . P^T of half t, the weights of `w` (UNDER) between its products.
      auto pv = [&](const f32x16_t& s, int t, auto under, f32x16_t& w) __attribute__((always_inline)) {
        constexpr bool UNDER = decltype(under)::value;
        const float nm = UNDER ? bias() : 0.f;
        float sum = 0.f;
        // Entry i is key 32 t + 8 (i / 4) + 4 hh + i % 4; f32_swz_v on floats: bit 5 of the row's float index flips
        // with bit 2 of the key, which is hh.
        auto read = [&](int i, int j) __attribute__((always_inline)) {
          return sV[(32 * t + 8 * (i / 4) + 4 * hh + i % 4) * kF32Row + ((32 * j + col) ^ (32 * hh))];
        };
        float x[kTiles], next[kTiles];
#pragma unroll
        for (int j = 0; j < kTiles; ++j) x[j] = read(0, j);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
#pragma unroll
          for (int j = 0; j < kTiles; ++j) next[j] = i + 1 < 16 ? read(i + 1, j) : 0.f;
#pragma unroll
          for (int j = 0; j < kTiles; ++j) {
            o[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[j], s[i], o[j], 0, 0, 0);
            x[j] = next[j];
          }
          if constexpr (UNDER) {
            float y = w[i];
            weight(y, nm, sum);
            w[i] = y;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (UNDER) l += sum;
      };
      // Half 0's weights under half 1's score product, half 1's under half 0's second product (a product is 16 passes,
      // a weight three VALU instructions): a wave left alone on its SIMD still keeps the matrix core busy.
      f32x16_t none;
      f32x16_t s0 = score(0, std::false_type{}, none);
      raise(mask_max(s0, 0), nullptr);
      f32x16_t s1 = score(1, std::true_type{}, s0);
      raise(mask_max(s1, 1), &s0);
      pv(s0, 0, std::true_type{}, s1);
      pv(s1, 1, std::false_type{}, none);
    }
    if ((blk - blk0) % kF32Fold == kF32Fold - 1 || !more || next >= bound) {
#pragma unroll
      for (int j = 0; j < kTiles; ++j) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          total[j][i] += o[j][i];
          o[j][i] = 0.f;
        }
      }
    }
    if (more && next >= bound) fold(next);
    __syncthreads();
    if (more) {
      store_block();
      __syncthreads();
    }
  }
  join();

  if constexpr (SPLIT) {
    split_publish(p, item, team, qt);
    if (item.first > 0 || item.end < pieces.count) {
      float* slot = split_slot(p, team, qt);
      const int ql = w * 32 + col;
#pragma unroll
      for (int j = 0; j < kTiles; ++j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int d0 = 32 * j + 8 * g + 4 * hh;
          if (d0 < D) {
            split_store(slot, d0, ql, total[j][4 * g], total[j][4 * g + 1], total[j][4 * g + 2], total[j][4 * g + 3]);
          }
        }
      }
      if (hh == 0) {
        slot[kQTile * D + ql] = m;
        slot[kQTile * (D + 1) + ql] = l;
      }
      return;
    }
  }
  if (q_ok) {
    // No key at all (L = 0, or no attended key): zeros, as the bf16 kernel writes.
    const float inv = l == 0.f ? 0.f : 1.f / l;
    float* out = p.o + b * p.so_b + h * p.so_h + q * p.so_q;
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int d = 32 * j + 8 * (i / 4) + 4 * hh + i % 4;
        if (d < D) out[d] = total[j][i] * inv;
      }
    }
  }
}

template <int D, bool VT, bool KMASK>
static void launch_f32(const XattnF32Params& p, unsigned grid, hipStream_t s) {
  if (p.teams) {
    xattn_f32_kernel<D, VT, KMASK, true><<<static_cast<unsigned>(p.teams) * p.q_tiles, kThreads, 0, s>>>(p);
    split_join_kernel<float><<<split_join_grid(grid, D), kThreads, 0, s>>>(p);
  } else {
    xattn_f32_kernel<D, VT, KMASK, false><<<grid, kThreads, 0, s>>>(p);
  }
}

template <int D>
static void launch_f32(const XattnF32Params& p, unsigned grid, hipStream_t s, bool vt) {
  if (p.kv_mask) {
    vt ? launch_f32<D, true, true>(p, grid, s) : launch_f32<D, false, true>(p, grid, s);
  } else {
    vt ? launch_f32<D, true, false>(p, grid, s) : launch_f32<D, false, false>(p, grid, s);
  }
}

}  // namespace svhip

using namespace svhip;

static int xattn_f32_impl(const float* q, const float* k, const float* v, float* o, const uint8_t* kv_mask,
                          int64_t sm_b, const int32_t* kv_blocks, int64_t sb_b, const int32_t* kv_len,
                          const int32_t* cu_seqlens, int64_t B, int64_t H,
                          int64_t Q, int64_t D, int64_t kv_cap, int64_t sq_b, int64_t sq_h, int64_t sq_q,
                          int64_t sk_b, int64_t sk_h, int64_t sk_k, int64_t sv_b, int64_t sv_h, int64_t sv_k,
                          int64_t sv_d, int64_t so_b, int64_t so_h, int64_t so_q, float scale, void* workspace,
                          size_t workspace_bytes, void* stream, const char* name) {
  clear_error();
  SVHIP_REQUIRE(q && k && v && o, "%s: null pointer", name);
  if (kv_mask) {
    SVHIP_REQUIRE(sm_b >= 0, "%s: negative mask row stride", name);
  } else {
    SVHIP_REQUIRE(kv_len || cu_seqlens, "%s: need kv_len or cu_seqlens", name);
  }
  // With lists of attended blocks kv_len may come with cu_seqlens (svhip_mask_blocks gives both).
  const bool listed = kv_mask && kv_len && kv_blocks;
  SVHIP_REQUIRE(!(kv_len && cu_seqlens) || listed, "%s: kv_len and cu_seqlens are exclusive", name);
  SVHIP_REQUIRE(B >= 0 && H >= 1 && Q >= 0, "%s: bad sizes", name);
  SVHIP_REQUIRE(D == 16 || D == 32 || D == 48 || D == 64, "%s: head_dim %lld unsupported (16, 32, 48 or 64)", name,
                (long long)D);
  SVHIP_REQUIRE(scale > 0.f && scale < 3.0e38f, "%s: softmax scale must be positive and finite", name);
  SVHIP_REQUIRE(kv_cap >= 0 && kv_cap < (1ll << 31), "%s: kv_cap out of range", name);
  SVHIP_REQUIRE(sv_k == 1 || sv_d == 1, "%s: V needs a unit stride along keys or head_dim", name);
  const bool vt = sv_k == 1 && sv_d != 1;
  SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(q) % 16 == 0 && sq_q % 4 == 0 && sq_h % 4 == 0 && sq_b % 4 == 0,
                "%s: Q rows must be 16-byte aligned", name);
  SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(k) % 16 == 0 && sk_k % 4 == 0 && sk_h % 4 == 0 && sk_b % 4 == 0,
                "%s: K rows must be 16-byte aligned", name);
  SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(v) % 16 == 0 && (vt ? sv_d : sv_k) % 4 == 0 && sv_h % 4 == 0 &&
                    sv_b % 4 == 0,
                "%s: V rows must be 16-byte aligned", name);
  SVHIP_REQUIRE(!listed || B <= 1 || sb_b > cdiv(kv_cap, kKB), "%s: block rows shorter than the windows' lists", name);
  if (B == 0 || Q == 0) return SVHIP_OK;
  XattnF32Params p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = o;
  p.kv_len = kv_len;
  p.cu_seqlens = cu_seqlens;
  p.kv_mask = kv_mask;
  p.v_scale = nullptr;
  p.sm_b = sm_b;
  p.kv_blocks = nullptr;
  p.sb_b = 0;
  p.B = B;
  p.H = H;
  p.Q = Q;
  p.D = D;
  p.kv_cap = kv_cap;
  p.sq_b = sq_b;
  p.sq_h = sq_h;
  p.sq_q = sq_q;
  p.sk_b = sk_b;
  p.sk_h = sk_h;
  p.sk_k = sk_k;
  p.sv_b = sv_b;
  p.sv_h = sv_h;
  p.sv_k = sv_k;
  p.sv_d = sv_d;
  p.so_b = so_b;
  p.so_h = so_h;
  p.so_q = so_q;
  p.scale_log2 = scale * kLog2e;
  p.q_tiles = static_cast<int>(cdiv(Q, kQTile));
  const int64_t grid = static_cast<int64_t>(p.q_tiles) * H * B;
  SVHIP_REQUIRE(grid < (1ll << 31), "%s: grid too large", name);
  p.lone = lone_teams(Q);
  p.piece_blocks = kF32PieceBlocks;
  p.part = nullptr;
  p.teams = 0;
  p.resident = 0;
  // With a key mask the split form needs the windows' lists of attended blocks (svhip_mask_blocks).
  if (workspace && (!kv_mask || listed)) {
    const int teams = split_teams(B, H, Q, kv_cap, kF32Resident, kF32PieceBlocks, 0);
    const size_t need = split_workspace_bytes(B, H, Q, D, kv_cap, kF32Resident, kF32PieceBlocks, 0);
    if (teams) {
      SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0 && workspace_bytes >= need,
                    "%s: workspace too small or unaligned (%zu < %zu bytes)", name, workspace_bytes, need);
      p.part = static_cast<float*>(workspace);
      p.teams = teams;
      p.resident = resident_teams(Q, kF32Resident);
      if (listed) {
        p.kv_blocks = kv_blocks;
        p.sb_b = sb_b;
      }
    }
  }
  hipStream_t s = as_stream(stream);
  const unsigned g = static_cast<unsigned>(grid);
  switch (D) {
    case 16:
      launch_f32<16>(p, g, s, vt);
      break;
    case 32:
      launch_f32<32>(p, g, s, vt);
      break;
    case 48:
      launch_f32<48>(p, g, s, vt);
      break;
    default:
      launch_f32<64>(p, g, s, vt);
      break;
  }
  SVHIP_LAUNCHED(name);
  return SVHIP_OK;
}

extern "C" size_t svhip_xattn_f32_workspace_bytes(int64_t B, int64_t H, int64_t Q, int64_t D, int64_t kv_cap) {
  if (H < 1 || D < 1 || kv_cap < 0) return 0;
  return split_workspace_bytes(B, H, Q, D, kv_cap, kF32Resident, kF32PieceBlocks, 0);
}

extern "C" int svhip_xattn_fwd_f32_ws(const float* q, const float* k, const float* v, float* o, const uint8_t* kv_mask,
                                      int64_t sm_b, const int32_t* kv_len, const int32_t* kv_blocks, int64_t sb_b,
                                      const int32_t* cu_seqlens, int64_t B,
                                      int64_t H, int64_t Q, int64_t D, int64_t kv_cap, int64_t sq_b, int64_t sq_h,
                                      int64_t sq_q, int64_t sk_b, int64_t sk_h, int64_t sk_k, int64_t sv_b,
                                      int64_t sv_h, int64_t sv_k, int64_t sv_d, int64_t so_b, int64_t so_h,
                                      int64_t so_q, float scale, void* workspace, size_t workspace_bytes,
                                      void* stream) {
  return xattn_f32_impl(q, k, v, o, kv_mask, sm_b, kv_blocks, sb_b, kv_len, cu_seqlens, B, H, Q, D, kv_cap, sq_b, sq_h,
                        sq_q, sk_b, sk_h, sk_k, sv_b, sv_h, sv_k, sv_d, so_b, so_h, so_q, scale, workspace,
                        workspace_bytes, stream, "svhip_xattn_fwd_f32_ws");
}

extern "C" int svhip_xattn_fwd_f32(const float* q, const float* k, const float* v, float* o, const int32_t* kv_len,
                                   const int32_t* cu_seqlens, int64_t B, int64_t H, int64_t Q, int64_t D,
                                   int64_t kv_cap, int64_t sq_b, int64_t sq_h, int64_t sq_q, int64_t sk_b,
                                   int64_t sk_h, int64_t sk_k, int64_t sv_b, int64_t sv_h, int64_t sv_k, int64_t sv_d,
                                   int64_t so_b, int64_t so_h, int64_t so_q, float scale, void* stream) {
  return xattn_f32_impl(q, k, v, o, nullptr, 0, nullptr, 0, kv_len, cu_seqlens, B, H, Q, D, kv_cap, sq_b, sq_h, sq_q,
                        sk_b, sk_h, sk_k, sv_b, sv_h, sv_k, sv_d, so_b, so_h, so_q, scale, nullptr, 0, stream,
                        "svhip_xattn_fwd_f32");
}

extern "C" int svhip_xattn_fwd_f32_masked(const float* q, const float* k, const float* v, float* o,
                                          const uint8_t* kv_mask, int64_t sm_b, const int32_t* kv_len,
                                          const int32_t* cu_seqlens, int64_t B, int64_t H, int64_t Q, int64_t D,
                                          int64_t kv_cap, int64_t sq_b, int64_t sq_h, int64_t sq_q, int64_t sk_b,
                                          int64_t sk_h, int64_t sk_k, int64_t sv_b, int64_t sv_h, int64_t sv_k,
                                          int64_t sv_d, int64_t so_b, int64_t so_h, int64_t so_q, float scale,
                                          void* stream) {
  const char* name = "svhip_xattn_fwd_f32_masked";
  clear_error();
  SVHIP_REQUIRE(kv_mask, "%s: null key mask", name);
  return xattn_f32_impl(q, k, v, o, kv_mask, sm_b, nullptr, 0, kv_len, cu_seqlens, B, H, Q, D, kv_cap, sq_b, sq_h, sq_q,
                        sk_b, sk_h, sk_k, sv_b, sv_h, sv_k, sv_d, so_b, so_h, so_q, scale, nullptr, 0, stream,
                        name);
}
