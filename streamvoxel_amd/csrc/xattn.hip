// Cross attention: the launches of the unsplit kernel and the entry points (the kernel is in xattn_kernel.hpp).
#include "xattn_kernel.hpp"

namespace svhip {

// The instantiation for DT = head_dim / 32 rounded up: bf16 K and V directly to LDS (V^T of the padded layout,
// V rows of either layout; head_dim 32 DT without exec masking), with or without a key mask; e4m3, V^T of the
// packed layout and K/V spans past 32-bit offsets through registers.
template <int DT, bool ONES>
void launch_dt(const XattnParams& p, unsigned g, hipStream_t s, bool fp8, bool pv8, bool vt, bool direct) {
  constexpr int RS = ONES ? kRegister : kRegisterFull;
  if (p.teams) {
    launch_split<DT, ONES>(p, g, s, vt, direct);
    return;
  }
  if (p.kv_mask) {  // bf16 only (checked by the entry point)
    constexpr int DS = ONES ? kDirect : kDirectFull;
    if (direct && vt) {
      xattn_fwd_kernel<false, true, DS, DT, ONES, true><<<g, kThreads, 0, s>>>(p);
    } else if (direct) {
      xattn_fwd_kernel<false, false, DS, DT, ONES, true><<<g, kThreads, 0, s>>>(p);
    } else if (vt) {
      xattn_fwd_kernel<false, true, RS, DT, ONES, true><<<g, kThreads, 0, s>>>(p);
    } else {
      xattn_fwd_kernel<false, false, RS, DT, ONES, true><<<g, kThreads, 0, s>>>(p);
    }
    return;
  }
  if (fp8 && pv8) {
    if (vt && direct) {
      xattn_fwd_kernel<true, true, RS, DT, ONES, false, true, true><<<g, kThreads, 0, s>>>(p);
    } else if (vt) {
      xattn_fwd_kernel<true, true, RS, DT, ONES, false, true><<<g, kThreads, 0, s>>>(p);
    } else {
      xattn_fwd_kernel<true, false, RS, DT, ONES, false, true><<<g, kThreads, 0, s>>>(p);
    }
  } else if (fp8) {
    if (vt) {
      xattn_fwd_kernel<true, true, RS, DT, ONES, false, false><<<g, kThreads, 0, s>>>(p);
    } else {
      xattn_fwd_kernel<true, false, RS, DT, ONES, false, false><<<g, kThreads, 0, s>>>(p);
    }
  } else if (direct && !ONES) {
    if (vt) {
      xattn_fwd_kernel<false, true, kDirectFull, DT, false><<<g, kThreads, 0, s>>>(p);
    } else {
      xattn_fwd_kernel<false, false, kDirectFull, DT, false><<<g, kThreads, 0, s>>>(p);
    }
  } else if (direct) {
    if (vt) {
      xattn_fwd_kernel<false, true, kDirect, DT, true><<<g, kThreads, 0, s>>>(p);
    } else {
      xattn_fwd_kernel<false, false, kDirect, DT, true><<<g, kThreads, 0, s>>>(p);
    }
  } else if (vt) {
    xattn_fwd_kernel<false, true, RS, DT, ONES><<<g, kThreads, 0, s>>>(p);
  } else {
    xattn_fwd_kernel<false, false, RS, DT, ONES><<<g, kThreads, 0, s>>>(p);
  }
}

// The instantiation for DT = head_dim / 32 rounded up (see launch_dt); head_dim below 32 DT takes the row sum from
// the matrix cores.
template <int DT>
void launch(const XattnParams& p, unsigned g, hipStream_t s, bool fp8, bool pv8, bool vt, bool direct) {
  if (p.D < 32 * DT) {
    launch_dt<DT, true>(p, g, s, fp8, pv8, vt, direct);
  } else {
    launch_dt<DT, false>(p, g, s, fp8, pv8, vt, direct);
  }
}

// Workgroups of the split kernels resident on a CU: their registers allow three waves per SIMD up to head_dim 64.
static int resident(int64_t D) { return D <= 64 ? 3 : 2; }
// (key_split.hpp)
constexpr int kTilesPerBlock = 8;

static int xattn_impl(const void* q, const void* k, const void* v, void* o, int kv_dtype, const int32_t* kv_len,
                      const int32_t* cu_seqlens, const float* k_scale, const float* v_scale, const uint8_t* kv_mask,
                      int64_t sm_b, const int32_t* kv_blocks, int64_t sb_b, int64_t B, int64_t H, int64_t Q,
                      int64_t D, int64_t kv_cap, int64_t sq_b,
                      int64_t sq_h, int64_t sq_q, int64_t sk_b, int64_t sk_h, int64_t sk_k, int64_t sv_b,
                      int64_t sv_h, int64_t sv_k, int64_t sv_d, int64_t so_b, int64_t so_h, int64_t so_q,
                      float scale, void* workspace, size_t workspace_bytes, void* stream, const char* name) {
  SVHIP_REQUIRE(q && k && v && o, "%s: null pointer", name);
  SVHIP_REQUIRE(B >= 0 && H >= 1 && Q >= 0, "%s: bad sizes", name);
  SVHIP_REQUIRE(D >= 8 && D <= kMaxD && D % 8 == 0, "%s: head_dim %lld unsupported (multiple of 8, <= %d)", name,
                (long long)D, kMaxD);
  SVHIP_REQUIRE(scale > 0.f && scale < 3.0e38f, "%s: softmax scale must be positive and finite", name);
  SVHIP_REQUIRE(kv_dtype == SVHIP_BF16 || kv_dtype == SVHIP_FP8_E4M3 || kv_dtype == SVHIP_FP8_E4M3_PFP8,
                "%s: kv dtype %d unsupported", name, kv_dtype);
  const bool fp8 = kv_dtype != SVHIP_BF16;
  const bool pv8 = kv_dtype == SVHIP_FP8_E4M3_PFP8;
  SVHIP_REQUIRE(!fp8 || (k_scale && v_scale), "%s: fp8 K/V need k_scale and v_scale", name);
  SVHIP_REQUIRE(!kv_mask || !fp8, "%s: the key mask takes bf16 K/V", name);
  SVHIP_REQUIRE(sv_k == 1 || sv_d == 1, "%s: V needs a unit stride along keys or head_dim", name);
  const bool vt = sv_k == 1 && sv_d != 1;
  const size_t eb = fp8 ? 1 : 2;
  // Row starts must allow 16-byte (bf16) / 8-byte (fp8) vector loads.
  const uintptr_t align = fp8 ? 8 : 16;
  SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(q) % 16 == 0 && (sq_q * 2) % 16 == 0 && (sq_h * 2) % 16 == 0 &&
                    (sq_b * 2) % 16 == 0,
                "%s: Q rows must be 16-byte aligned", name);
  SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(o) % 8 == 0 && (so_q * 2) % 8 == 0 && (so_h * 2) % 8 == 0 &&
                    (so_b * 2) % 8 == 0,
                "%s: O rows must be 8-byte aligned", name);
  SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(k) % align == 0 && (sk_k * eb) % align == 0 &&
                    (sk_h * eb) % align == 0 && (sk_b * eb) % align == 0,
                "%s: K rows must be %d-byte aligned", name, (int)align);
  if (!vt) {
    SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(v) % align == 0 && (sv_k * eb) % align == 0 &&
                      (sv_h * eb) % align == 0 && (sv_b * eb) % align == 0,
                  "%s: V rows must be %d-byte aligned", name, (int)align);
  }
  const bool listed = kv_mask && kv_len && kv_blocks;
  SVHIP_REQUIRE(!listed || B <= 1 || sb_b > cdiv(kv_cap, kKB), "%s: block rows shorter than the windows' lists", name);
  if (B == 0 || Q == 0) return SVHIP_OK;
  SVHIP_REQUIRE(kv_cap >= 0 && kv_cap < (1ll << 31), "%s: kv_cap out of range", name);
  XattnParams p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = o;
  p.kv_len = kv_len;
  p.cu_seqlens = cu_seqlens;
  p.k_scale = k_scale;
  p.v_scale = v_scale;
  p.kv_mask = kv_mask;
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
  // Direct-to-LDS staging: bf16 K and V whose rows (and every 8-key run of V^T) start on 16-byte boundaries and
  // whose byte offsets from a (window, head) base fit 32 bits: V^T of the padded layout, row-major V of either
  // layout (a packed window starts at any key, which keeps its rows aligned but not the 8-key runs of V^T).
  // e4m3 with the fp8 second product: V^T alone takes direct loads, rows of 16-byte aligned 16-key runs.
  const bool direct =
      fp8 ? (pv8 && vt && !cu_seqlens && reinterpret_cast<uintptr_t>(v) % 16 == 0 && sv_d % 16 == 0 &&
             sv_h % 16 == 0 && sv_b % 16 == 0 && D * sv_d + kv_cap < (1ll << 32))
          : (reinterpret_cast<uintptr_t>(v) % 16 == 0 && sv_h % 8 == 0 && sv_b % 8 == 0 &&
             (kv_cap * sk_k + D) * 2 < (1ll << 32) &&
             (vt ? !cu_seqlens && sv_d % 8 == 0 && (D * sv_d + kv_cap) * 2 < (1ll << 32)
                 : sv_k % 8 == 0 && (kv_cap * sv_k + D) * 2 < (1ll << 32)));
  // Every bf16 form cuts the same keys into the same pieces, split or not, so that all layouts give the same bits. With
  // a key mask the split form needs the windows' lists of attended blocks (svhip_mask_blocks). An e4m3 cache's windows
  // are one piece each.
  p.lone = lone_teams(Q);
  p.piece_blocks = kPieceBlocks;
  p.part = nullptr;
  p.teams = 0;
  p.resident = 0;
  if (workspace && !fp8 && (!kv_mask || listed)) {
    const int teams = split_teams(B, H, Q, kv_cap, resident(D), kPieceBlocks, kTilesPerBlock);
    if (teams) {
      SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0 &&
                        workspace_bytes >= svhip_xattn_workspace_bytes(B, H, Q, D, kv_cap),
                    "%s: workspace too small or unaligned (%zu < %zu bytes)", name, workspace_bytes,
                    svhip_xattn_workspace_bytes(B, H, Q, D, kv_cap));
      p.part = static_cast<float*>(workspace);
      p.teams = teams;
      p.resident = resident_teams(Q, resident(D));
      if (listed) {
        p.kv_blocks = kv_blocks;
        p.sb_b = sb_b;
      }
    }
  }
  hipStream_t s = as_stream(stream);
  const unsigned g = static_cast<unsigned>(grid);
  if (D <= 64) {
    launch<2>(p, g, s, fp8, pv8, vt, direct);
  } else if (D <= 96) {
    launch<3>(p, g, s, fp8, pv8, vt, direct);
  } else {
    launch<4>(p, g, s, fp8, pv8, vt, direct);
  }
  SVHIP_LAUNCHED(name);
  return SVHIP_OK;
}

// One workgroup per window: out[b] = 1 + the last attended key among the window's first min(kv_len[b], kv_cap)
// keys (kv_cap without kv_len), 0 when it has none.
__global__ __launch_bounds__(kThreads) void mask_lengths_kernel(const uint8_t* mask, int64_t sm_b,
                                                                const int32_t* kv_len, int64_t kv_cap, int32_t* out) {
  __shared__ int s_last;
  const int64_t b = blockIdx.x;
  int64_t n = kv_cap;
  if (kv_len) n = min(max(static_cast<int64_t>(kv_len[b]), int64_t{0}), kv_cap);
  if (threadIdx.x == 0) s_last = -1;
  __syncthreads();
  const int last = last_attended(mask + b * sm_b, static_cast<int>(n));
  if (last >= 0) atomicMax(&s_last, last);
  __syncthreads();
  if (threadIdx.x == 0) out[b] = s_last + 1;
}

// One workgroup per window: mask_lengths_kernel's result, and the list of the window's 64-key blocks that hold an
// attended key. A wave looks at one block at a time (a byte a lane, eight blocks' loads in flight), then every thread
// places one block by the flags before it. Rounds of kListBlocks blocks.
constexpr int kListThreads = 1024;
constexpr int kListBlocks = kListThreads;
__global__ __launch_bounds__(kListThreads) void mask_blocks_kernel(const uint8_t* mask, int64_t sm_b,
                                                                   const int32_t* kv_len, int64_t kv_cap,
                                                                   int32_t* lengths, int32_t* blocks, int64_t sb_b) {
  constexpr int kWaves = kListThreads / 64, kAhead = 8;
  __shared__ uint8_t s_flag[kListBlocks];
  __shared__ int s_count[kWaves];
  __shared__ int s_last;
  const int64_t b = blockIdx.x;
  int64_t cap = kv_cap;
  if (kv_len) cap = min(max(static_cast<int64_t>(kv_len[b]), int64_t{0}), kv_cap);
  const int n = static_cast<int>(cap), nb = static_cast<int>((cap + kKB - 1) / kKB);
  const uint8_t* row = mask + b * sm_b;
  int32_t* list = blocks + b * sb_b;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (threadIdx.x == 0) s_last = -1;
  int placed = 0, last = -1;
  for (int base = 0; base < nb; base += kListBlocks) {
    const int count = min(nb - base, kListBlocks);
    __syncthreads();  // the flags of the round before have been read
    for (int k0 = w; k0 < count; k0 += kWaves * kAhead) {
      uint8_t v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int64_t j = static_cast<int64_t>(base + k0 + u * kWaves) * kKB + lane;
        v[u] = row[j < n ? j : n - 1];
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int k = k0 + u * kWaves;
        if (k >= count) break;
        const int64_t j = static_cast<int64_t>(base + k) * kKB + lane;
        const uint64_t bits = __ballot(j < n && v[u] != 0);
        if (lane == 0) s_flag[k] = bits != 0ull;
        if (bits != 0ull) last = max(last, (base + k) * kKB + 63 - __clzll(bits));
      }
    }
    __syncthreads();
    const bool on = static_cast<int>(threadIdx.x) < count && s_flag[threadIdx.x] != 0;
    const uint64_t flags = __ballot(on);
    if (lane == 0) s_count[w] = __popcll(flags);
    __syncthreads();
    int at = placed + __popcll(flags & ((1ull << lane) - 1ull));
    for (int i = 0; i < kWaves; ++i) {
      at += i < w ? s_count[i] : 0;
      placed += s_count[i];
    }
    if (on) list[1 + at] = base + static_cast<int>(threadIdx.x);
  }
  if (lane == 0 && last >= 0) atomicMax(&s_last, last);
  __syncthreads();
  if (threadIdx.x == 0) {
    lengths[b] = s_last + 1;
    list[0] = placed;
  }
}

}  // namespace svhip

using namespace svhip;

extern "C" int svhip_mask_lengths(const uint8_t* kv_mask, int64_t sm_b, const int32_t* kv_len, int64_t B,
                                  int64_t kv_cap, int32_t* out, void* stream) {
  const char* name = "svhip_mask_lengths";
  clear_error();
  SVHIP_REQUIRE(kv_mask && out, "%s: null pointer", name);
  SVHIP_REQUIRE(B >= 0 && B < (1ll << 31), "%s: bad window count", name);
  SVHIP_REQUIRE(kv_cap >= 0 && kv_cap < (1ll << 31), "%s: kv_cap out of range", name);
  if (B == 0) return SVHIP_OK;
  mask_lengths_kernel<<<static_cast<unsigned>(B), kThreads, 0, as_stream(stream)>>>(kv_mask, sm_b, kv_len, kv_cap,
                                                                                      out);
  SVHIP_LAUNCHED(name);
  return SVHIP_OK;
}

extern "C" int svhip_mask_blocks(const uint8_t* kv_mask, int64_t sm_b, const int32_t* kv_len, int64_t B,
                                 int64_t kv_cap, int32_t* lengths, int32_t* blocks, int64_t sb_b, void* stream) {
  const char* name = "svhip_mask_blocks";
  clear_error();
  SVHIP_REQUIRE(kv_mask && lengths && blocks, "%s: null pointer", name);
  SVHIP_REQUIRE(B >= 0 && B < (1ll << 31), "%s: bad window count", name);
  SVHIP_REQUIRE(kv_cap >= 0 && kv_cap < (1ll << 31) - kKB, "%s: kv_cap out of range", name);
  SVHIP_REQUIRE(B <= 1 || sb_b > cdiv(kv_cap, kKB), "%s: block rows shorter than the windows' lists", name);
  if (B == 0) return SVHIP_OK;
  mask_blocks_kernel<<<static_cast<unsigned>(B), kListThreads, 0, as_stream(stream)>>>(kv_mask, sm_b, kv_len, kv_cap,
                                                                                         lengths, blocks, sb_b);
  SVHIP_LAUNCHED(name);
  return SVHIP_OK;
}

#ifdef SVHIP_XATTN_TRACE
// Trace build only: the device buffer the instrumented kernel writes (kTraceWords words per wave), or NULL to stop.
extern "C" int svhip_xattn_trace_set(void* buffer) {
  return hipMemcpyToSymbol(HIP_SYMBOL(g_trace), &buffer, sizeof(buffer)) == hipSuccess ? 0 : -1;
}
#endif

extern "C" size_t svhip_xattn_workspace_bytes(int64_t B, int64_t H, int64_t Q, int64_t D, int64_t kv_cap) {
  if (H < 1 || D < 8 || D > kMaxD || kv_cap < 0) return 0;
  return split_workspace_bytes(B, H, Q, D, kv_cap, resident(D), kPieceBlocks, kTilesPerBlock);
}

extern "C" int svhip_xattn_fwd(const void* q, const void* k, const void* v, void* o, int kv_dtype,
                               const int32_t* kv_len, const int32_t* cu_seqlens, const float* k_scale,
                               const float* v_scale, int64_t B, int64_t H, int64_t Q, int64_t D, int64_t kv_cap,
                               int64_t sq_b, int64_t sq_h, int64_t sq_q, int64_t sk_b, int64_t sk_h, int64_t sk_k,
                               int64_t sv_b, int64_t sv_h, int64_t sv_k, int64_t sv_d, int64_t so_b, int64_t so_h,
                               int64_t so_q, float scale, void* stream) {
  return svhip_xattn_fwd_ws(q, k, v, o, kv_dtype, kv_len, cu_seqlens, k_scale, v_scale, B, H, Q, D, kv_cap, sq_b, sq_h,
                            sq_q, sk_b, sk_h, sk_k, sv_b, sv_h, sv_k, sv_d, so_b, so_h, so_q, scale, nullptr, 0,
                            stream);
}

extern "C" int svhip_xattn_fwd_ws(const void* q, const void* k, const void* v, void* o, int kv_dtype,
                                  const int32_t* kv_len, const int32_t* cu_seqlens, const float* k_scale,
                                  const float* v_scale, int64_t B, int64_t H, int64_t Q, int64_t D, int64_t kv_cap,
                                  int64_t sq_b, int64_t sq_h, int64_t sq_q, int64_t sk_b, int64_t sk_h, int64_t sk_k,
                                  int64_t sv_b, int64_t sv_h, int64_t sv_k, int64_t sv_d, int64_t so_b, int64_t so_h,
                                  int64_t so_q, float scale, void* workspace, size_t workspace_bytes, void* stream) {
  const char* name = "svhip_xattn_fwd";
  clear_error();
  SVHIP_REQUIRE(kv_len || cu_seqlens, "%s: need kv_len or cu_seqlens", name);
  if (cu_seqlens) kv_len = nullptr;  // the packed lengths alone hold
  return xattn_impl(q, k, v, o, kv_dtype, kv_len, cu_seqlens, k_scale, v_scale, nullptr, 0, nullptr, 0, B, H, Q, D,
                    kv_cap, sq_b, sq_h, sq_q, sk_b, sk_h, sk_k, sv_b, sv_h, sv_k, sv_d, so_b, so_h, so_q, scale,
                    workspace, workspace_bytes, stream, name);
}

extern "C" int svhip_xattn_fwd_masked(const void* q, const void* k, const void* v, void* o, const uint8_t* kv_mask,
                                      int64_t sm_b, const int32_t* kv_len, const int32_t* cu_seqlens, int64_t B,
                                      int64_t H, int64_t Q, int64_t D, int64_t kv_cap, int64_t sq_b, int64_t sq_h,
                                      int64_t sq_q, int64_t sk_b, int64_t sk_h, int64_t sk_k, int64_t sv_b,
                                      int64_t sv_h, int64_t sv_k, int64_t sv_d, int64_t so_b, int64_t so_h,
                                      int64_t so_q, float scale, void* stream) {
  clear_error();
  SVHIP_REQUIRE(!(kv_len && cu_seqlens), "svhip_xattn_fwd_masked: kv_len and cu_seqlens are exclusive");
  return svhip_xattn_fwd_masked_ws(q, k, v, o, kv_mask, sm_b, kv_len, nullptr, 0, cu_seqlens, B, H, Q, D, kv_cap, sq_b,
                                   sq_h, sq_q, sk_b, sk_h, sk_k, sv_b, sv_h, sv_k, sv_d, so_b, so_h, so_q, scale,
                                   nullptr, 0,
                                   stream);
}

extern "C" int svhip_xattn_fwd_masked_ws(const void* q, const void* k, const void* v, void* o, const uint8_t* kv_mask,
                                      int64_t sm_b, const int32_t* kv_len, const int32_t* kv_blocks, int64_t sb_b,
                                         const int32_t* cu_seqlens, int64_t B,
                                      int64_t H, int64_t Q, int64_t D, int64_t kv_cap, int64_t sq_b, int64_t sq_h,
                                      int64_t sq_q, int64_t sk_b, int64_t sk_h, int64_t sk_k, int64_t sv_b,
                                      int64_t sv_h, int64_t sv_k, int64_t sv_d, int64_t so_b, int64_t so_h,
                                      int64_t so_q, float scale, void* workspace,
                                         size_t workspace_bytes, void* stream) {
  const char* name = "svhip_xattn_fwd_masked";
  clear_error();
  SVHIP_REQUIRE(kv_mask, "%s: null key mask", name);
  return xattn_impl(q, k, v, o, SVHIP_BF16, kv_len, cu_seqlens, nullptr, nullptr, kv_mask, sm_b, kv_blocks, sb_b, B, H,
                    Q, D, kv_cap, sq_b, sq_h, sq_q, sk_b, sk_h, sk_k, sv_b, sv_h, sv_k, sv_d, so_b, so_h, so_q, scale,
                    workspace, workspace_bytes, stream, name);
}
