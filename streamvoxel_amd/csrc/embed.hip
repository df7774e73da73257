// Gather patchify: the embedding of a window's voxel tokens as patch tokens, without the one-hot tensor.
//
//   out[b, n, :] = bias + sum_{o < p^3} table[tokens[b, voxel(n, o)] * p^3 + o, :]
//
// where patch token n (row-major over the (Y/p, Z/p, X/p) patch grid) covers voxel (p*gy + dy, p*gz + dz, p*gx + dx)
// at kernel offset o = (dy*p + dz)*p + dx, and table[c * p^3 + o, :] = conv.weight[:, c, dy, dz, dx], i.e.
// Conv3d(C+1 -> W, kernel p, stride p) of the one-hot tokens (models/unconditional_md4_timefree.py:141-147) written
// as the reference's embedding bag (stream/fast_ops.py:54-75, GatherPatch). The p^3 rows are summed in fp32 in
// offset order, rounded to bf16, then the bias is added in bf16 (one more rounding), as embedding_bag(mode='sum')
// followed by `out + bias` compute it in bf16.
//
// Bound: 64 gathered rows a token (805 MB of 16-byte gathers for 8 windows at width 768), from the L2s; the table
// (30 MB) does not fit an XCD's 4 MB. So the columns are cut into 8 slices, one per XCD (consecutive workgroups go
// round robin to the XCDs): an XCD gathers from its slice of the table only (3.75 MB at width 768), and the rows of the
// few cells that fill a window (the mask token, air) stay in the CUs' L1. A lane holds one 16-byte column chunk of one
// token and takes the offsets in order, kEmbedBatch loads in flight. 8 windows, width 768, half of the voxels masked:
// 44.3 us with whole rows per workgroup (18 TB/s of gathers), 34.8 us here (23 TB/s); 16 loads in flight 35.4 us.
#include "common.hpp"

namespace svhip {

constexpr int kEmbedThreads = 256;
constexpr int kEmbedSlices = 8;         // column slices, one per XCD
constexpr int kEmbedBatch = 8;          // table loads a lane has in flight
constexpr int kEmbedMaxTokens = 64;     // patch tokens per workgroup
constexpr int64_t kEmbedGroups = 1 << 20;  // token groups per launch (a launch holds fewer than 2^32 threads)
constexpr int kEmbedMaxOffsets = 64;    // p^3 up to 4^3
constexpr int kEmbedMaxWidth = 2048;

struct EmbedArgs {
  const int64_t* tokens;  // (b, y, z, x) at b*stb + ((y*Z) + z)*X + x
  const uint16_t* table;  // [(C+1) * p^3, W]
  const uint16_t* bias;   // [W] or null
  uint16_t* out;          // (b, n, c) at b*sob + n*son + c
  int64_t B, Y, Z, X, p, cells, W;
  int64_t stb, sob, son;
  int* bad;               // set when a token lies outside [0, cells)
  int slice_chunks;       // 16-byte chunks of a column slice
  int wg_tokens;          // patch tokens of a workgroup: kEmbedThreads / slice_chunks, at most kEmbedMaxTokens
  uint32_t first_group;   // token group of the launch's first workgroups
};

// P: the patch edge 4 at compile time (the index arithmetic of the table rows is a third of the work otherwise), or 0.
// WIDE: the table holds 2^32 16-byte chunks or more.
template <int P, bool WIDE>
__global__ __launch_bounds__(kEmbedThreads) void patch_embed_kernel(EmbedArgs a) {
  // First 16-byte chunk (WIDE: the index) of every (token, offset)'s table row; offsets past p^3 are never read.
  __shared__ __attribute__((aligned(16))) uint32_t s_row[kEmbedMaxTokens][kEmbedMaxOffsets + 4];
  __shared__ int64_t s_base[kEmbedMaxTokens];  // element of every token's first voxel
  const int p = P ? P : static_cast<int>(a.p), p3 = p * p * p;
  const uint32_t gx = static_cast<uint32_t>(a.X / p), gzx = static_cast<uint32_t>(a.Z / p) * gx;
  const uint32_t per_window = static_cast<uint32_t>(a.Y / p) * gzx;  // B per_window < 2^31 (checked by the host)
  const int slice = static_cast<int>(blockIdx.x % kEmbedSlices);
  const uint32_t first = (a.first_group + blockIdx.x / kEmbedSlices) * a.wg_tokens;  // flat (b, n) of token 0
  const int chunks = static_cast<int>(a.W / 8);
  const int chunk0 = slice * a.slice_chunks;
  if (chunk0 >= chunks) return;
  const int count = min(static_cast<int>(static_cast<uint32_t>(a.B) * per_window - first), a.wg_tokens);
  if (static_cast<int>(threadIdx.x) < count) {
    const uint32_t flat = first + threadIdx.x;
    const uint32_t b = flat / per_window, n = flat - b * per_window;
    const uint32_t py = n / gzx, zx = n - py * gzx, pz = zx / gx, px = zx - pz * gx;
    s_base[threadIdx.x] = b * a.stb + (static_cast<int64_t>(py) * a.Z + pz) * p * a.X + static_cast<int64_t>(px) * p;
  }
  __syncthreads();
  const uint32_t row_units = static_cast<uint32_t>(chunks);
  for (int i = threadIdx.x; i < count * p3; i += kEmbedThreads) {
    const int t = i / p3, o = i - t * p3;  // with P = 4 a thread keeps its offset o
    const int dy = o / (p * p), dz = (o / p) % p, dx = o % p;
    int64_t cell = a.tokens[s_base[t] + (dy * a.Z + dz) * a.X + dx];
    if (cell < 0 || cell >= a.cells) {
      atomicOr(a.bad, 1);
      cell = 0;
    }
    s_row[t][o] = (static_cast<uint32_t>(cell) * p3 + o) * (WIDE ? 1u : row_units);
  }
  __syncthreads();
  const int t = static_cast<int>(threadIdx.x) / a.slice_chunks;
  const int ch = chunk0 + static_cast<int>(threadIdx.x) % a.slice_chunks;
  if (t >= count || ch >= chunks) return;
  const uint4* base = reinterpret_cast<const uint4*>(a.table) + ch;
  auto chunk = [&](uint32_t row) __attribute__((always_inline)) -> const uint4& {
    return base[WIDE ? static_cast<int64_t>(row) * row_units : static_cast<int64_t>(row)];
  };
  float acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.f;
  auto add = [&](const uint4& w) __attribute__((always_inline)) {
    const uint32_t e[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[2 * j] += __uint_as_float(e[j] << 16);
      acc[2 * j + 1] += __uint_as_float(e[j] & 0xffff0000u);
    }
  };
  // Offsets in order: the sum of each column is taken o = 0, 1, 2, ...
  int o0 = 0;
  for (; o0 + kEmbedBatch <= p3; o0 += kEmbedBatch) {
    uint4 w[kEmbedBatch];
#pragma unroll
    for (int u = 0; u < kEmbedBatch; ++u) {
      w[u] = chunk(s_row[t][o0 + u]);
    }
#pragma unroll
    for (int u = 0; u < kEmbedBatch; ++u) add(w[u]);
  }
  for (; o0 < p3; ++o0) {
    add(chunk(s_row[t][o0]));
  }
  const uint32_t flat = first + t;
  const uint32_t b = flat / per_window, n = flat - b * per_window;
  uint32_t out[4];
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    float v0 = acc[j], v1 = acc[j + 1];
    bf16_round2(v0, v1);
    if (a.bias) {
      v0 += bf16_bits_to_float(a.bias[8 * ch + j]);
      v1 += bf16_bits_to_float(a.bias[8 * ch + j + 1]);
    }
    out[j / 2] = bf16_pack2(v0, v1);
  }
  *reinterpret_cast<uint4*>(a.out + b * a.sob + n * a.son + 8 * ch) = make_uint4(out[0], out[1], out[2], out[3]);
}

}  // namespace svhip

using namespace svhip;

extern "C" int svhip_patch_embed(const int64_t* tokens, const void* table, const void* bias, void* out, int* bad,
                                 int64_t B, int64_t Y, int64_t Z, int64_t X, int64_t patch, int64_t cells, int64_t W,
                                 int64_t st_b, int64_t so_b, int64_t so_n, void* stream) {
  const char* name = "svhip_patch_embed";
  clear_error();
  SVHIP_REQUIRE(tokens && table && out && bad, "%s: null pointer", name);
  SVHIP_REQUIRE(B >= 0 && Y >= 1 && Z >= 1 && X >= 1 && cells >= 1, "%s: bad sizes", name);
  SVHIP_REQUIRE(patch >= 1 && patch * patch * patch <= kEmbedMaxOffsets && Y % patch == 0 && Z % patch == 0 &&
                    X % patch == 0,
                "%s: patch %lld must divide the window and have at most %d offsets", name, (long long)patch,
                kEmbedMaxOffsets);
  SVHIP_REQUIRE(W >= 8 && W % 8 == 0 && W <= kEmbedMaxWidth, "%s: width %lld unsupported (a multiple of 8 up to %d)",
                name, (long long)W, kEmbedMaxWidth);
  SVHIP_REQUIRE(cells * patch * patch * patch < (1ll << 31), "%s: table too large", name);
  SVHIP_REQUIRE(reinterpret_cast<uintptr_t>(table) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                    so_b % 8 == 0 && so_n % 8 == 0,
                "%s: table and output rows must start on 16-byte boundaries", name);
  const int64_t tokens_total = B * (Y / patch) * (Z / patch) * (X / patch);
  if (tokens_total == 0) return SVHIP_OK;
  const int64_t slice_chunks = cdiv(W / 8, kEmbedSlices);
  const int64_t wg_tokens = kEmbedThreads / slice_chunks < kEmbedMaxTokens ? kEmbedThreads / slice_chunks
                                                                          : kEmbedMaxTokens;
  EmbedArgs a{tokens, static_cast<const uint16_t*>(table), static_cast<const uint16_t*>(bias),
              static_cast<uint16_t*>(out), B, Y, Z, X, patch, cells, W, st_b, so_b, so_n, bad,
              static_cast<int>(slice_chunks), static_cast<int>(wg_tokens), 0};
  SVHIP_REQUIRE(tokens_total < (1ll << 31), "%s: grid too large", name);
  const bool wide = cells * patch * patch * patch * (W / 8) >= (1ll << 32);
  const int64_t groups = cdiv(tokens_total, wg_tokens);
  for (int64_t first = 0; first < groups; first += kEmbedGroups) {
    a.first_group = static_cast<uint32_t>(first);
    const int64_t count = groups - first < kEmbedGroups ? groups - first : kEmbedGroups;
    const unsigned grid = static_cast<unsigned>(count * kEmbedSlices);
    if (wide) {
      patch_embed_kernel<0, true><<<grid, kEmbedThreads, 0, as_stream(stream)>>>(a);
    } else if (patch == 4) {
      patch_embed_kernel<4, false><<<grid, kEmbedThreads, 0, as_stream(stream)>>>(a);
    } else {
      patch_embed_kernel<0, false><<<grid, kEmbedThreads, 0, as_stream(stream)>>>(a);
    }
  }
  SVHIP_LAUNCHED(name);
  return SVHIP_OK;
}
