// Codec twins of the CPU NF4 codec on gfx950: full-matrix dequant to fp32,
// embedding-row gather to bf16, and the quantiser that makes synthetic weights.
// Device counterparts of internal/nf4/nf4.go:46-121,129-185 and
// gpu/host/embedding.py:74-107; each is bit-exact against the CPU codec.

#include "nf4_common.h"

namespace chr {
namespace {

typedef __attribute__((ext_vector_type(4))) float F32x4;

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xF, 0xF, true));
}

// largest of sixteen neighbouring lanes, in all of them
__device__ __forceinline__ uint32_t group_max16_u32(uint32_t v) {
  v = max(v, dpp_u32<kDppQuadXor1>(v));
  v = max(v, dpp_u32<kDppQuadXor2>(v));
  v = max(v, dpp_u32<kDppRowHalfMirror>(v));
  return max(v, dpp_u32<kDppRowMirror>(v));
}

__device__ __forceinline__ void load_lut_lds(float *lut) {
  if (threadIdx.x < 16) {
    lut[threadIdx.x] = bits_to_f32(kLutBits[threadIdx.x]);
  }
  __syncthreads();
}

// ---- codec twins -------------------------------------------------------------
// A grid holds fewer than 2^32 threads: more workgroups of 256 than this go in several launches, which
// take their blocks from `first` on.
constexpr int64_t kLaunchBlocks = int64_t{1} << 23;

// out is [M, K] fp32, four weights a thread and kDequantQuads such quads, a workgroup's quads
// back to back: every store is a 16-byte piece of a wavefront's whole kilobyte, and the loads (two
// bytes a quad) are all issued before the first store.  Bound by the fp32 it writes, past the caches
// (the non-temporal hint): 5120x27648 in 90 us (7.1 TB/s; 128 without the hint, 93 / 102 with one or
// eight quads), where eight weights a thread in eight 4-byte stores 32 bytes apart took 332.  For every
// size: decoding and a pass over the result behind it (from a graph, eight 4-byte stores before) 512x512
// to 13824x5120 0.5 to 1.0 of the time, but 1024x1024 7.1 / 7.3 us.  The
// 16-entry table has no bank conflicts (equal codes read one address, others other banks).
constexpr int kDequantQuads = 4;

template <typename Index>
__global__ __launch_bounds__(256) void dequant_f32(const uint8_t *__restrict__ packed,
                                                   const uint16_t *__restrict__ scale,
                                                   float *__restrict__ out, Index first, Index quads,
                                                   int K4, int K_pad) {
  __shared__ float lut[16];
  load_lut_lds(lut);
  const Index q0 = (first + blockIdx.x) * (256 * kDequantQuads) + threadIdx.x;
  uint32_t w[kDequantQuads];
  uint16_t s[kDequantQuads];
#pragma unroll
  for (int u = 0; u < kDequantQuads; ++u) {
    const Index q = min(q0 + static_cast<Index>(256 * u), quads - 1);
    const Index r = q / static_cast<Index>(K4);
    const int d = static_cast<int>(q - r * static_cast<Index>(K4));
    w[u] = reinterpret_cast<const uint16_t *>(packed + static_cast<size_t>(r) * (K_pad >> 1))[d];
    s[u] = scale[static_cast<size_t>(r) * (K_pad >> 6) + (d >> 4)];
  }
#pragma unroll
  for (int u = 0; u < kDequantQuads; ++u) {
    const Index q = q0 + static_cast<Index>(256 * u);
    if (q < quads) {
      const float f = f16_to_f32(s[u]);
      const F32x4 v = {lut[w[u] & 0xFu] * f, lut[(w[u] >> 4) & 0xFu] * f, lut[(w[u] >> 8) & 0xFu] * f,
                       lut[w[u] >> 12] * f};
      __builtin_nontemporal_store(v, reinterpret_cast<F32x4 *>(out) + q);
    }
  }
}

// Rows that are no whole quads (K % 4 != 0, or an output that is not 16-byte aligned): one weight a
// store, so a wavefront still writes 256 consecutive bytes, and Q of them a thread: eight where there
// is work for them (9000x5001 in 45 us, 59 with four, 107 before), four below.
constexpr int64_t kManyWeights = int64_t{1} << 23;

template <typename Index, int Q>
__global__ __launch_bounds__(256) void dequant_f32_ragged(const uint8_t *__restrict__ packed,
                                                          const uint16_t *__restrict__ scale,
                                                          float *__restrict__ out, Index first, Index count,
                                                          int K, int K_pad) {
  __shared__ float lut[16];
  load_lut_lds(lut);
  const Index i0 = (first + blockIdx.x) * (256 * Q) + threadIdx.x;
  uint8_t w[Q];
  uint16_t s[Q];
  bool odd[Q];
#pragma unroll
  for (int u = 0; u < Q; ++u) {
    const Index i = min(i0 + static_cast<Index>(256 * u), count - 1);
    const Index r = i / static_cast<Index>(K);
    const int k = static_cast<int>(i - r * static_cast<Index>(K));
    w[u] = packed[static_cast<size_t>(r) * (K_pad >> 1) + (k >> 1)];
    s[u] = scale[static_cast<size_t>(r) * (K_pad >> 6) + (k >> 6)];
    odd[u] = (k & 1) != 0;
  }
#pragma unroll
  for (int u = 0; u < Q; ++u) {
    const Index i = i0 + static_cast<Index>(256 * u);
    if (i < count) {
      __builtin_nontemporal_store(lut[odd[u] ? w[u] >> 4 : w[u] & 0xF] * f16_to_f32(s[u]), out + i);
    }
  }
}

// One workgroup per requested row; out is bf16 [n, K].
__global__ __launch_bounds__(256) void embed_rows(const uint8_t *__restrict__ packed,
                                                  const uint16_t *__restrict__ scale,
                                                  const int64_t *__restrict__ ids,
                                                  uint16_t *__restrict__ out, int M, int K,
                                                  int K_pad) {
  __shared__ float lut[16];
  load_lut_lds(lut);
  int64_t id = ids[blockIdx.x];
  if (id < 0 || id >= M) {
    // Out-of-range id: write zeros rather than read outside the table.
    for (int k = threadIdx.x; k < K; k += 256) {
      out[static_cast<size_t>(blockIdx.x) * K + k] = 0;
    }
    return;
  }
  const uint32_t *prow =
      reinterpret_cast<const uint32_t *>(packed + static_cast<size_t>(id) * (K_pad >> 1));
  const uint16_t *srow = scale + static_cast<size_t>(id) * (K_pad >> 6);
  uint16_t *o = out + static_cast<size_t>(blockIdx.x) * K;
  for (int d = threadIdx.x; d < (K_pad >> 3); d += 256) {
    const uint32_t w = prow[d];
    const float s = f16_to_f32(srow[d >> 3]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = (d << 3) + j;
      if (k < K) {
        o[k] = f32_to_bf16(lut[(w >> (4 * j)) & 0xFu] * s);
      }
    }
  }
}

// ---- quantiser ---------------------------------------------------------------
// The CPU encoder takes the level with the smallest squared distance, in fp32, the first of equal
// ones (internal/nf4/nf4.go:129-185).  Between two neighbouring levels both distances are monotone
// in u, also after rounding, so there is one smallest u from which the upper level wins:
// crossing(j), found here by bisection over binary32 patterns with the same fp32 operations.
constexpr float level_at(int j) { return __builtin_bit_cast(float, kLevelBits[j]); }
constexpr float square_from(float u, int j) {
  const float d = u - level_at(j);
  return d * d;
}
// binary32 patterns in numeric order, for bisection over both signs
constexpr int64_t ordered(float f) {
  const uint32_t b = __builtin_bit_cast(uint32_t, f);
  return (b >> 31) != 0 ? -static_cast<int64_t>(b & 0x7FFFFFFFu) : static_cast<int64_t>(b);
}
constexpr float from_ordered(int64_t o) {
  return __builtin_bit_cast(float, static_cast<uint32_t>(o < 0 ? (0x80000000u | static_cast<uint32_t>(-o)) : static_cast<uint32_t>(o)));
}
constexpr float crossing(int j) {
  int64_t lo = ordered(level_at(j)), hi = ordered(level_at(j + 1));  // lower wins at lo, upper at hi
  while (hi - lo > 1) {
    const int64_t mid = lo + (hi - lo) / 2;
    const float u = from_ordered(mid);
    if (square_from(u, j + 1) < square_from(u, j)) {
      hi = mid;
    } else {
      lo = mid;
    }
  }
  return from_ordered(hi);
}

// [-1, 1] in 32 cells of 1/16 (and one for u = 1): neighbouring crossings are further apart than a
// cell and none lies within 2^-12 of a cell's border, where rounding (u + 1) * 16 could name the
// neighbour (cells_hold), so a u's code is the number of crossings left of its cell plus one comparison.
constexpr int kCells = 33;
struct CellTable {
  float cross[kCells];  // the crossing inside the cell, or one no u reaches
  uint32_t below[kCells];
};
constexpr CellTable make_cells() {
  CellTable t{};
  for (int c = 0; c < kCells; ++c) {
    t.cross[c] = 4.f;
    t.below[c] = 0;
    for (int j = 0; j < 15; ++j) {
      const float x = (crossing(j) + 1.f) * 16.f;
      if (x < static_cast<float>(c)) {
        ++t.below[c];
      } else if (x < static_cast<float>(c + 1)) {
        t.cross[c] = crossing(j);
      }
    }
  }
  return t;
}
constexpr bool cells_hold() {
  for (int j = 0; j < 15; ++j) {
    const float x = (crossing(j) + 1.f) * 16.f;
    const float off = x - static_cast<float>(static_cast<int>(x));
    if (off < 0x1p-12f || off > 1.f - 0x1p-12f) {
      return false;
    }
    if (j > 0 && static_cast<int>(x) == static_cast<int>((crossing(j - 1) + 1.f) * 16.f)) {
      return false;
    }
  }
  return true;
}
static_assert(cells_hold(), "one crossing a cell, none at a border");
__device__ __constant__ const CellTable kCellTable = make_cells();

// Sixteen lanes a group, four weights a lane (VEC: one 16-byte load; otherwise rows are not whole
// pieces and the four are loaded one by one), kQuantUnroll groups a lane with all loads first.
// Steps are those of the CPU encoder: absmax, binary16 scale, divide by the widened scale, clip,
// nearest level.  Bound by reading the fp32; one weight a lane, a wavefront a group and fifteen
// squared distances a weight took 302 us at 13824x5120 (vector arithmetic), dividing every weight 90,
// so 72 (4 TB/s, launches back to back; 25 and 29 at 5120x5120).  Four groups a lane, or loads past the
// caches, are no faster.
constexpr int kQuantUnroll = 2;

template <bool VEC>
__global__ __launch_bounds__(256) void quantize_groups(const float *__restrict__ src,
                                                       uint8_t *__restrict__ packed,
                                                       uint16_t *__restrict__ scale,
                                                       int32_t *status, int64_t first, int64_t groups,
                                                       int K, int ng) {
  __shared__ float cross[kCells];
  __shared__ uint32_t below[kCells];
  if (threadIdx.x < kCells) {
    cross[threadIdx.x] = kCellTable.cross[threadIdx.x];
    below[threadIdx.x] = kCellTable.below[threadIdx.x];
  }
  __syncthreads();
  const int lane = threadIdx.x & 15;
  const int64_t g0 = (first + blockIdx.x) * (16 * kQuantUnroll) + (threadIdx.x >> 4);
  F32x4 v[kQuantUnroll];
#pragma unroll
  for (int n = 0; n < kQuantUnroll; ++n) {
    const int64_t gi = min(g0 + 16 * n, groups - 1);
    // (a 32-bit division wherever the index allows it)
    const int64_t r = groups <= INT32_MAX ? static_cast<int64_t>(static_cast<uint32_t>(gi) / static_cast<uint32_t>(ng)) : gi / ng;
    const int c = (static_cast<int>(gi - r * ng) << 6) + 4 * lane;
    const float *p = src + r * K + c;
    if constexpr (VEC) {
      v[n] = c < K ? *reinterpret_cast<const F32x4 *>(p) : F32x4{0.f, 0.f, 0.f, 0.f};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[n][e] = c + e < K ? p[e] : 0.f;
      }
    }
  }
#pragma unroll
  for (int n = 0; n < kQuantUnroll; ++n) {
    const int64_t gi = g0 + 16 * n;
    if (gi >= groups) {
      break;
    }
    uint32_t top = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      // magnitudes as integers order like the numbers, non-finite ones above all finite
      top = max(top, f32_to_bits(v[n][e]) & 0x7FFFFFFFu);
    }
    top = group_max16_u32(top);
    if (top >= 0x7F800000u) {
      if (lane == 0 && status != nullptr) {
        atomicOr(status, 1);
      }
      continue;
    }
    float s32 = bits_to_f32(top);
    if (s32 == 0.f) {
      s32 = 1.f;
    }
    uint16_t s16 = __builtin_bit_cast(uint16_t, static_cast<_Float16>(s32));
    float s = f16_to_f32(s16);
    if (((f32_to_bits(s) & 0x7F800000u) == 0x7F800000u) || !(s > 0.f)) {
      s16 = s32 > 65504.f ? 0x7BFFu : 0x3C00u;  // the largest finite scale, or one
      s = f16_to_f32(s16);
    }
    // v / s decides nothing but the side of a crossing: the product with the reciprocal (an ulp off, as its
    // product: 2^-22 at most) decides the same wherever it is further from it.  Nearer, one weight in 10^5, the
    // wavefront divides.
    const float inv = __builtin_amdgcn_rcpf(s);
    uint32_t codes = 0;
    bool near = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float u = fminf(fmaxf(v[n][e] * inv, -1.f), 1.f);
      const int cell = static_cast<int>((u + 1.f) * 16.f);
      const float past = u - cross[cell];
      near |= fabsf(past) < 0x1p-21f;
      codes |= (below[cell] + (past >= 0.f ? 1u : 0u)) << (4 * e);
    }
    if (__builtin_expect(__any(near), 0)) {
      codes = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float u = v[n][e] / s;
        u = u > 1.f ? 1.f : (u < -1.f ? -1.f : u);
        const int cell = static_cast<int>((u + 1.f) * 16.f);
        codes |= (below[cell] + (u >= cross[cell] ? 1u : 0u)) << (4 * e);
      }
    }
    if (aligned2(packed)) {
      reinterpret_cast<uint16_t *>(packed)[gi * 16 + lane] = static_cast<uint16_t>(codes);
    } else {
      packed[gi * 32 + 2 * lane] = static_cast<uint8_t>(codes);
      packed[gi * 32 + 2 * lane + 1] = static_cast<uint8_t>(codes >> 8);
    }
    if (lane == 0) {
      scale[gi] = s16;
    }
  }
}

int desc_rc(const chr_nf4_dev_t *w) {
  if (w->M < 1 || w->K < 1 || w->packed == nullptr || w->scale == nullptr) {
    return -3;
  }
  if (!k_pad_ok(w->K, w->K_pad)) {
    return -4;
  }
  return 0;
}

}  // namespace
}  // namespace chr

using namespace chr;

extern "C" int chr_nf4_dequant(const chr_nf4_dev_t *w, float *out, void *stream) {
  if (w == nullptr || out == nullptr) {
    return -1;
  }
  if (const int rc = desc_rc(w)) {
    return rc;
  }
  if ((reinterpret_cast<uintptr_t>(w->packed) & 3u) != 0 || !aligned2(w->scale)) {
    return -5;
  }
  const int64_t count = static_cast<int64_t>(w->M) * w->K;
  const bool whole = (w->K & 3) == 0 && aligned16(out);
  const int64_t items = whole ? count / 4 : count;
  const int per = 256 * (whole || count < kManyWeights ? kDequantQuads : 8);
  const int64_t blocks = (items + per - 1) / per;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // 32-bit indexes (and divisions) unless the last workgroup's would pass 2^32
  const bool narrow = items < (int64_t{1} << 32) - per;
  auto run = [&](auto kernel, auto n, int row) {
    for (int64_t b = 0; b < blocks; b += kLaunchBlocks) {
      const dim3 grid(static_cast<unsigned>(blocks - b < kLaunchBlocks ? blocks - b : kLaunchBlocks));
      kernel<<<grid, dim3(256), 0, st>>>(w->packed, w->scale, out, static_cast<decltype(n)>(b), n, row, w->K_pad);
    }
  };
  if (whole && narrow) {
    run(dequant_f32<uint32_t>, static_cast<uint32_t>(items), w->K / 4);
  } else if (whole) {
    run(dequant_f32<uint64_t>, static_cast<uint64_t>(items), w->K / 4);
  } else if (count < kManyWeights) {
    run(dequant_f32_ragged<uint32_t, kDequantQuads>, static_cast<uint32_t>(items), w->K);
  } else if (narrow) {
    run(dequant_f32_ragged<uint32_t, 8>, static_cast<uint32_t>(items), w->K);
  } else {
    run(dequant_f32_ragged<uint64_t, 8>, static_cast<uint64_t>(items), w->K);
  }
  return launch_rc();
}

extern "C" int chr_nf4_embed_rows(const chr_nf4_dev_t *table, const void *ids, int32_t n,
                                  void *out, void *stream) {
  if (table == nullptr || ids == nullptr || out == nullptr) {
    return -1;
  }
  if (n < 1) {
    return -2;
  }
  if (const int rc = desc_rc(table)) {
    return rc;
  }
  if ((reinterpret_cast<uintptr_t>(table->packed) & 3u) != 0 || !aligned2(table->scale)) {
    return -5;
  }
  embed_rows<<<dim3(static_cast<unsigned>(n)), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
      table->packed, table->scale, static_cast<const int64_t *>(ids),
      static_cast<uint16_t *>(out), table->M, table->K, table->K_pad);
  return launch_rc();
}

extern "C" int chr_nf4_quantize(const float *src, const chr_nf4_dev_t *dst, int32_t *status,
                                void *stream) {
  if (src == nullptr || dst == nullptr) {
    return -1;
  }
  if (const int rc = desc_rc(dst)) {
    return rc;
  }
  const int ng = dst->K_pad >> 6;
  const int64_t groups = static_cast<int64_t>(dst->M) * ng;
  const int64_t blocks = (groups + 16 * kQuantUnroll - 1) / (16 * kQuantUnroll);
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint8_t *packed = const_cast<uint8_t *>(dst->packed);
  uint16_t *scale = const_cast<uint16_t *>(dst->scale);
  for (int64_t b = 0; b < blocks; b += kLaunchBlocks) {
    const dim3 grid(static_cast<unsigned>(blocks - b < kLaunchBlocks ? blocks - b : kLaunchBlocks)), block(256);
    if ((dst->K & 3) == 0 && aligned16(src)) {
      quantize_groups<true><<<grid, block, 0, st>>>(src, packed, scale, status, b, groups, dst->K, ng);
    } else {
      quantize_groups<false><<<grid, block, 0, st>>>(src, packed, scale, status, b, groups, dst->K, ng);
    }
  }
  return launch_rc();
}

extern "C" int chr_nf4_abi_version(void) { return 1; }
